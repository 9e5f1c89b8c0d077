"""The workloads whose speed this repository keeps track of, as a user's program runs them.

A two-phase cut-cell time step is: momentum predictor, pressure projection, interface transport and, when
a solid has moved, the geometry update.  Every listed case is one such call (or a short chain of them) on
device-resident arrays through the public entry points:

* ``project``   one projection (``Projector.project_dev``): GFM assembly, multigrid-preconditioned CG to
                max|div u| <= 1e-10, velocity correction, divergence check.  ``outlet``: the east wall is a
                pressure outlet (Dirichlet), as in the reference's channel drivers; closed walls otherwise.
* ``gradient``  a projection and its reverse pass through ``projection.project`` (torch.autograd): gradients
                for u*, v*, w* and the three face-coefficient fields.
* ``predict``   one momentum predictor step (``Projector.predict_uvw``) around three spherical solids.
* ``geometry``  the cut-cell update after a solid has moved: GridPreprocess, the momentum-exchange cells,
                the four cell numberings and NewCellFace.
* ``transport`` one interface-transport step (``clsvof_scheme``) and the U/V/W liquid fields made from it.

``cfg`` names the synthetic configurations of ``simcoflow3d_amd.configs`` (0: sphere under an interface,
1: cylinder, stretched grid, 2: breaking-wave interface, 3: as 0, 4: wave tank with three boxes).
"""

import math

import numpy as np
import torch

from simcoflow3d_amd import configs
from simcoflow3d_amd import projection as proj
from simcoflow3d_amd.engine import GEOM_FIELDS, INTERP_FIELDS, LIQUID_FIELDS, Projector, geom_shapes

PREC = {"fp64": 0, "mixed": 1}
NAMES = configs.HALO_FIELDS + configs.FLAG_FIELDS
VEL = ("u_star", "v_star", "w_star")


def listed():
    def project(cfg, size, prec, outlet=False):
        return dict(kind="project", cfg=cfg, I=size[0], J=size[1], K=size[2], prec=prec, outlet=outlet)

    def other(kind, size, **kw):
        return dict(kind=kind, I=size[0], J=size[1], K=size[2], **kw)

    return [
        # a unit test's or a first set-up's grid at the engine's default precision: launches and latency
        dict(name="project_32_fp64", **project(0, (32, 32, 32), "fp64")),
        # the small benchmark configuration, a coarse production run
        dict(name="project_64_mixed", **project(0, (64, 64, 64), "mixed")),
        # a grid nobody chose for the machine: odd sizes, a stretched direction, a cylinder
        dict(name="project_97x130x75_mixed", **project(1, (97, 130, 75), "mixed")),
        # a channel with a pressure outlet: the non-singular system and its refinement
        dict(name="project_outlet_160x96x96_mixed", **project(4, (160, 96, 96), "mixed", True)),
        # the stretched-grid configuration in all FP64
        dict(name="project_128_fp64", **project(1, (128, 128, 128), "fp64")),
        # the headline workload, and the same in all FP64
        dict(name="project_256_mixed", **project(2, (256, 256, 256), "mixed")),
        dict(name="project_256_fp64", **project(2, (256, 256, 256), "fp64")),
        # the largest: a wave tank
        dict(name="project_tank_512x256x256_mixed", **project(4, (512, 256, 256), "mixed")),
        # forward and backward of the differentiable projection
        dict(name="gradient_128_mixed", **other("gradient", (128, 128, 128), cfg=3, prec="mixed")),
        # the other parts of the time step, at grids of a few million cells
        dict(name="predict_192x160x128_order2", **other("predict", (192, 160, 128), order=2)),
        dict(name="geometry_160x128x112", **other("geometry", (160, 128, 112))),
        dict(name="transport_160", **other("transport", (160, 160, 160))),
    ]


def draw(rng):
    """A case of the same ranges: projections most often, the sizes spread over their logarithm."""
    kind = rng.choice(["project"] * 5 + ["gradient", "predict", "geometry", "transport"])
    top = {"project": 24.9, "gradient": 21.0, "predict": 22.0, "geometry": 21.2, "transport": 22.0}[kind]
    low = {"project": 14.0, "gradient": 14.0, "predict": 17.0, "geometry": 17.0, "transport": 17.0}[kind]
    side = 2.0 ** (rng.uniform(low, top) / 3.0)
    I, J, K = (max(9, int(side * f + rng.random())) for f in rng.choice(
        [(1.0, 1.0, 1.0), (1.6, 0.8, 0.75), (0.7, 1.2, 1.15), (1.3, 1.1, 0.65)]))
    if rng.random() < 0.4:  # round sizes are as common as odd ones
        I, J, K = (max(8, 8 * ((n + 4) // 8)) for n in (I, J, K))
    c = dict(kind=kind, I=I, J=J, K=K)
    if kind == "project":
        c.update(cfg=rng.randrange(5), prec=rng.choice(["mixed", "mixed", "fp64"]),
                 outlet=rng.random() < 0.2)
    elif kind == "gradient":
        c.update(cfg=rng.choice([0, 1, 3]), prec=rng.choice(["mixed", "fp64"]))
    elif kind == "predict":
        c.update(order=rng.choice([1, 2]))
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


def _size(case):
    return case["I"], case["J"], case["K"]


def _dev(a, device="cuda"):
    """A host (Fortran-ordered) array as the device tensor with the same bytes."""
    return torch.from_numpy(np.ascontiguousarray(np.asarray(a).T)).to(device)


def _case(case, seed):
    c = configs.generate(case["cfg"], size=_size(case), seed=seed)
    bc, val = [1] * 6, [None] * 6
    if case.get("outlet"):
        bc[1], val[1] = 0, np.zeros((c.J, c.K), order="F")
    return c, bc, val


def _cotangents(shape, seed, device):
    return [torch.from_numpy(configs.uniform(seed, 60 + q, 0.0, 1.0, shape).T.copy()).to(device)
            for q in range(4)]


def _zeros(shape, dtype=torch.float64):
    return torch.zeros(shape, dtype=dtype, device="cuda")


def _spheres(case, seed):
    """Three spheres of solid on a unit cube, z stretched: the four staggered grids and, on each, the
    level set, its normal and the fluid fraction, on the GPU."""
    I, J, K = _size(case)
    z = 1.02 ** np.minimum(np.arange(K), 120)
    d = [np.full(I, 1.0 / I), np.full(J, 1.0 / J), z / z.sum()]
    centre = [np.cumsum(q) - 0.5 * q for q in d]
    face = [c + 0.5 * q for c, q in zip(centre, d)]
    wide = [np.append(c[1:] - c[:-1], q[-1]) for c, q in zip(centre, d)]
    rng = np.random.default_rng(seed)
    balls = [(rng.uniform(0.2, 0.8, 3), rng.uniform(0.08, 0.2)) for _ in range(3)]

    def along(v, axis):
        s = [1, 1, 1]
        s[2 - axis] = len(v)
        return torch.from_numpy(np.ascontiguousarray(v)).cuda().view(s).expand(K, J, I).contiguous()

    grids = []
    for q in range(4):
        x = [along(face[a] if q == a + 1 else centre[a], a) for a in range(3)]
        w = [along(wide[a] if q == a + 1 else d[a], a) for a in range(3)]
        best = None
        for c, r in balls:
            e = [x[a] - float(c[a]) for a in range(3)]
            rho = (e[0] * e[0] + e[1] * e[1] + e[2] * e[2]).sqrt().clamp_min(1e-12)
            new = [rho - float(r)] + [v / rho for v in e]
            best = new if best is None else [torch.where(new[0] < best[0], a, b)
                                             for a, b in zip(new, best)]
        phi, n = best[0], best[1:]
        h = sum(n[a].abs() * w[a] for a in range(3))
        grids.append(dict(x=x, d=w, phi=phi, n=n, vof=(0.5 + phi / h).clamp(0.0, 1.0)))
    return d, wide, grids


def _geometry_cells(case, seed):
    """The P, U, V, W cells as the geometry update takes them."""
    d, wide, grids = _spheres(case, seed)
    sh = geom_shapes(*_size(case))
    g = torch.Generator("cuda").manual_seed(seed)
    cells = []
    for s in grids:
        vof = s["vof"].contiguous()
        c = dict(dx=s["d"][0], dy=s["d"][1], dz=s["d"][2], phi=s["phi"].contiguous(),
                 nx=s["n"][0].contiguous(), ny=s["n"][1].contiguous(), nz=s["n"][2].contiguous(), vof=vof,
                 vof_l=vof * torch.rand(vof.shape, generator=g, dtype=torch.float64, device="cuda"))
        for n in GEOM_FIELDS:
            if n not in c:
                c[n] = _zeros(sh[n][::-1], torch.int32 if n == "cell_type" else torch.float64)
        cells.append(c)
    return d, wide, cells


def _interp(case):
    I, J, K = _size(case)
    return [dict(moex=_zeros((K, J, I), torch.int32), msce=_zeros((3, K, J, I), torch.int32),
                 **{n: _zeros((K + 2, J + 2, I + 2)) for n in INTERP_FIELDS[2:]}) for _ in range(3)]


def _projector(c, case):
    P = Projector(c.shape, precision=PREC[case["prec"]], rho_l=c.rho_l, rho_g=c.rho_g, rho_ref=c.rho_l,
                  pin_i=1, pin_j=1, pin_k=1, div_tol=1e-10)
    P.set_grid_1d(c.dxp, c.dyp, c.dzp, c.dxu, c.dyv, c.dzw)
    return P


def _prepare_project(case, seed):
    c, bc, val = _case(case, seed)
    halo = (c.K + 2, c.J + 2, c.I + 2)
    return dict(P=_projector(c, case), fields={n: _dev(c.fields[n]) for n in NAMES}, bc=bc,
                val=[None if v is None else _dev(v) for v in val], dt=c.dt,
                out={n: _zeros(halo) for n in ("p", "u", "v", "w")})


def _run_project(s):
    st = s["P"].project_dev(s["fields"], s["bc"], s["dt"], s["out"], bc_val=s["val"])
    if not st.converged:
        raise RuntimeError("the projection did not converge")
    return dict(s["out"])


def _prepare_gradient(case, seed):
    c, bc, _ = _case(case, seed)
    grid = (c.dxp, c.dyp, c.dzp, c.dxu, c.dyv, c.dzw)
    E = proj.DeviceProjection(c.shape, grid, {n: _dev(c.fields[n]) for n in NAMES if n not in VEL}, bc, c.dt,
                              precision=PREC[case["prec"]], rho_l=c.rho_l, rho_g=c.rho_g, rho_ref=c.rho_l,
                              pin_i=1, pin_j=1, pin_k=1, div_tol=1e-10)
    us = [_dev(c.fields[n]) for n in VEL]
    leaves = us + E.gfm_beta(*us)
    for t in leaves:
        t.requires_grad_(True)
    return dict(E=E, leaves=leaves, cot=_cotangents(c.halo_shape, seed, "cuda"))


def _run_gradient(s):
    out = proj.project(s["E"], *s["leaves"][:3], s["leaves"][3:])
    grads = torch.autograd.grad(out, s["leaves"], s["cot"])
    return [t.detach() for t in out] + list(grads)


def _prepare_predict(case, seed):
    size = _size(case)
    d, wide, cells = _geometry_cells(case, seed)
    P = Projector(size)
    P.set_grid_1d(*d, *wide)
    x = _interp(case)
    torch.cuda.synchronize()
    P.grid_preprocess(cells, device=True)
    P.define_moex(*(c["cell_type"] for c in cells), *(e["moex"] for e in x), device=True)
    P.new_cell_face(cells, x, device=True)
    source = {"ee": "ee_area", "ne": "ne_area", "te": "te_area", "cent": "cell_cent"}
    view = [{n: (c if source.get(n, n) in c else e)[source.get(n, n)] for n in configs.PRED_CELL_FIELDS}
            for c, e in zip(cells[1:], x)]
    f = configs.predictor_fields(size, seed=seed, time_order=1, itt=2)
    f = dict(f, vel=[_dev(a) for a in f["vel"]], vel_n=None, flux_div_old=_dev(f["flux_div_old"]),
             bcv=[_dev(a) for a in f["bcv"]], params=dict(f["params"], space_order=case["order"]))
    halo = tuple(n + 2 for n in size[::-1])
    return dict(P=P, areas=[cells[0][n] for n in ("ee_area", "ne_area", "te_area")], view=view, f=f,
                pred=[_zeros(halo) for _ in range(3)], dp=[_zeros(halo) for _ in range(3)])


def _run_predict(s):
    s["P"].predict_uvw(s["areas"], s["view"], s["view"], s["f"], s["pred"], s["dp"], device=True)
    return s["pred"] + s["dp"] + [s["f"]["flux_div_old"]]


NUMBERED = ((0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1))


def _prepare_geometry(case, seed):
    I, J, K = _size(case)
    _, _, cells = _geometry_cells(case, seed)
    return dict(P=Projector((I, J, K)), cells=cells, x=_interp(case),
                new=[{n: c[n].clone() for n in ("vof", "vof_l", "cell_type")} for c in cells],
                pos=[_zeros((K - c, J - b, I - a), torch.int32) for a, b, c in NUMBERED])


def _run_geometry(s):
    P, cells, x = s["P"], s["cells"], s["x"]
    for c, new in zip(cells, s["new"]):  # the moved solid's fractions arrive with each step
        for n, t in new.items():
            c[n].copy_(t)
    for e in x:
        e["moex"].zero_()
    torch.cuda.synchronize()
    P.grid_preprocess(cells, device=True)
    P.define_moex(*(c["cell_type"] for c in cells), *(e["moex"] for e in x), device=True)
    ext = [P.number_external(c["cell_type"], *q, posnu=p, device=True)[1]
           for c, q, p in zip(cells, NUMBERED, s["pos"])]
    P.new_cell_face(cells, x, device=True)
    return dict(cells=[{n: c[n] for n in ("vof", "cell_type", "ee_area", "ne_area", "te_area", "fce",
                                          "cell_cent", "wllh", "delh")} for c in cells],
                x=[{n: e[n] for n in ("moex", "msce", "sxe", "etan", "alt")} for e in x],
                pos=s["pos"], ext=ext)


def _prepare_transport(case, seed):
    I, J, K = _size(case)
    rng = np.random.default_rng(seed)
    at, r0 = rng.uniform(0.3, 0.4, 3), rng.uniform(0.12, 0.18)
    e = [torch.linspace(0.0, 1.0, n + 1, dtype=torch.float64, device="cuda") for n in (I, J, K)]
    view = [(1, 1, -1), (1, -1, 1), (-1, 1, 1)]
    x, d = [], []
    for a in range(3):
        x.append((0.5 * (e[a][1:] + e[a][:-1])).view(view[a]).expand(K, J, I).contiguous())
        d.append((e[a][1:] - e[a][:-1]).view(view[a]).expand(K, J, I).contiguous())

    def halo(t):
        return torch.nn.functional.pad(t[None, None], (1,) * 6, mode="replicate")[0, 0].contiguous()

    def radius(shift):
        return sum((x[a] + shift[a] * d[a] - float(at[a])) ** 2 for a in range(3)).sqrt()
    vof = sum((radius((a, b, c)) < r0).double() * 0.125
              for a in (-0.25, 0.25) for b in (-0.25, 0.25) for c in (-0.25, 0.25))
    s2 = [(math.pi * q).sin() ** 2 for q in x]
    t2 = [(2 * math.pi * q).sin() for q in x]
    vel = [2.0 * s2[0] * t2[1] * t2[2], -t2[0] * s2[1] * t2[2], -t2[0] * t2[1] * s2[2]]
    vel = [halo(v) for v in vel]
    hs = (K + 2, J + 2, I + 2)
    faces = [(K, J), (K, J), (K, I), (K, I), (J, I), (J, I)]
    inp = dict(u=vel[0], v=vel[1], w=vel[2], x=x[0], y=x[1], z=x[2], dx=d[0], dy=d[1], dz=d[2],
               nx=_zeros(hs), ny=_zeros(hs), nz=torch.ones(hs, dtype=torch.float64, device="cuda"),
               bcu_w=vel[0][1:-1, 1:-1, 0].contiguous(), bcv_s=vel[1][1:-1, 0, 1:-1].contiguous(),
               bcw_b=vel[2][0, 1:-1, 1:-1].contiguous(), lvs_flag=[1] * 6, lvs_const=[0.0] * 6,
               vof_flag=[1] * 6, vof_const=[0.0] * 6, dt=0.2 / max(I, J, K))
    state = dict(vof_l=halo(vof), phi_l=halo(radius((0, 0, 0)) - float(r0)), nx_l=_zeros(hs), ny_l=_zeros(hs),
                 nz_l=_zeros(hs), lvs_var=[_zeros(q) for q in faces], vof_var=[_zeros(q) for q in faces])
    liquid = [dict(dx=d[0], dy=d[1], dz=d[2], **{n: state[n] for n in LIQUID_FIELDS[3:]})]
    liquid += [dict(dx=d[0], dy=d[1], dz=d[2], **{n: _zeros(hs) for n in LIQUID_FIELDS[3:]}) for _ in range(3)]
    return dict(P=Projector((I, J, K)), inp=inp, state=state, liquid=liquid,
                old={n: state[n].clone() for n in ("vof_l", "phi_l")})


def _run_transport(s):
    for n, t in s["old"].items():  # the same step each time, not the next one
        s["state"][n].copy_(t)
    torch.cuda.synchronize()
    s["P"].clsvof_scheme(s["inp"], s["state"], device=True)
    s["P"].uvw_liquid_field(s["liquid"], device=True, halo_fields=True)
    return dict(state={n: s["state"][n] for n in LIQUID_FIELDS[3:]},
                liquid=[{n: c[n] for n in LIQUID_FIELDS[3:]} for c in s["liquid"][1:]])


_PREPARE = dict(project=_prepare_project, gradient=_prepare_gradient, predict=_prepare_predict,
                geometry=_prepare_geometry, transport=_prepare_transport)
_RUN = dict(project=_run_project, gradient=_run_gradient, predict=_run_predict, geometry=_run_geometry,
            transport=_run_transport)


def prepare(case, seed):
    s = _PREPARE[case["kind"]](case, seed)
    s["kind"] = case["kind"]
    torch.cuda.synchronize()
    return s


def run(state):
    return _RUN[state["kind"]](state)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------


def work(case):
    """Bytes: each input read once, each output written once.  Operations: the face coefficients, the
    matrix rows and the correction (about 300 a cell), and for a solve a dozen CG iterations of about 150
    a cell, which is what multigrid leaves of it."""
    n = case["I"] * case["J"] * case["K"]
    solve = 12 * 150
    bytes_, flops = {
        # 13 halo fields and 7 flags in, p, u, v, w out
        "project": (13 * 8 + 7 * 4 + 4 * 8, 300 + solve),
        # u*, beta, Dp, apertures, vof x 2, flags; p, u, v, w; four cotangents; six gradients
        "gradient": (14 * 8 + 7 * 4 + 4 * 8 + 4 * 8 + 6 * 8, 600 + 2 * solve),
        # velocities, apertures, geometry and interpolation factors in; u*, Dp and the flux divergence out
        "predict": ((3 + 3 + 9 + 18 + 18 + 12) * 8 + 3 * 4 + 9 * 8, 600),
        # per grid: 9 fields in, 19 out; the interpolation factors of three grids
        "geometry": (4 * (9 * 8 + 19 * 8 + 4) + 3 * (12 * 8 + 16) + 4 * 4, 4 * 800),
        # velocities, coordinates, fractions, level set in; the five liquid fields of four grids out
        "transport": ((3 + 3 + 2 + 3) * 8 + 4 * 5 * 8, 1500),
    }[case["kind"]]
    return {"bytes": float(n * bytes_), "flops": float(n * flops)}


def tolerance(case):
    if case["kind"] == "project":
        # the solve stops at max|r|/V <= 1e-10; what is left of a smooth residual moves the pressure by
        # up to about 1e-10 of itself (measured against exact(): 1e-14 to 3e-13)
        return {"rel": 1e-10, "max": 1e-8}
    if case["kind"] == "gradient":
        # the reverse solve stops at 1e-10 of its source (measured against exact(): 1.6e-10)
        return {"rel": 2e-9, "max": 1e-7}
    if case["kind"] == "transport":
        # pow and the Newton steps of the reconstruction leave the last bits open
        return {"rel": 1e-10, "max": 1e-8}
    return "exact"  # the reference's expressions in its order: bit for bit


# ---------------------------------------------------------------------------
# the projection in plain torch, 64 bits
# ---------------------------------------------------------------------------


def _shift(h, axis, s):
    """The interior of a halo tensor, moved by s cells along axis (0: i, 1: j, 2: k)."""
    sl = [slice(1, -1)] * 3
    sl[2 - axis] = slice(1 + s, h.shape[2 - axis] - 1 + s)
    return h[tuple(sl)]


def _line(v, axis, device):
    s = [1, 1, 1]
    s[2 - axis] = -1
    return torch.from_numpy(np.ascontiguousarray(v)).to(device).view(s)


def _gfm(c, f, device):
    """The six face coefficients Dp/d/rho' (W, S, B, E, N, T) of the ghost-fluid method.  A face whose
    neighbour is solid takes the density that the last such cell before it, with k innermost and i outermost,
    has used."""
    eps = 1e-3
    # 1/rho' of the liquid and of the gas, densities relative to the liquid's
    bp, bm = 1.0, c.rho_l / c.rho_g
    phi, full, liq = f["phi_l"], f["vof"], f["vof_l"]
    whole, cut = full > 1 - eps, (full <= 1 - eps) & (full > eps)
    wet = ((liq >= 0.5) & whole) | ((phi < 0) & cut)
    dry = ((liq < 0.5) & whole) | ((phi >= 0) & cut)
    kind = dry.to(torch.int8) * 2
    kind[wet] = 1
    P, here = _shift(kind, 0, 0), _shift(phi, 0, 0)
    out = []
    for face in range(6):
        axis, side = face % 3, -1 if face < 3 else 1
        Q, there = _shift(kind, axis, side), _shift(phi, axis, side)
        d = (c.dxu, c.dyv, c.dzw)[axis]
        d = _line(d if side > 0 else np.append(d[:1], d[:-1]), axis, device)
        dp = _shift(f[("dp_u", "dp_v", "dp_w")[axis]], axis, 0 if side > 0 else -1)
        lam = here.abs() / (here.abs() + there.abs() + 1e-30)
        own = torch.where(P == 1, torch.full_like(lam, bm), torch.full_like(lam, bp))
        other = torch.where(P == 1, torch.full_like(lam, bp), torch.full_like(lam, bm))
        beta = torch.where(Q == P, own, lam * own + (1 - lam) * other)
        if bool(((P > 0) & (Q == 0)).any()):
            order = lambda t: t.permute(2, 1, 0).reshape(-1)  # noqa: E731
            flat, fixed = order(beta), order(beta).clone()
            at = torch.arange(flat.numel(), device=device)
            for k in (1, 2):
                last = torch.where(order((P == k) & (Q > 0)), at, -1).cummax(0).values
                stale = order((P == k) & (Q == 0))
                fixed = torch.where(stale, torch.where(last >= 0, flat[last.clamp_min(0)], order(own)), fixed)
            beta = fixed.view(c.I, c.J, c.K).permute(2, 1, 0)
        t = torch.where(P > 0, dp / d * bp * bm / beta, 0.0).contiguous()
        n = t.shape[2 - axis]
        edge, inner = (0, 1) if side < 0 else (n - 1, n - 2)
        t.select(2 - axis, edge).copy_(t.select(2 - axis, inner).clone())
        out.append(t)
    return out


def _apply(cs, ex, v):
    r = ex * v
    for axis in range(3):
        dim, n = 2 - axis, v.shape[2 - axis]
        flux = cs[axis].narrow(dim, 0, n - 1) * (v.narrow(dim, 0, n - 1) - v.narrow(dim, 1, n - 1))
        r.narrow(dim, 0, n - 1).add_(flux)
        r.narrow(dim, 1, n - 1).sub_(flux)
    return r


class _Solve(torch.autograd.Function):
    """x of A x = b on the active cells, by diagonally preconditioned conjugate gradients in 64 bits."""

    @staticmethod
    def solve(b, cs, ex, act, singular):
        diag = ex.clone()
        for axis in range(3):
            dim, n = 2 - axis, b.shape[2 - axis]
            for at in (0, 1):
                diag.narrow(dim, at, n - 1).add_(cs[axis].narrow(dim, 0, n - 1))
        inv = torch.where(act, 1.0 / diag, 0.0)
        if singular:
            b = torch.where(act, b - b[act].mean(), 0.0)
        x, r = torch.zeros_like(b), b.clone()
        # in the variable scaled by the diagonal's root, so that the residual there says how good x is
        z = inv * r
        p, rz = z.clone(), (r * z).sum()
        first, best, since = float(rz), float(rz), 0
        for it in range(20000):
            q = _apply(cs, ex, p)
            alpha = rz / (p * q).sum()
            x += alpha * p
            r -= alpha * q
            z = inv * r
            new = (r * z).sum()
            p = z + (new / rz) * p
            rz = new
            if it % 25 == 24:
                now = float(rz)
                best, since = (now, 0) if now < 0.5 * best else (best, since + 1)
                if now <= 1e-32 * first or since >= 8:
                    break
        return x

    @staticmethod
    def forward(ctx, b, cx, cy, cz, ex, act, singular):
        x = _Solve.solve(b, (cx, cy, cz), ex, act, singular)
        ctx.save_for_backward(x, cx, cy, cz, ex, act)
        ctx.singular = singular
        return x

    @staticmethod
    def backward(ctx, g):
        x, cx, cy, cz, ex, act = ctx.saved_tensors
        lam = _Solve.solve(torch.where(act, g, 0.0), (cx, cy, cz), ex, act, ctx.singular)
        if ctx.singular:
            lam = torch.where(act, lam - lam[act].mean(), 0.0)
        grads = []
        for axis in range(3):
            dim, n = 2 - axis, x.shape[2 - axis]
            t = torch.zeros_like(x)
            t.narrow(dim, 0, n - 1).copy_(-(lam.narrow(dim, 0, n - 1) - lam.narrow(dim, 1, n - 1))
                                          * (x.narrow(dim, 0, n - 1) - x.narrow(dim, 1, n - 1)))
            grads.append(t)
        return (lam, *grads, None, None, None)


def _project(c, f, bc, coef, device):
    """p, u, v, w (halo tensors) of the projection with face coefficients ``coef``; the pressure of a closed
    box is zero in its first cell, outlet pressures are zero."""
    ct = f["cell_type_p"]
    fluid = ct != 2
    d = [_line(v, a, device) for a, v in enumerate((c.dxp, c.dyp, c.dzp))]
    vol = d[0] * d[1] * d[2]
    area = [vol / d[a] for a in range(3)]
    ap = [f[n] for n in ("ee_area", "ne_area", "te_area")]
    cs, ex = [], torch.zeros_like(vol)
    rhs = torch.zeros_like(vol)
    for a in range(3):
        dim, n = 2 - a, ct.shape[2 - a]
        hi, lo = _shift(ap[a], a, 0), _shift(ap[a], a, -1)
        for side in (0, 1):  # minus, plus
            edge = torch.zeros_like(fluid)
            edge.select(dim, 0 if side == 0 else n - 1).fill_(True)
            beyond = fluid.roll(1 if side == 0 else -1, dim)
            closed = torch.where(edge, torch.full_like(edge, bc[2 * a + side] == 0), ~beyond)
            own = coef[a + 3 * side] * (lo if side == 0 else hi) * area[a]
            ex = ex + torch.where(fluid & closed, own.detach(), 0.0)
            if side == 1:
                cs.append(torch.where(fluid & beyond & ~edge, own, 0.0))
        vel = f[VEL[a]]
        rhs = rhs - area[a] * (hi * _shift(vel, a, 0) - lo * _shift(vel, a, -1))
    rhs = torch.where(fluid, rhs + (_shift(f["vof"], 0, 0) - _shift(f["vof_old"], 0, 0)) * vol / c.dt, 0.0)
    diag = ex.detach().clone()
    for a in range(3):
        dim, n = 2 - a, ct.shape[2 - a]
        for at in (0, 1):
            diag.narrow(dim, at, n - 1).add_(cs[a].detach().narrow(dim, 0, n - 1))
    act = fluid & (diag > 0)
    singular = not bool((ex[act] != 0).any())
    if singular:
        rhs = torch.where(act, rhs - rhs[act].mean(), 0.0)
    x = _Solve.apply(torch.where(act, rhs, 0.0), *cs, ex, act, singular)
    if singular:
        x = x - (x[0, 0, 0] if bool(act[0, 0, 0]) else x[act].mean())
    x = torch.where(act, x, 0.0)
    p = torch.nn.functional.pad(x, (1,) * 6)
    p = p.clone()
    for a in range(3):
        dim, n = 2 - a, x.shape[2 - a]
        for side, at, ghost in ((0, 0, 0), (1, n - 1, n + 1)):
            sl = [slice(1, -1)] * 3
            sl[dim] = ghost
            p[tuple(sl)] = bc[2 * a + side] * x.select(dim, at)
    out = [p]
    for a in range(3):
        m = (f[("moex_u", "moex_v", "moex_w")[a]] != 1) & (f[("cell_type_u", "cell_type_v", "cell_type_w")[a]] != 2)
        new = _shift(f[VEL[a]], a, 0) - (_shift(p, a, 1) - _shift(p, a, 0)) * coef[a + 3]
        out.append(torch.nn.functional.pad(torch.where(m, new, 0.0), (1,) * 6))
    return out


def exact(case, seed):
    """Projections and their gradients in plain torch (64 bits).  The other kinds repeat the reference's
    expressions bit for bit and have no second form here."""
    if case["kind"] not in ("project", "gradient") or case["I"] * case["J"] * case["K"] > 5_000_000:
        return None
    device = "cuda" if torch.cuda.is_available() else "cpu"
    c, bc, _ = _case(case, seed)
    f = {n: _dev(c.fields[n], device) for n in NAMES}
    coef = _gfm(c, f, device)
    if case["kind"] == "project":
        return dict(zip(("p", "u", "v", "w"), _project(c, f, bc, coef, device)))
    d = [_line(v, a, device) for a, v in enumerate((c.dxu, c.dyv, c.dzw))]
    dp = [_shift(f[n], 0, 0) for n in ("dp_u", "dp_v", "dp_w")]
    leaves = [f[n].requires_grad_(True) for n in VEL]
    leaves += [(coef[a + 3] * d[a] / dp[a]).requires_grad_(True) for a in range(3)]
    plus = [dp[a] / d[a] * leaves[3 + a] for a in range(3)]
    minus = []
    for a in range(3):
        n = plus[a].shape[2 - a]
        minus.append(torch.cat([plus[a].narrow(2 - a, 0, 1), plus[a].narrow(2 - a, 0, n - 1)], 2 - a))
    p, u, v, w = _project(c, f, bc, minus + plus, device)
    out = [u, v, w, p]
    grads = torch.autograd.grad(out, leaves, _cotangents(c.halo_shape, seed, device))
    return [t.detach() for t in out] + list(grads)
