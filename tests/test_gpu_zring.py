"""The iterate formed from the kept preconditioned residuals (a ring of 16):
a solve stopped after m steps must return the x that its recursive residual
belongs to, on both sides of every ring boundary."""

import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [dict(precision=1, mg_levels=2), dict(precision=0, mg_levels=2),
                                dict(precision=0, precond=1),
                                dict(precision=1, mg_levels=2, flags=1)])
@pytest.mark.parametrize("steps", [1, 2, 15, 16, 17, 32, 33])
def test_iterate_belongs_to_its_residual(gpu_available, kw, steps):
    """max |div u| of the corrected field (from x) against max |r|/V of the
    recursion (from q).  Both are sums of FP64 terms of the size of the first
    residual, over at most 33 steps: they agree to 1e-12 of it."""
    c = H.case(2, size=(33, 20, 26))
    print(f"[zring] {kw} steps={steps}", flush=True)
    P = H.projector(c, max_iter=steps, div_tol=1e-14, **kw)
    out, st = P.project(H.fields(c), c.bc_flag, c.dt)
    P.close()
    assert st.iterations == steps
    assert st.residual_div < st.initial_div
    assert abs(st.final_div - st.residual_div) <= 1e-12 * st.initial_div


@pytest.mark.parametrize("kw", [dict(precision=1, mg_levels=2), dict(precision=0, mg_levels=2),
                                dict(precision=0, precond=1),
                                dict(precision=1, mg_levels=2, flags=2)])
@pytest.mark.parametrize("steps", [7, 400])
def test_result_does_not_depend_on_the_depth(gpu_available, kw, steps):
    """Rings of 1, 2, 4, 8 and 16 (sp_set_solver_memory): the same iterations
    and the same bytes, for a solve cut short and for one that converges over
    several rings; with an outlet, whose refinement solves again, too."""
    size = (33, 20, 26)
    z = size[0] * size[1] * size[2] * (4 if kw["precision"] and not kw.get("precond") else 8) + 512
    for cfg, bc in ((2, None), (4, 1)):
        c = H.case(cfg, size=size)
        flag, val = list(c.bc_flag), None
        if bc is not None:
            flag[bc], val = 0, [None] * 6
            val[bc] = np.zeros((c.J, c.K), order="F")
        first = None
        for depth in (16, 1, 2, 4, 8):
            print(f"[zring] {kw} steps={steps} cfg={cfg} depth={depth}", flush=True)
            P = H.projector(c, max_iter=steps, **kw)
            P.set_solver_memory((depth - 1) * z)
            out, st = P.project(H.fields(c), flag, c.dt, bc_val=val)
            P.close()
            assert steps == 7 or st.iterations > 16
            if first is None:
                first = out, st.iterations
            assert st.iterations == first[1]
            for n in ("p", "u", "v", "w"):
                assert np.array_equal(out[n], first[0][n]), (depth, n)


@pytest.mark.parametrize("prec", (0, 1))
@pytest.mark.parametrize("depth", (16, 4))
def test_bytes_of_the_pass_that_forms_x(gpu_available, prec, depth):
    """sp_kernel_times counts the z that the pass reads, not the ring."""
    c = H.case(0, size=(32, 32, 32))
    n, z = 32 ** 3, 4 if prec else 8
    print(f"[zring] bytes prec={prec} depth={depth}", flush=True)
    P = H.projector(c, precision=prec)
    P.set_solver_memory((depth - 1) * (n * z + 512))
    P.set_profiling(True)
    _, st = P.project(H.fields(c), c.bc_flag, c.dt)
    t = next(k for k in P.kernel_times() if k["name"] == "cg_xflush")
    P.close()
    full = t["launches"] - 1  # passes that keep p: it is written, and read by the next
    assert full == st.iterations // depth  # one more step was under way
    assert t["bytes"] == n * (z * st.iterations + 9 + full * (9 + 8 + 8 + 8))


@pytest.mark.parametrize("prec", (0, 1))
def test_adjoint_after_the_ring_was_given_back(gpu_available, prec):
    """The ring may go between a forward and its adjoint: the same gradients."""
    c = H.case(2, size=(33, 20, 26))
    print(f"[zring] adjoint prec={prec}", flush=True)
    g = []
    for q in range(3):
        a = np.zeros(c.halo_shape, order="F")
        a[1:-1, 1:-1, 1:-1] = np.random.default_rng(q).uniform(0.0, 1.0, c.shape)
        g.append(a)
    P = H.projector(c, precision=prec, mg_levels=2)
    P.project(H.fields(c), c.bc_flag, c.dt)
    first, st = P.adjoint(*g)
    P.set_solver_memory(0)
    second, st2 = P.adjoint(*g)
    P.close()
    assert st.iterations == st2.iterations > 16
    for n in first:
        if first[n] is not None:
            assert np.array_equal(first[n], second[n]), n
