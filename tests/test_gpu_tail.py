"""The V-cycle's tail workgroup at the sizes where its levels begin and end:
first levels of just under, exactly and just over two pairs per thread, odd
rows (pairs cut in two), thin grids, a hierarchy that lies in it whole, one
level alone, and cells without couplings (solids)."""

import numpy as np
import pytest

from oracle import orc
from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", (0, 1))
@pytest.mark.parametrize("cfg,size,levels", [
    (0, (16, 16, 16), 0), (0, (15, 17, 16), 0), (1, (17, 16, 16), 0), (2, (33, 31, 32), 0),
    (0, (16, 16, 15), 1), (3, (8, 8, 8), 1), (4, (128, 4, 4), 0), (2, (5, 40, 9), 0),
    (1, (7, 5, 60), 0), (0, (34, 34, 34), 2)])
def test_tail_levels_match_oracle(gpu_available, cfg, size, levels, prec):
    """Pressure and velocities against the oracle's solve (the bars of the
    configurations: 1e-8 of the largest value)."""
    c = H.case(cfg, size=size, seed=5)
    print(f"[tail] cfg={cfg} size={size} levels={levels} prec={prec}", flush=True)
    ref = orc.project(c, pin=(1, 1, 1))
    P = H.projector(c, precision=prec, mg_levels=levels, max_iter=400)
    out, st = P.project(H.fields(c), c.bc_flag, c.dt)
    P.close()
    assert st.converged == 1 and st.final_div <= 1e-10, st.as_dict()
    assert H.rel_inf(out["p"], ref.Pp) <= 1e-8
    inner = (slice(1, -1),) * 3
    umax = max(np.max(np.abs(getattr(ref, n))) for n in "uvw")
    for n in "uvw":
        assert np.max(np.abs(out[n][inner] - getattr(ref, n)[inner])) <= 1e-8 * umax, n


@pytest.mark.parametrize("prec", (0, 1))
@pytest.mark.parametrize("size,levels", [
    ((16, 16, 16), 0), ((15, 17, 16), 0), ((17, 16, 16), 0), ((33, 31, 32), 0), ((16, 16, 15), 1),
    ((128, 4, 4), 0), ((5, 40, 9), 0), ((7, 5, 60), 0), ((34, 34, 34), 2)])
def test_tail_levels_with_a_diagonal_only_term(gpu_available, size, levels, prec):
    """One Dirichlet wall along every axis.  34^3 over two levels ends in 17^3,
    2601 pairs of cells: in the tail in FP32 only (at most 2048 in FP64).  The oracle runs one solve to a
    hundredth of the engine's stop (its search for the rounding floor gives up
    early on thin grids)."""
    for face in (0, 3, 4):
        c = H.case(0, size=size, seed=5)
        c.bc_flag[face] = 0
        dims = [(c.J, c.K), (c.J, c.K), (c.I, c.K), (c.I, c.K), (c.I, c.J), (c.I, c.J)]
        val = [None] * 6
        val[face] = np.asfortranarray(np.random.default_rng(7).uniform(-1.0, 1.0, dims[face]))
        print(f"[tail] size={size} levels={levels} prec={prec} face={face}", flush=True)
        ref = orc.project(c, pin=(1, 1, 1), bc_val=val, tol=1e-12, max_iter=3000)
        assert ref.stats.converged and not ref.singular
        P = H.projector(c, precision=prec, mg_levels=levels, max_iter=400)
        P.set_profiling(True)
        out, st = P.project(H.fields(c), c.bc_flag, c.dt, bc_val=val, po_coef=True)
        names = {k["name"] for k in P.kernel_times() if k["launches"]}
        P.close()
        assert ("mg_tail" in names) == (prec == 1 or size != (34, 34, 34)), names
        assert st.converged == 1, st.as_dict()
        H.assert_matches_oracle(c, out, st, ref)
