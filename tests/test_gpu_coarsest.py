"""Multigrid hierarchies with a large coarsest level: a hierarchy cut short by
mg_levels, and a grid too thin to coarsen.  The tail kernel holds it up to two
pairs of cells per thread (2048 pairs) in FP64 and four in FP32; beyond that
it is smoothed in global memory (the tail's coarsest sweeps with the plain
red-black kernels).  Bar: the parity bars of the oracle comparison
(PoCoef bit-identical, pressure and corrected velocity within 1e-8) and
convergence to max |div u| <= 1e-10, both precisions."""

import numpy as np
import pytest

from oracle import orc
from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", (0, 1))
@pytest.mark.parametrize("size,levels", [
    ((48, 40, 32), 2),  # coarsest 24x20x16: 3840 pairs, outside the tail in FP64
    ((64, 3, 40), 0),   # J = 3 does not coarsen: one level of 3840 pairs
    ((40, 40, 3), 0),   # one level of 2400 pairs
])
def test_coarsest_level_outside_the_tail(gpu_available, size, levels, prec):
    print(f"[coarsest] size={size} mg_levels={levels} precision={prec}", flush=True)
    c = H.case(0, size=size)
    out, st = H.run_engine(c, prec, mg_levels=levels)
    assert st.converged == 1, st.as_dict()
    assert st.final_div <= 1e-10
    ref = orc.project(c, pin=(1, 1, 1))
    H.assert_matches_oracle(c, out, st, ref)


def _walls(c, dirichlet):
    """Pressure walls: all Neumann, or one Dirichlet face with values."""
    if dirichlet is None:
        return None
    I, J, K = c.shape
    c.bc_flag[dirichlet] = 0
    n = [(J, K), (J, K), (I, K), (I, K), (I, J), (I, J)][dirichlet]
    val = [None] * 6
    val[dirichlet] = np.asfortranarray(np.random.default_rng(21).uniform(-2.0, 2.0, n))
    return val


@pytest.mark.parametrize("dirichlet", (None, 1, 2))
@pytest.mark.parametrize("size,levels,prec,tail", [
    ((40, 40, 3), 0, 1, True), ((50, 50, 2), 0, 1, True),
    ((3, 32, 33), 0, 1, True),   # 2112 pairs: one row of three cells takes two
    ((2, 32, 64), 0, 1, True),   # 2048 pairs: two per thread
    ((2, 33, 63), 0, 1, True),   # 2079
    ((2, 64, 64), 0, 1, True),   # 4096: four per thread
    ((2, 64, 65), 0, 1, False),  # 4160
    ((18, 19, 17), 1, 1, True), ((36, 37, 33), 2, 1, True),
    ((2, 32, 64), 0, 0, True), ((2, 33, 63), 0, 0, False)])
def test_coarsest_level_of_up_to_four_pairs_per_thread(gpu_available, size, levels, prec, tail,
                                                       dirichlet):
    """A coarsest FP32 level runs in the tail up to 4096 pairs of cells, an
    FP64 one up to 2048; with and without a diagonal-only term.  The oracle
    runs one solve to a hundredth of the engine's stop (its search for the
    rounding floor gives up early on grids this thin)."""
    print(f"[coarsest] size={size} mg_levels={levels} prec={prec} dirichlet={dirichlet}", flush=True)
    c = H.case(0, size=size)
    bcv = _walls(c, dirichlet)
    ref = orc.project(c, pin=(1, 1, 1), bc_val=bcv, tol=1e-12, max_iter=3000)
    assert ref.stats.converged
    P = H.projector(c, precision=prec, mg_levels=levels, max_iter=400)
    P.set_profiling(True)
    out, st = P.project(H.fields(c), c.bc_flag, c.dt, bc_val=bcv, po_coef=True)
    names = {k["name"] for k in P.kernel_times() if k["launches"]}
    P.close()
    assert ("mg_tail" in names) == tail, names
    assert st.converged == 1, st.as_dict()
    H.assert_matches_oracle(c, out, st, ref)
