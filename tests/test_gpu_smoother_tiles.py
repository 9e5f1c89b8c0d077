"""The fused smoother legs at the edges of their tiles: rows of every length
modulo the four cells of a thread, grids one cell around the tile interiors
and around the limits between the tile sizes, one and two sweeps."""

import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu

SIZES = [(111, 113, 6), (113, 112, 7), (63, 66, 9), (64, 64, 12), (65, 64, 10), (66, 65, 7), (67, 66, 8), (64, 65, 17),
         (127, 33, 6), (129, 49, 5), (9, 17, 130)]


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("prec", (0, 1))
@pytest.mark.parametrize("sweeps", (1, 2))
def test_legs_match_plain_sweeps(gpu_available, size, prec, sweeps):
    """Same V-cycle as one kernel per half-sweep (SP_FLAG_UNFUSED_SMOOTHER),
    there with the flexible CG.  These flat grids take up to 300 iterations,
    whose count rounding alone moves by 3 %; the pressures agree to what the
    stop at max |div u| <= 1e-10 leaves (bound of the existing comparison)."""
    c = H.case(4 if size[2] < size[0] else 1, size=size, seed=3)
    print(f"[tiles] size={size} prec={prec} sweeps={sweeps}", flush=True)
    res = []
    for flags in (0, 1):
        P = H.projector(c, precision=prec, flags=flags, mg_pre=sweeps, mg_post=sweeps,
                        max_iter=400)
        out, st = P.project(H.fields(c), c.bc_flag, c.dt)
        P.close()
        assert st.converged == 1
        res.append((out, st))
    (a, sa), (b, sb) = res
    assert abs(sa.iterations - sb.iterations) <= max(1, 0.05 * sb.iterations)
    assert np.max(np.abs(a["p"] - b["p"])) <= 1e-9 * np.max(np.abs(b["p"]))
