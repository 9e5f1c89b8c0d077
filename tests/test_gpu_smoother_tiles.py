"""The fused smoother legs at the edges of their tiles: grids one cell around
the tile interiors and around the limits between the tile sizes, one and two
sweeps, closed and with a Dirichlet wall (a diagonal-only term).  SIZES take
one cell per thread in FP32; FOUR and FOUR_1 (one sweep) or FOUR_2 (two) take
four there (test_leg_rule.py), with rows of every length modulo four, odd and
even numbers of rows and planes."""

import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu

SIZES = [(111, 113, 6), (113, 112, 7), (63, 66, 9), (64, 64, 12), (65, 64, 10), (66, 65, 7), (67, 66, 8), (64, 65, 17),
         (127, 33, 6), (129, 49, 5), (9, 17, 130)]

FOUR = [(127, 111, 70), (191, 97, 61), (61, 114, 200), (190, 65, 131), (193, 64, 129),
        (126, 129, 101), (63, 98, 250), (192, 97, 141), (257, 100, 101)]
FOUR_1 = [(192, 97, 90)]
FOUR_2 = [(129, 113, 80), (65, 97, 251), (194, 81, 75)]


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


def _both(c, prec, sweeps, bc_val=None):
    """The same projection with fused legs and with one kernel per half-sweep."""
    res = []
    for flags in (0, 1):
        P = H.projector(c, precision=prec, flags=flags, mg_pre=sweeps, mg_post=sweeps,
                        max_iter=400)
        out, st = P.project(H.fields(c), c.bc_flag, c.dt, bc_val=bc_val)
        P.close()
        assert st.converged == 1
        res.append((out, st))
    return res


@pytest.mark.parametrize("size,sweeps", [(s, w) for s in FOUR for w in (1, 2)] +
                         [(s, 1) for s in FOUR_1] + [(s, 2) for s in FOUR_2])
def test_four_cell_legs_match_plain_sweeps(gpu_available, size, sweeps):
    """FP32, bounds of the test above; grids of at most about four to one, whose
    count (30 to 130) is far from the rounding floor: flatter ones stagnate at
    the stop in both forms and at times do not reach it in 400 iterations."""
    c = H.case(0, size=size, seed=3)
    print(f"[tiles] four cells size={size} sweeps={sweeps}", flush=True)
    (a, sa), (b, sb) = _both(c, 1, sweeps)
    assert abs(sa.iterations - sb.iterations) <= max(1, 0.05 * sb.iterations)
    assert np.max(np.abs(a["p"] - b["p"])) <= 1e-9 * np.max(np.abs(b["p"]))


@pytest.mark.parametrize("size", SIZES + [(126, 113, 9), (33, 130, 11)])
@pytest.mark.parametrize("prec", (0, 1))
@pytest.mark.parametrize("sweeps", (1, 2))
def test_legs_with_a_diagonal_only_term(gpu_available, size, prec, sweeps):
    """A pressure outlet on the east face.  Iterations are not compared: the
    count includes the refinement that only one of the two may need."""
    c = H.case(4 if size[2] < size[0] else 1, size=size, seed=3)
    c.bc_flag[1] = 0
    val = [None, np.zeros((c.J, c.K), order="F")] + [None] * 4
    print(f"[tiles] outlet size={size} prec={prec} sweeps={sweeps}", flush=True)
    (a, _), (b, _) = _both(c, prec, sweeps, val)
    assert np.max(np.abs(a["p"] - b["p"])) <= 1e-9 * np.max(np.abs(b["p"]))
