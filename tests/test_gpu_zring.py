"""The iterate formed from the kept preconditioned residuals (a ring of 16):
a solve stopped after m steps must return the x that its recursive residual
belongs to, on both sides of every ring boundary."""

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
