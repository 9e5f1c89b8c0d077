"""The CG's product and update on both sides of the limit between short and
long columns (four workgroups per CU: 960 and 1024 workgroups of the long
form here), with remainders of both lengths."""

import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(9, 255, 239), (9, 255, 241), (5, 3, 2), (65, 5, 17)])
def test_columns(gpu_available, size):
    """The recursive residual that k_cg_update leaves is checked against the
    true one, formed by another kernel, before a solve counts as converged;
    a wrong product or update ends in restarts.  FP64 and FP32 V-cycles agree to
    what the stop at max |div u| <= 1e-10 leaves (bound of the comparison of the
    smoother legs)."""
    c = H.case(1, size=size, seed=5)
    print(f"[columns] size={size}", flush=True)
    res = []
    for prec in (0, 1):
        P = H.projector(c, precision=prec, max_iter=400)
        out, st = P.project(H.fields(c), c.bc_flag, c.dt)
        P.close()
        assert st.converged == 1
        res.append((out, st))
    (a, sa), (b, sb) = res
    assert abs(sa.iterations - sb.iterations) <= max(2, 0.1 * sb.iterations)
    assert np.max(np.abs(a["p"] - b["p"])) <= 1e-9 * np.max(np.abs(b["p"]))
