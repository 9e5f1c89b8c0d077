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
