"""The event sums of operation 3 at the edges of their layout: rows of 63,
64, 65 and 129 cells, row counts that are no multiple of 4, segments of one
event, of 64 and of more, every event or a few of them accepted; against a
host FP64 sum of the same turned grids (1e-12: the same terms, the segments
added in another order)."""
import numpy as np
import pytest

import parity_helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("maxx,maxy,nev,every", [
    (3.1, 3.1, 20, 1),      # 63 x 63
    (3.2, 3.15, 2048, 3),   # 65 x 64 (dy 0.1), segments of 64
    (6.4, 3.2, 2100, 1),    # 129 x 65, segments of 66
    (3.15, 6.4, 33, 5),     # 64 x 129, segments of 2
])
def test_sums(maxx, maxy, nev, every):
    from supermc_amd import Context
    p = H.glauber_params("PbPb", max_events=nev, maxx=maxx, maxy=maxy, finalFactor=1.3)
    with Context(p) as ctx:
        ctx.run(seed=3, event0=0, nev=nev, fetch=False)
        accept = (np.arange(nev) % every == 0).astype(np.uint8)
        sums = ctx.average_profiles(2, 2, accept=accept)
        rho, _, _ = ctx.density()  # the grids are left turned by the order-2 angle
    ref = p.finalFactor * rho[accept == 1].astype(np.float64).sum(axis=0)
    np.testing.assert_allclose(sums[0], ref, rtol=1e-12, atol=1e-12 * np.abs(ref).max())
