"""MFMA smearing of short and full source groups: nuclei of 1 to 40 nucleons
at small b give events of one source up to several groups of 32, on grids
whose tiles end inside a wave's 32 x 64 cells.  Against the VALU tiles (the
exact footprint): FP32 and BF16x6 at the parity bar 1e-5, BF16x3 at 3 * 2^-16
per term more."""
import numpy as np
import pytest

import parity_helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("A", [1, 5, 9, 17, 40])
@pytest.mark.parametrize("path,bar", [(1, 1e-5), (4, 1e-5), (3, 1e-5 + 3 * 2.0 ** -16)])
def test_groups_match_valu_tiles(A, path, bar):
    from supermc_amd import Context
    nev = 24
    rng = np.random.default_rng(A)
    xa, xb = (np.round(rng.normal(0.0, 1.2, (nev, A, 2)) * 2 ** 24) / 2 ** 24 for _ in range(2))
    got = []
    for p in (0, path):
        with Context(H.glauber_params("AuAu", Aproj=A, Atarg=A, max_events=nev, maxx=6.45, maxy=4.8, dx=0.1, dy=0.075,
                                      Npmin=0, smear_path=p)) as ctx:
            ctx.set_positions(xa, xb, np.zeros(nev))
            got.append(ctx.density()[0])
    assert got[0].any()
    for e in range(nev):
        assert np.abs(got[1][e] - got[0][e]).max() <= bar * got[0][e].max()
