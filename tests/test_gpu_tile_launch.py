"""Tile shapes on a batch whose sixteen-wave launch would need more than 2^32
work-items (100,000 events of 45 tiles): the same records as by default."""
import numpy as np
import pytest

import parity_helpers as H

pytestmark = pytest.mark.gpu


def test_shapes_of_a_large_batch():
    from supermc_amd import Context
    nev = 100000
    with Context(H.glauber_params("AuAu", Aproj=1, Atarg=1, max_events=nev, max_pairs=16, bmax=1.0)) as ctx:
        out = []
        for v in range(4):
            ctx.set_tile_variant(v)
            out.append(ctx.run(seed=2, event0=0, nev=nev))
    assert (out[0][:, 57] == 0).all()
    for r in out[1:]:
        np.testing.assert_allclose(r, out[0], rtol=1e-12, atol=1e-14)
