"""Records of a large batch are the same to the bit in every tile shape: the
centre-of-mass sums follow row order whatever the number of waves, and a shape
whose launch would need 2^32 work-items gives way to a smaller one."""
import numpy as np
import pytest

import parity_helpers as H

pytestmark = pytest.mark.gpu


def test_records_of_every_shape():
    from supermc_amd import Context
    nev = 100000
    with Context(H.glauber_params("AuAu", Aproj=1, Atarg=1, max_events=nev, max_pairs=16, bmax=1.0)) as ctx:
        out = []
        for v in range(4):
            ctx.set_tile_variant(v)
            out.append(ctx.run(seed=2, event0=0, nev=nev))
    assert (out[0][:, 57] == 0).all()
    for r in out[1:]:
        assert np.array_equal(r, out[0], equal_nan=True)
