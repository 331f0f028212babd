"""Records through the pinned slots: a batch of 20 MB, whose copy is large
enough to make them, against the same events fetched a part at a time."""
import numpy as np
import pytest

import parity_helpers as H

pytestmark = pytest.mark.gpu


def test_records_through_the_slots():
    from supermc_amd import Context
    nev, part = 40001, 3000
    with Context(H.glauber_params("AuAu", max_events=nev)) as ctx:
        a = ctx.run(seed=4, event0=0, nev=nev)
        assert np.array_equal(a, ctx.fetch_events(nev))
    with Context(H.glauber_params("AuAu", max_events=part)) as ctx:  # 1.5 MB: never staged
        for e in range(0, nev, 4 * part):
            n = min(part, nev - e)
            assert np.array_equal(a[e:e + n], ctx.run(seed=4, event0=e, nev=n))
