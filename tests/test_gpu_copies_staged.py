"""Copies large enough to make the pinned slots: records of a 20 MB batch
against the same events fetched a part at a time, and grids."""
import numpy as np
import pytest
import torch

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


@pytest.mark.parametrize("nev", [90, 103])
def test_grids_through_the_slots(nev):
    """FP64 grids of 49 and 56 MB into memory that was written before, whose
    last piece is a partial one, and FP32 grids after them, at an odd offset:
    the bytes of the copies into page-locked memory, and none beside them."""
    from supermc_amd import Context
    with Context(H.glauber_params("PbPb", max_events=nev)) as ctx:
        ctx.sample(seed=9, event0=0, nev=nev)
        n = nev * ctx.nx * ctx.ny
        for call, dt, tdt in ((lambda out: ctx.density_f64(out=out), np.float64, torch.float64),
                              (lambda out: ctx.density(out=out), np.float32, torch.float32)):
            pin = torch.empty(n, dtype=tdt, pin_memory=True).numpy().reshape(nev, ctx.nx, ctx.ny)
            page = np.full(n + 3, -1, dt)
            call(pin)
            call(page[1:n + 1].reshape(nev, ctx.nx, ctx.ny))
            assert np.array_equal(page[1:n + 1], pin.ravel())
            assert page[0] == -1 and (page[n + 1:] == -1).all()
