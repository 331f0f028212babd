"""Grids and records copied into ordinary memory (worker threads through
pinned slots from 4 MiB on) equal the copies into page-locked memory, byte
for byte."""
import numpy as np
import pytest
import torch

import parity_helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nev", [1, 15, 16, 23, 40])
def test_pageable_grids_equal_pinned_ones(nev):
    """261^2 FP32 grids: 15 events are just below 4 MiB, 16 above, 23 end in a
    partial piece; FP64 grids twice that.  Destinations at odd offsets."""
    from supermc_amd import Context
    with Context(H.glauber_params("PbPb", max_events=nev)) as ctx:
        ctx.sample(seed=9, event0=0, nev=nev)
        n = nev * ctx.nx * ctx.ny
        for call, dt, tdt in ((ctx.density, np.float32, torch.float32),
                              (lambda out: (ctx.density_f64(out=out),), np.float64, torch.float64)):
            pin = torch.empty(n, dtype=tdt, pin_memory=True).numpy().reshape(nev, ctx.nx, ctx.ny)
            page = np.full(n + 3, -1, dt)
            call(out=pin)
            call(out=page[1:n + 1].reshape(nev, ctx.nx, ctx.ny))
            assert np.array_equal(page[1:n + 1], pin.ravel())
            assert page[0] == -1 and (page[n + 1:] == -1).all()


def test_records_of_a_large_batch_equal_fetched_ones():
    """9,000 records are 4.6 MB: run's copy, a second fetch and a stream in
    batches that do not divide the total give the same bytes."""
    from supermc_amd import Context
    with Context(H.glauber_params("AuAu", max_events=9000)) as ctx:
        a = ctx.run(seed=4, event0=0, nev=9000)
        assert np.array_equal(a, ctx.fetch_events(9000))
    with Context(H.glauber_params("AuAu", max_events=8300)) as ctx:
        assert np.array_equal(a, ctx.run_stream(seed=4, event0=0, nev_total=9000))
