"""Smearing of light collision systems, whose source lists are short: the
shape chosen for the batch, and the cells of every shape at batch sizes around
the limits of that choice."""
import numpy as np
import pytest

import parity_helpers as H

pytestmark = pytest.mark.gpu

PB = dict(targ_ws_R=6.62, targ_ws_a=0.546)
SYSTEMS = {"pPb": dict(Aproj=1, Atarg=208, **PB), "dAu": dict(Aproj=2, Atarg=197, targ_ws_R=6.38, targ_ws_a=0.535),
           "NeNe": dict(Aproj=20, Atarg=20, proj_ws_R=3.04, proj_ws_a=0.54, targ_ws_R=3.04, targ_ws_a=0.54)}


def _context(system, nev, **kw):
    from supermc_amd import Context
    return Context(H.glauber_params("PbPb", **dict(SYSTEMS[system], max_events=nev, bmax=8.0, **kw)))


@pytest.mark.parametrize("system", ["pPb", "dAu"])
@pytest.mark.parametrize("nev", [200, 1000])
def test_chosen_shape_is_near_the_fastest(system, nev):
    """The time of shape 0 against the fastest of the fixed ones.  Bar 1.6:
    means of 40 launches of 20 to 60 us repeat to a tenth, and sixteen
    waves take 2.8 times as long as four at 200 events."""
    with _context(system, nev) as ctx:
        ctx.sample(seed=5, event0=0, nev=nev)
        ctx.autotune(reps=40)
        ctx.set_tile_variant(0)
        _, ms = ctx.autotune(reps=40)
    assert ms[0] <= 1.6 * min(ms[1:]), ms


@pytest.mark.parametrize("system", list(SYSTEMS))
@pytest.mark.parametrize("nev", [15, 16, 200, 201, 450])
def test_every_shape_gives_the_same_cells(system, nev):
    got = []
    with _context(system, nev) as ctx:
        ctx.sample(seed=7, event0=0, nev=nev)
        for v in range(4):
            ctx.set_tile_variant(v)
            got.append((ctx.density()[0], ctx.moments()))
    assert got[0][0].any()
    for s, ev in got[1:]:
        assert np.array_equal(s, got[0][0]) and np.array_equal(ev, got[0][1], equal_nan=True)
