"""Tile shapes of the exact-footprint smearing (smc_set_tile_variant) and the
autotuner (smc_autotune): every shape gives bit-identical grids, so the
choice cannot move results; the event records differ at most by the order
of the centre-of-mass partial sums (relative 1e-12)."""
import numpy as np
import pytest

import parity_helpers as H

pytestmark = pytest.mark.gpu


def test_tile_variants_identical_and_autotune_picks_fastest():
    from supermc_amd import Context, SmcError
    p = H.glauber_params("PbPb", max_events=24)
    with Context(p) as ctx:
        ctx.run(seed=3, event0=0, nev=24, fetch=False)
        out = []
        for v in range(4):
            ctx.set_tile_variant(v)
            s, dndy, _ = ctx.density()
            ta, tb = ctx.thickness()
            out.append((s, dndy, ta, tb, ctx.moments()))
        for v in range(1, 4):
            for a, b in zip(out[v][:4], out[0][:4]):
                assert np.array_equal(a, b), v
            np.testing.assert_allclose(out[v][4][:, :54], out[0][4][:, :54], rtol=1e-12, atol=1e-14)
            assert np.array_equal(out[v][4][:, 54:58], out[0][4][:, 54:58])
        best, ms = ctx.autotune(reps=2)
        assert 0 <= best < 4 and (ms > 0).all() and ms[best] == ms.min()
        s2, _, _ = ctx.density()
        assert np.array_equal(s2, out[0][0])
        with pytest.raises(SmcError):
            ctx.set_tile_variant(4)


@pytest.mark.parametrize("model", ["glauber", "sqrt", "kln"])
@pytest.mark.parametrize("maxx,maxy", [(13.0, 13.0), (3.3, 0.8), (0.7, 6.4), (9.6, 3.1)])
@pytest.mark.parametrize("nev", [1, 5, 70])
def test_every_tile_shape_gives_the_cells_of_the_per_cell_path(model, maxx, maxy, nev):
    """One, four and sixteen waves per tile: bit-identical grids and records,
    on grids with partial tiles in both directions (67 x 17, 15 x 129, 193 x
    63 cells), batches below and above the spread and ordering limits, and
    central events whose lists take several rounds of each selection.  Against
    the per-cell exponentials (smear_path 2): FP32 rounding of at most 2,000
    terms per cell, below the paths' 1e-5 relative L-inf bar."""
    from supermc_amd import Context
    kw = dict(glauber={}, sqrt=dict(which_mc_model=7),
              kln=dict(which_mc_model=1, sub_model=7, ecm=2760.0, tmax=71, tmax_subdivision=3, kln_n_pt=8, kln_n_kt=8,
                       kln_n_phi=8))[model]
    kw = dict(kw, maxx=maxx, maxy=maxy, max_events=nev, bmax=12.0)
    grids = []
    for v in range(4):
        with Context(H.glauber_params("PbPb", **kw)) as ctx:
            ctx.set_tile_variant(v)
            ctx.sample(seed=5, event0=0, nev=nev)
            s, _, _ = ctx.density()
            grids.append((s, ctx.moments(), *ctx.thickness()))
    for v in range(1, 4):
        for a, b in zip(grids[v], grids[0]):
            assert np.array_equal(a, b, equal_nan=True), v
    with Context(H.glauber_params("PbPb", smear_path=2, **kw)) as ctx:
        ctx.sample(seed=5, event0=0, nev=nev)
        s, _, _ = ctx.density()
        ta, tb = ctx.thickness()
    for a, ref in zip((grids[0][0], *grids[0][2:]), (s, ta, tb)):
        assert ref.max() > 0
        assert H.rel_linf(a, ref) <= 1e-5
