"""Edges of the differentiable batch's kernels: the gather over windows of
every width (3 columns, more than 256 columns and 64 rows, clipped by the
grid or empty) and repeated calls.

Bars: gradients as in test_gpu_adjoint (1e-4 relative per component against
the FP64 adjoint, components below 1e-3 of the largest against that);
repeated calls bit for bit."""
import numpy as np
import pytest

import diff_oracle as D
import parity_helpers as H

pytestmark = pytest.mark.gpu

COT = np.array([1.0, 1.0, 0.01])


@pytest.mark.parametrize("maxx,maxy,dx,dy,w", [
    (13.0, 13.0, 0.1, 0.1, 0.5),   # 40 or 41 and 50 or 51 cells
    (13.0, 13.0, 1.3, 1.3, 0.5),   # 3 and 4 cells
    (6.0, 6.0, 0.02, 0.02, 0.6),   # up to 300 columns and rows, clipped
    (4.0, 2.5, 0.1, 0.08, 0.5),    # clipped and empty windows, 63 columns
])
def test_gather_windows(maxx, maxy, dx, dy, w):
    from supermc_amd import Context
    nev = 2
    with Context(H.glauber_params("PbPb", max_events=nev, maxx=maxx, maxy=maxy, dx=dx, dy=dy, gauss_nucl_width=w,
                                  bmax=7.0)) as ctx:
        th = ctx.diff_setup(seed=5, event0=0, nev=nev)
        evs = [D.event_from_context(ctx, e) for e in range(nev)]
        ctx.diff_forward(th)
        g = ctx.diff_backward(np.tile(COT, (nev, 1)))
        ref = sum(ev.adjoint(th, COT) for ev in evs)
        scale = np.abs(ref).max()
        for q in range(5):
            assert abs(g[q] - ref[q]) <= 1e-4 * max(abs(ref[q]), 1e-3 * scale), (q, g[q], ref[q])


def test_repeated_calls_agree_to_the_bit():
    from supermc_amd import Context
    nev = 200
    with Context(H.glauber_params("PbPb", max_events=nev)) as ctx:
        th = ctx.diff_setup(seed=9, event0=0, nev=nev)
        first = None
        for _ in range(5):
            out = ctx.diff_forward(th)
            g = ctx.diff_backward(np.tile(COT, (nev, 1)))
            if first is None:
                first = out, g
            np.testing.assert_array_equal(out, first[0])
            np.testing.assert_array_equal(g, first[1])


@pytest.mark.parametrize("k", [0.1, 0.8, 5.0, 30.0])
def test_gamma_quantiles(k):
    """Shapes with and without a quantile table (pairs at k = 0.1: 0.014) up
    to 13: forward and gradient against FP64 at test_gpu_adjoint's bars."""
    from supermc_amd import Context
    nev = 2
    with Context(H.glauber_params("PbPb", max_events=nev)) as ctx:
        th = ctx.diff_setup(seed=21, event0=0, nev=nev)
        evs = [D.event_from_context(ctx, e) for e in range(nev)]
        th = np.array([*th[:4], k])
        out = ctx.diff_forward(th)
        g = ctx.diff_backward(np.tile(COT, (nev, 1)))
        for e, ev in enumerate(evs):
            ref = ev.forward(th)
            assert abs(out[e, 0] - ref[0]) <= 1e-6 and abs(out[e, 1] - ref[1]) <= 1e-6
            assert out[e, 2] == pytest.approx(ref[2], rel=1e-5)
        ref = sum(ev.adjoint(th, COT) for ev in evs)
        scale = np.abs(ref).max()
        for q in range(5):
            assert abs(g[q] - ref[q]) <= 1e-4 * max(abs(ref[q]), 1e-3 * scale), (q, g[q], ref[q])
