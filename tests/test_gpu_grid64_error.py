"""Rounding of the FP64 density grids against sums of the same sources in
80-bit arithmetic.

Bar: participants and pairs summed one after the other in FP64, in sums of
their own.  Rounding to a spacing d leaves d / sqrt(12) in the mean square.
An addition rounds to the spacing of its partial sum S, a term t to its own
about twice (two exponentials to less than an ulp and a product), so a
cell's error has the variance sigma^2 = (sum spacing(S)^2 + 2 sum
spacing(t)^2) / 12; the errors of all cells together may be 1.25 sigma.  One
sum through participants and pairs has about 1.8."""
import numpy as np
import pytest

import parity_helpers as H

pytestmark = pytest.mark.gpu

LD = np.longdouble


def ulp2(x):
    return np.spacing(x.astype(np.float64)) ** 2


def sums80(p, w, nuc, pairs, nx, ny):
    """The grid in 80 bits and each cell's sigma."""
    xs, ys = -p.maxx + np.arange(nx) * p.dx, -p.maxy + np.arange(ny) * p.dy
    norm = 1 / (2 * LD("3.14159265358979323846264338327950288") * LD(w) ** 2)
    total, var = np.zeros((nx, ny), LD), np.zeros((nx, ny))
    ones = [nuc["xy_" + s][nuc["wound_" + s] >= 0] for s in ("proj", "targ")]
    mid = (nuc["xy_proj"][pairs[0]] + nuc["xy_targ"][pairs[1]]) / 2
    for xy, weight, half in ((np.concatenate(ones), (1 - LD(p.alpha)) / 2, 4 * max(w, p.quark_width)),
                             (mid, LD(p.alpha), 5 * w)):
        part = np.zeros((nx, ny), LD)
        for x, y in xy:
            x0, x1 = (int(np.clip(int((x + d + p.maxx) / p.dx), 0, nx)) for d in (-half, half))
            y0, y1 = (int(np.clip(int((y + d + p.maxy) / p.dy), 0, ny)) for d in (-half, half))
            dx, dy = xs[x0:x1] - x, ys[y0:y1] - y
            gx, gy = (np.exp(-d.astype(LD) ** 2 / (2 * LD(w) ** 2)) for d in (dx, dy))
            t = np.where(dx[:, None] ** 2 + dy[None] ** 2 <= 25.0 * w * w, weight * norm * gx[:, None] * gy[None], 0)
            part[x0:x1, y0:y1] += t
            var[x0:x1, y0:y1] += np.where(t > 0, ulp2(part[x0:x1, y0:y1]) + 2 * ulp2(t), 0)
        total += part
    return total, np.sqrt((var + ulp2(total)) / 12)


@pytest.mark.parametrize("w", [0.35, 0.5, 0.8])
def test_rounding_of_central_events(w):
    from supermc_amd import Context
    p = H.glauber_params("PbPb", max_events=2, cc_fluctuation_model=0, gauss_nucl_width=w)
    xa, xb, bs = H.cpu_configs(p, 2, seed=3, bvals=np.array([0.0, 2.0]))
    with Context(p) as ctx:
        ctx.set_positions(xa, xb, bs)
        s = ctx.density_f64()
        for e in range(2):
            ref, sigma = sums80(p, w, ctx.nucleons(e), ctx.pairs(e)[:2], ctx.nx, ctx.ny)
            err = (s[e] - ref).astype(np.float64)
            assert np.abs(err).max() <= 1e-14 * float(ref.max())  # the same cells
            assert np.sqrt((err ** 2).sum()) <= 1.25 * np.sqrt((sigma ** 2).sum())
