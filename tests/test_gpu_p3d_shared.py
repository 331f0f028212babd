"""One 3D-profile handle under several threads, and with more events than the
grid buffer it keeps: its source lists and grids are kept from call to call."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_threads_share_a_handle():
    """Four threads with lists of other lengths each, through generate, sample
    and smear at once, get what the same calls give one after the other."""
    from supermc_amd import Profile3D
    rng = np.random.default_rng(31)

    def lists(k):
        sizes = rng.integers(0, 60 * (k + 1), 3)
        return ([np.column_stack([rng.uniform(-5, 5, (n, 2)), rng.integers(1, 3, n)]) for n in sizes],
                [rng.uniform(-4, 4, (n, 2)) for n in sizes[::-1]])

    jobs = [lists(k) for k in range(4)]
    with Profile3D(grid_nx=61, grid_ny=61, grid_neta=21, ecm=200.0, random_flag=3) as P:
        def job(k):
            parts, bins = jobs[k]
            got = list(P.generate(parts, bins, seed=k, event0=k))
            ps, bs = P.sample(parts, bins, seed=k, event0=k)
            return got + [np.concatenate(ps), np.concatenate(bs), P.smear(ps)]

        alone = [job(k) for k in range(4)]
        with ThreadPoolExecutor(4) as pool:
            for _ in range(5):
                for k, got in enumerate(pool.map(job, range(4))):
                    for a, b in zip(got, alone[k]):
                        assert np.array_equal(a, b), k


def test_more_events_than_the_grid_buffer_holds():
    """Reference grids of 27.5 MB, nine to the kept buffer: 20 events with
    unequal and empty lists go through it in three parts and equal the same
    events one at a time; then a smaller and a larger call on the handle."""
    from supermc_amd import Profile3D
    rng = np.random.default_rng(32)
    sizes = [0, 70, 3, 0, 41, 1, 120, 8, 0, 0, 55, 2, 17, 0, 90, 6, 33, 1, 0, 25]
    parts = [np.column_stack([rng.uniform(-6, 6, (n, 2)), rng.integers(1, 3, n)]) for n in sizes]
    bins = [rng.uniform(-5, 5, (n, 2)) for n in sizes[::-1]]
    with Profile3D(ecm=200.0, random_flag=2) as P:
        one = [P.generate(parts[e:e + 1], bins[e:e + 1], seed=5, event0=e) for e in range(20)]
        for e0, e1 in ((0, 20), (6, 8), (1, 19)):
            rp, rb, ps, bs = P.generate(parts[e0:e1], bins[e0:e1], seed=5, event0=e0)
            for e in range(e0, e1):
                assert np.array_equal(rp[e - e0], one[e][0][0]) and np.array_equal(rb[e - e0], one[e][1][0]), e
            assert np.array_equal(ps, np.concatenate([o[2] for o in one[e0:e1]]))
            assert np.array_equal(bs, np.concatenate([o[3] for o in one[e0:e1]]))
        assert all(o[0].any() == (n > 0) for o, n in zip(one, sizes))
