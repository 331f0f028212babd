"""One 3D-profile handle under several threads: its source lists and grids
are kept from call to call, so calls have to take turns."""
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
