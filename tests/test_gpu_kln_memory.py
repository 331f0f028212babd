"""The per-cell KLN quadrature without the memory for its breakpoint tables
(151 MB at 32 x 768 nodes): the node-by-node kernel gives the grids, and a
context stays with it.  In a process of its own, under a hipMalloc that
refuses large allocations (native/hip_refuse.cpp)."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))


def child():
    import ctypes as C
    refuse = C.CDLL(os.path.join(HERE, "native", "hip_refuse.so"), mode=C.RTLD_GLOBAL)
    import torch  # noqa: F401  (its HIP runtime, as in the other tests)
    refuse.refuse_init(C.cast(C.CDLL("libamdhip64.so.7").hipMalloc, C.c_void_p))
    import numpy as np
    sys.path[:0] = [os.path.dirname(HERE), os.path.join(os.path.dirname(HERE), "oracle"), HERE]
    import parity_helpers as H
    from supermc_amd import Context
    p = H.glauber_params("PbPb", which_mc_model=1, sub_model=7, ecm=2760.0, lambda_=0.138, kln_direct=1, max_events=2,
                         kln_n_pt=32, kln_n_kt=32, kln_n_phi=48)
    xa, xb, bs = H.cpu_configs(p, 2, seed=12, bvals=np.array([3.0, 12.0]))
    grids = []
    for refused in (True, False):
        with Context(p) as ctx:
            ctx.set_positions(xa, xb, bs)
            refuse.refuse_from(C.c_size_t(64 << 20 if refused else 2 ** 64 - 1))
            s, _, _ = ctx.density()
            assert (refuse.refuse_count() > 0), "nothing was refused"
            refuse.refuse_from(C.c_size_t(2 ** 64 - 1))
            count = refuse.refuse_count()
            ctx.set_positions(xa, xb, bs)
            again, _, _ = ctx.density()
            assert np.array_equal(again, s) and refuse.refuse_count() == count
            ta, tb = ctx.thickness()
            for e in range(2):
                ref = ctx.kln_dndy(ta[e].ravel().astype(np.float64), tb[e].ravel().astype(np.float64))
                assert ref.max() > 0 and H.rel_linf(s[e].ravel(), ref) <= 1e-5
            # graph capture allocates nothing whichever kernel the context has
            for seed in (1, 2, 3):
                rg = ctx.run_graph(seed, 0, 2)
                assert np.array_equal(rg, ctx.run(seed, 0, 2), equal_nan=True)
            grids.append(s)
    print("without tables", np.abs(grids[0] - grids[1]).max() / grids[1].max())


def test_density_without_memory_for_the_tables():
    if not os.path.exists(os.path.join(HERE, "native", "hip_refuse.so")):
        pytest.fail("tests/native/hip_refuse.so not built: run python -m supermc_amd.build")
    r = subprocess.run([sys.executable, os.path.abspath(__file__)], capture_output=True, text=True, timeout=110)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "without tables" in r.stdout


if __name__ == "__main__":
    child()
