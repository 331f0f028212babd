"""The host side of the copies into ordinary memory (smc_copy.cpp), by a
program that runs it on the CPU (native/copy_check.cpp)."""
import os
import subprocess

import pytest

CHECK = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "copy_check.bin")


@pytest.mark.parametrize("name", ["memcpy", "allocations", "slots", "first"])
def test_copies(name):
    if not os.path.exists(CHECK):
        pytest.fail(f"{CHECK} not built: run python -m supermc_amd.build")
    r = subprocess.run([CHECK, name], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
