"""The locator's index and memory, on the CPU against stubs of the runtime:
whichever of its allocations fails, the search falls back to the full one (it
does not fail), and giving the index back frees all of it."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = "/opt/rocm/include"


@pytest.mark.skipif(not os.path.isdir(ROCM), reason="no HIP headers")
def test_every_allocation_may_fail(tmp_path):
    exe = str(tmp_path / "index_memory")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__",
                    "-isystem", ROCM, "-o", exe,
                    os.path.join(ROOT, "tests", "index_memory_check.cpp")],
                   check=True)
    out = [int(v) for v in subprocess.run(
        [exe], check=True, capture_output=True, text=True).stdout.split()]
    first, calls = out[:2]
    assert first == 0 and calls > 10
    assert out[2:2 + calls] == [1] * calls
    # afterwards a search works; the index is given back whole, once
    assert out[2 + calls:] == [0, 1, 0, 0]
