"""Calls that would rather have more memory give the same results without it: tests/cpp/out_of_memory_example.cpp, built by
__graft_entry__.build(), refuses single allocations from the host (no memory is filled)."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu
BIN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "out_of_memory_example.bin")


@pytest.mark.parametrize("case", ["early_output", "pool_workspace", "slab"])
def test_results_without_the_memory_a_call_would_like(case):
    assert os.path.exists(BIN), "build it with __graft_entry__.build()"
    res = subprocess.run([BIN, case], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=100)
    assert res.returncode == 0, res.stderr
