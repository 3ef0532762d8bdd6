"""Kernels with more than 64 KB of LDS on a second device of the process: tests/cpp/lds_limit_devices.cpp, built by
__graft_entry__.build(), stands in for the runtime calls, so no device is needed."""
import os
import subprocess

BIN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "lds_limit_devices.bin")


def test_the_limit_is_raised_on_every_device():
    assert os.path.exists(BIN), "build it with __graft_entry__.build()"
    res = subprocess.run([BIN], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=100)
    assert res.returncode == 0, res.stderr
