"""Calls that would rather have more memory, or threads, give the same results without them:
tests/cpp/doing_without_example.cpp, built by __graft_entry__.build(), refuses them from the host (no memory is filled)."""
import os
import subprocess

import pytest

from tpu_compiler_amd import graphs, mlir_text

pytestmark = pytest.mark.gpu
BIN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "doing_without_example.bin")


def _run(*args):
    assert os.path.exists(BIN), "build it with __graft_entry__.build()"
    res = subprocess.run([BIN] + [str(a) for a in args], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=100)
    assert res.returncode == 0, res.stderr


@pytest.mark.parametrize("case", ["early_output", "pool_workspace", "slab"])
def test_results_without_the_memory_a_call_would_like(case):
    _run(case)


def test_several_results_without_room_for_their_dense_forms_together():
    _run("many_results")


def test_results_without_threads(tmp_path):
    path = tmp_path / "model.mlir"
    mlir_text.write_mlir(graphs.cfg3_resnet50(batch=1, hw=64), path)
    _run("threads", path)
