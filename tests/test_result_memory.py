"""The memory results are handed out in: never handed out again while a caller can still see it, however the
interpreter counts references."""
import gc
import sys

import numpy as np
import pytest

from tpu_compiler_amd.pymodule import _ResultMemory

SHAPE = (3, 300, 100)


def _held(out, how):
    return {"array": lambda: out, "row of a slice": lambda: out[1:][0], "transposed bytes": lambda: out.T.view(np.int32),
            "memoryview": lambda: memoryview(out), "inside a container": lambda: {"y": [out]}}[how]()


@pytest.mark.parametrize("how", ["array", "row of a slice", "transposed bytes", "memoryview", "inside a container"])
@pytest.mark.parametrize("uncounted", [0, 1, 2, 3])
def test_a_held_result_is_not_handed_out_again(monkeypatch, how, uncounted):
    count = sys.getrefcount      # interpreters that borrow locals or arguments count that many fewer
    monkeypatch.setattr(sys, "getrefcount", lambda o: count(o) - uncounted)
    memory = _ResultMemory()
    memory.take(SHAPE, np.float32)
    out, address = memory.take(SHAPE, np.float32)
    assert out.shape == SHAPE and out.dtype == np.float32 and out.flags.writeable and out.flags.c_contiguous
    assert out.ctypes.data == address
    held = _held(out, how)
    del out
    others = [memory.take(SHAPE, np.float32) for _ in range(3)]
    assert len({address} | {a for _, a in others}) == 4
    del held, others
    gc.collect()


def test_dropped_memory_is_used_again_and_bounded(monkeypatch):
    memory = _ResultMemory()
    memory.take(SHAPE, np.int8)                    # the first of a shape is the caller's alone
    out, address = memory.take(SHAPE, np.int8)
    out[:] = 7
    del out
    again, second = memory.take(SHAPE, np.int8)
    assert second == address
    monkeypatch.setattr(_ResultMemory, "LIMIT", 4 * again.nbytes)
    kept = [memory.take(SHAPE, np.int8) for _ in range(6)]
    assert memory._bytes <= 4 * again.nbytes and len({a for _, a in kept} | {second}) == 7
    memory.clear()                                 # what a caller holds stays the caller's
    again[:] = 9
    more = [memory.take(SHAPE, np.int8) for _ in range(3)]
    for m, _ in more:
        m[:] = 1
    assert (again == 9).all()
