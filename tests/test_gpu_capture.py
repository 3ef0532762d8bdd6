"""HIP graphs recorded from a module's or a context's stream: replays give what plain calls give, whatever is called in
between, and what cannot be recorded is refused."""
import numpy as np
import pytest

from gpu_capture import Graph
from tpu_compiler_amd import capi, graphs, module

pytestmark = pytest.mark.gpu


def _two_outputs(shape):
    """"first" is complete before the last kernel, and large enough to be read early"""
    g = graphs.Graph("early", 1)
    g.add(graphs.Op("tpu.input", "x", [], shape))
    g.add(graphs.Op("tpu.relu", "first", ["x"], shape))
    g.add(graphs.Op("tpu.upsample", "second", ["x"], shape[:2] + (2 * shape[2], 2 * shape[3]), dict(scale_h=2, scale_w=2)))
    g.outputs = ["first", "second"]
    m = module()
    m.load(g)
    return m


@pytest.mark.parametrize("all_batch", [False, True])
def test_results_of_replays_are_read_not_those_of_earlier_invokes(all_batch):
    shape = (1, 70, 50, 41)
    m = _two_outputs(shape)
    rng = np.random.default_rng(17)
    xs = [rng.integers(-128, 128, shape).astype(np.int8) for _ in range(8)]

    def check(x):
        assert np.array_equal(m.get_tensor_i8("first"), np.maximum(x, 0))
        assert np.array_equal(m.get_tensor("second"), x.repeat(2, 2).repeat(2, 3))

    for x in xs[:2]:            # the results are read: the next invokes expect it
        m.set_tensor_i8("x", x)
        m.invoke()
        check(x)
    graph = Graph(m.context_handle())
    with graph.recording():
        if all_batch:
            m.fast_invoke_all_batch("second", 1)
        else:
            m.invoke()
    for k, x in enumerate(xs[2:]):
        if k % 2 == 0:          # a plain invoke in between, read once
            m.set_tensor_i8("x", xs[0])
            m.invoke()
            check(xs[0])
        m.set_tensor_i8("x", x)
        graph.replay()
        check(x)
    graph.close()
    m.close()
