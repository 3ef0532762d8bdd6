"""Tensors between host memory and the device: the layout kernels at the edges of their tiles, and set_tensor /
get_tensor in one piece, in several, and through more than the staging buffer holds."""
import time

import numpy as np
import pytest

from gpu_capture import Graph
from tpu_compiler_amd import capi, graphs, module

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("shape,cs", [
    ((2, 3, 5, 7), 16), ((2, 3, 5, 7), 4), ((3, 4, 1, 127), 4), ((1, 1, 32, 32), 16), ((2, 2, 33, 31), 4),   # images
    ((5, 1000, 1, 1), None), ((3, 13, 1, 1), None), ((1, 16, 1, 1), 48), ((70, 255, 1, 1), None),            # vectors
    ((2, 64, 16, 8), None), ((2, 65, 1, 129), None), ((1, 17, 3, 43), 64), ((3, 255, 13, 13), None),         # tiles
    ((2, 128, 2, 1), None), ((1, 5, 300, 1), None)])
def test_layout_conversions(ctx, shape, cs):
    rng = np.random.default_rng(sum(shape))
    x = rng.integers(-128, 128, shape).astype(np.int8)
    t = ctx.tensor(shape, cs)
    ctx._ck(ctx.lib.tpuhip_memset(ctx.h, t.ptr, 0x55, t.nbytes))
    t2 = ctx.from_nchw(x, cs)
    raw = ctx.raw(t2)
    assert np.array_equal(raw[..., :shape[1]], x.transpose(0, 2, 3, 1)) and not raw[..., shape[1]:].any()
    assert np.array_equal(ctx.to_nchw(t2), x)
    t.free()
    t2.free()


def _relu_module(shape, quant="INT8"):
    g = graphs.Graph("io", 1)
    op = g.add(graphs.Op("tpu.input", "x", [], shape))
    if quant == "NONE":
        op.quant = "NONE"
        g.add(graphs.Op("tpu.quant", "q", ["x"], shape, dict(scale=1.0)))
        y = g.add(graphs.Op("tpu.quant", "y", ["q"], shape, dict(scale=1.0)))
        y.quant = "NONE"
    else:
        g.add(graphs.Op("tpu.relu", "y", ["x"], shape))
    g.outputs = ["y"]
    m = module()
    m.load(g)
    return m


# one piece; several pieces; spans with a ragged end; more than the staging buffer holds
SHAPES = [(1, 3, 20, 31), (2, 3, 181, 182), (4, 70, 61, 67), (3, 129, 130, 131), (5, 64, 331, 333)]


@pytest.mark.parametrize("shape", SHAPES)
def test_round_trip_of_float_and_int8_tensors(shape):
    m = _relu_module(shape)
    rng = np.random.default_rng(shape[3])
    for k in range(2):      # a second tensor behind the first: the staging buffer is in use again
        x = rng.integers(-128, 128, shape).astype(np.int8)
        want = np.maximum(x, 0)
        if k:
            m.set_tensor_i8("x", x)
        else:
            m.set_tensor("x", x.astype(np.float32))
        m.invoke()
        assert np.array_equal(m.get_tensor_i8("y"), want)
        assert np.array_equal(m.get_tensor("y"), want.astype(np.float32))
        assert np.array_equal(m.get_tensor("x"), x.astype(np.float32))
    m.close()


@pytest.mark.parametrize("shape", SHAPES[:4])
@pytest.mark.parametrize("value", [0.5, 128.0, -129.0, np.nan, np.inf])
def test_a_float_that_is_no_int8_is_refused_and_changes_nothing(shape, value):
    m = _relu_module(shape)
    x = np.random.default_rng(3).integers(-128, 128, shape).astype(np.float32)
    m.set_tensor("x", x)
    bad = np.zeros(shape, np.float32)
    bad.reshape(-1)[-2] = value
    with pytest.raises(capi.TpuHipError, match="element %d" % (bad.size - 2)):
        m.set_tensor("x", bad)
    assert np.array_equal(m.get_tensor("x"), x)
    m.close()


@pytest.mark.parametrize("shape", SHAPES[:3])
def test_round_trip_of_fp32_edges(shape):
    m = _relu_module(shape, "NONE")
    x = np.random.default_rng(5).integers(-128, 128, shape).astype(np.float32)
    m.set_tensor("x", x)
    m.invoke()
    assert np.array_equal(m.get_tensor("x"), x) and np.array_equal(m.get_tensor("y"), x)
    m.close()


# together straight into the staging buffer; several spans of one filling (test_gpu_dense_list.py has several fillings); a tensor
# larger than the buffer among small ones
@pytest.mark.parametrize("shapes", [[(1, 3, 20, 31), (2, 1000, 1, 1)], [(4, 70, 61, 67), (1, 255, 13, 13), (3, 129, 130, 131)],
                                    [(2, 17, 9, 9), (5, 64, 331, 333), (1, 5, 300, 1)]])
def test_all_tensors_at_once(shapes):
    g = graphs.Graph("io", 1)
    for i, s in enumerate(shapes):
        g.add(graphs.Op("tpu.input", "x%d" % i, [], s))
    for i, s in enumerate(shapes):
        g.add(graphs.Op("tpu.relu", "y%d" % i, ["x%d" % i], s))
    g.outputs = ["y%d" % i for i in range(len(shapes))]
    m = module()
    m.load(g)
    held = []
    for k in range(3):      # results that are still held keep their values
        xs = [np.random.default_rng(k + i).integers(-128, 128, s).astype(np.int8) for i, s in enumerate(shapes)]
        got = m.run(np.concatenate([x.reshape(-1) for x in xs]))
        held.append((xs, got, m.get_all_tensor()))
    for xs, got, every in held:
        assert sorted(every) == sorted(m.tensor_names())
        for i, x in enumerate(xs):
            assert np.array_equal(got["y%d" % i], np.maximum(x, 0)) and np.array_equal(every["y%d" % i], np.maximum(x, 0))
            assert np.array_equal(every["x%d" % i], x)
    m.close()


# results complete before the last kernel: large enough to be read ahead, and not
@pytest.mark.parametrize("shape", [(1, 70, 50, 41), (3, 64, 40, 40), (1, 5, 20, 20)])
def test_an_early_output_is_what_the_last_invoke_made_of_it(shape):
    g = graphs.Graph("early", 1)
    g.add(graphs.Op("tpu.input", "x", [], shape))
    g.add(graphs.Op("tpu.relu", "first", ["x"], shape))
    g.add(graphs.Op("tpu.upsample", "second", ["x"], shape[:2] + (2 * shape[2], 2 * shape[3]), dict(scale_h=2, scale_w=2)))
    g.outputs = ["first", "second"]
    m = module()
    m.load(g)
    rng = np.random.default_rng(9)
    xs = [rng.integers(-128, 128, shape).astype(np.int8) for _ in range(5)]
    for x in xs:
        m.set_tensor_i8("x", x)
        m.invoke()
        for _ in range(2):
            assert np.array_equal(m.get_tensor_i8("first"), np.maximum(x, 0))
        assert np.array_equal(m.get_tensor("second"), x.repeat(2, 2).repeat(2, 3))
    m.set_tensor_i8("x", xs[0])                     # no invoke: the old result
    assert np.array_equal(m.get_tensor_i8("first"), np.maximum(xs[-1], 0))
    m.invoke_to("first")
    assert np.array_equal(m.get_tensor("first"), np.maximum(xs[0], 0))
    m.set_tensor_i8("first", xs[1])                 # written by hand
    assert np.array_equal(m.get_tensor_i8("first"), xs[1])
    m.invoke()
    m.invoke()                                      # two in a row, the first one's result is never read
    got = m.run(xs[2])
    assert np.array_equal(got["first"], np.maximum(xs[2], 0)) and np.array_equal(got["second"], xs[2].repeat(2, 2).repeat(2, 3))
    m.close()


@pytest.mark.parametrize("read", ["get_tensor", "get_tensor_i8", "get_tensors", "run"])
def test_reading_an_early_output_waits_for_the_whole_invoke(read):
    shape, big, behind = (1, 70, 50, 41), (1, 64, 1024, 1024), 40      # 40 passes over 2 x 67 MB: about a millisecond
    g = graphs.Graph("early", 1)
    g.add(graphs.Op("tpu.input", "x", [], shape))
    g.add(graphs.Op("tpu.input", "z", [], big))
    g.add(graphs.Op("tpu.relu", "first", ["x"], shape))
    g.add(graphs.Op("tpu.relu", "other", ["x"], shape))
    last = "z"
    for i in range(behind):
        g.add(graphs.Op("tpu.relu", "z%d" % i, [last], big))
        last = "z%d" % i
    g.outputs = ["first", "other"]
    m = module()
    m.load(g)
    graph = Graph(m.context_handle())
    rng = np.random.default_rng(29)
    z = rng.integers(-128, 128, big).astype(np.int8)
    m.set_tensor_i8("z", z)
    for _ in range(3):
        x = rng.integers(-128, 128, shape).astype(np.int8)
        m.set_tensor_i8("x", x)
        m.invoke()
        got = m._get_tensors(["first"])["first"] if read == "get_tensors" else \
            m._get_tensors(["first", "other"])["first"] if read == "run" else getattr(m, read)("first")
        assert graph.idle()
        assert np.array_equal(got, np.maximum(x, 0))
        assert np.array_equal(m.get_tensor_i8("other"), np.maximum(x, 0)) and graph.idle()
    assert np.array_equal(m.get_tensor_i8(last), np.maximum(z, 0))
    m.close()


def test_a_read_behind_long_work_keeps_one_thread_waiting():
    shape, behind, invokes = (1, 64, 1024, 1024), 40, 30      # 1200 passes over 2 x 67 MB: some 30 ms
    g = graphs.Graph("long", 1)
    g.add(graphs.Op("tpu.input", "y0", [], shape))
    for i in range(behind):
        g.add(graphs.Op("tpu.relu", "y%d" % (i + 1), ["y%d" % i], shape))
    g.outputs = ["y%d" % behind]
    m = module()
    m.load(g)
    x = np.random.default_rng(41).integers(-128, 128, shape).astype(np.int8)
    m.set_tensor_i8("y0", x)
    for _ in range(3):                  # nothing is in the staging buffer any more, the result's memory is there
        m.invoke()
        got = m.get_tensor_i8(g.outputs[0])
    for _ in range(invokes):
        m.invoke()
    wall, cpu = time.perf_counter(), time.process_time()
    got = m.get_tensor_i8(g.outputs[0])
    wall, cpu = time.perf_counter() - wall, time.process_time() - cpu
    assert np.array_equal(got, np.maximum(x, 0))
    print("read: %.1f ms, CPU time %.1f ms" % (wall * 1e3, cpu * 1e3))
    # eight threads for the pieces of the result, a few milliseconds, one for the rest: eight for all of it would be 8
    assert cpu < 3 * wall
    m.close()
