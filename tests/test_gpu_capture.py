"""HIP graphs recorded from a module's or a context's stream: replays give what plain calls give, whatever is called in
between, and what cannot be recorded is refused."""
import numpy as np
import pytest

import oracle_graph
import oracle_lib as O
from gpu_capture import Graph
from gpu_helpers import conv_desc, pool_desc, run_conv
from tpu_compiler_amd import capi, graphs, mlir_text, module

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


def _run_files(m, g, folder):
    path = folder / "model.mlir"
    mlir_text.write_mlir(g, path)
    np.savez(folder / "in.npz", **{g.input_op().name: g.input_op().data.astype(np.float32)})
    m.interpret_files(path, folder / "in.npz", folder / "out.npz")


def _check_replays(m, g, graph, plain):
    rng = np.random.default_rng(3)
    name, shape = g.input_op().name, g.input_op().shape
    for k in range(4):
        x = rng.integers(-128, 128, shape).astype(np.int8)
        want = oracle_graph.run(g, input_data=x)
        m.set_tensor_i8(name, x)
        if k % 2:
            plain()
        else:
            graph.replay()
        for op in g.ops:
            assert np.array_equal(m.get_tensor_i8(op.name), want[op.name].reshape(op.shape)), (k, op.name)


# sides that nothing else here uses: no layer finds its tile remembered
@pytest.mark.parametrize("make", [lambda: graphs.cfg3_resnet50(batch=1, hw=72), lambda: graphs.cfg4_mobilenet_v2(batch=1, hw=72),
                                  lambda: graphs.cfg5_yolo_v3(batch=1, hw=96)])
def test_a_network_that_ran_once_from_files_can_be_recorded(make, tmp_path):
    g, m = make(), module()
    _run_files(m, g, tmp_path)
    graph = Graph(m.context_handle())
    with graph.recording():
        m.invoke()
    tiles = m.kernels()
    _check_replays(m, g, graph, m.invoke)
    assert m.kernels() == tiles          # the graph reads the filters as they were packed then
    graph.close()
    m.close()


def test_a_network_that_ran_once_from_files_chooses_its_tiles_at_the_next_use(tmp_path):
    g, m = graphs.cfg3_resnet50(batch=1, hw=104), module()
    _run_files(m, g, tmp_path)
    untimed = m.kernels()
    graph = Graph(m.context_handle())
    m.invoke()                           # times the variants and packs the filters again
    assert m.kernels() != untimed
    with graph.recording():
        m.invoke()
    _check_replays(m, g, graph, m.invoke)
    graph.close()
    m.close()


def test_a_layer_whose_first_use_is_recorded_is_refused():
    g = graphs.cfg3_resnet50(batch=1, hw=88)
    for remembered in (False, True):     # the second module's shapes have been timed by the first
        m = module()
        m.load(g)
        graph = Graph(m.context_handle())
        with graph.recording():
            with pytest.raises(capi.TpuHipError, match="captured"):
                m.invoke()
        graph.close()
        m.set_tensor_i8(g.input_op().name, g.input_op().data.astype(np.int8))
        m.invoke()
        m.sync()
        with graph.recording():
            m.invoke()
        _check_replays(m, g, graph, m.invoke)
        graph.close()
        m.close()


@pytest.mark.parametrize("shape", [(1, 3, 20, 31), (4, 70, 61, 67)])     # one piece of the staging buffer, several
def test_host_tensors_are_refused_while_the_stream_is_captured(shape):
    m = _two_outputs(shape)
    rng = np.random.default_rng(11)
    xs = [rng.integers(-128, 128, shape).astype(np.int8) for _ in range(4)]
    for x in xs[:2]:
        m.set_tensor_i8("x", x)
        m.invoke()
        assert np.array_equal(m.get_tensor_i8("first"), np.maximum(x, 0))
    m.invoke()                           # "first" of xs[1], laid out early where it is large enough
    graph = Graph(m.context_handle())
    with graph.recording():
        for call in (lambda: m.get_tensor_i8("first"), lambda: m.get_tensor("second"), lambda: m._get_tensors(["first", "second"]),
                     lambda: m.set_tensor_i8("x", xs[3]), lambda: m.set_tensor("x", xs[3])):
            with pytest.raises(capi.TpuHipError, match="being captured"):
                call()
        m.invoke()
    assert graph.nodes() == 2            # the two kernels of the invoke: nothing of the refused calls
    for x in xs[1:3] * 2:
        m.set_tensor_i8("x", x)
        graph.replay()
        assert np.array_equal(m.get_tensor_i8("first"), np.maximum(x, 0))
        assert np.array_equal(m.get_tensor("second"), x.repeat(2, 2).repeat(2, 3))
    graph.close()
    m.close()


# dense, stem, depthwise, grouped, transposed
@pytest.mark.parametrize("ic,oc,k,kw", [(32, 32, 1, {}), (3, 16, 3, {}), (32, 32, 3, dict(g=32)), (32, 32, 3, dict(g=4)),
                                        (16, 16, 3, dict(ins=(1, 1)))])
def test_packing_weights_is_refused_while_the_stream_is_captured(ic, oc, k, kw):
    ctx = capi.Context(0)
    rng = np.random.default_rng(31)
    x = rng.integers(-128, 128, (1, ic, 12, 12)).astype(np.int8)
    w = rng.integers(-64, 65, (oc, ic // kw.get("g", 1), k, k)).astype(np.int8)
    bias, rshift, mult = rng.integers(-500, 500, oc).astype(np.float32), np.full(oc, 9, np.float32), np.full(oc, 1 << 30, np.float32)
    want, _ = run_conv(ctx, x, w, bias, rshift, mult, **kw)
    a, y = ctx.from_nchw(x), ctx.tensor(want.shape)
    graph = Graph(ctx.h)
    with graph.recording():
        with pytest.raises(capi.TpuHipError, match="being captured"):
            ctx.conv_prepack(conv_desc(x.shape, w.shape, **kw), w, bias.astype(np.int32), mult.astype(np.int32), rshift.astype(np.int32))
        ctx._ck(ctx.lib.tpuhip_memset(ctx.h, y.ptr, 3, y.nbytes))
    assert graph.nodes() == 1
    graph.replay()
    again, _ = run_conv(ctx, x, w, bias, rshift, mult, **kw)
    assert np.array_equal(again, want) and (ctx.raw(y) == 3).all()
    graph.close()
    a.free()
    y.free()
    ctx.close()


@pytest.mark.parametrize("shape", [(1, 120, 40, 40), (2, 17, 75, 75), (1, 16, 33, 47)])
def test_a_recorded_average_over_a_large_window_needs_no_memory_of_its_context(shape):
    other = (2 * shape[0], 2 * shape[1], 100, 90)      # a plain pool that takes a larger workspace
    ctx = capi.Context(0)
    rng = np.random.default_rng(sum(shape))

    def pool(s):
        d = pool_desc(s, s[2:], (1, 1), (0, 0, 0, 0), (1, 1))
        x, y = ctx.tensor(s), ctx.tensor(s[:2] + (1, 1))
        mult = min(255, int(4428 / (s[2] * s[3]) ** 0.5))
        return d, x, y, lambda: ctx.pool_avg(d, x, y, mult, 13)

    def check(s, x, y, call):
        data = rng.integers(-128, 128, s).astype(np.int8)
        filled = ctx.from_nchw(data, x.cs)
        ctx._ck(ctx.lib.tpuhip_memset(ctx.h, y.ptr, 0x55, y.nbytes))
        ctx._ck(ctx.lib.tpuhip_download(ctx.h, host.ctypes.data, filled.ptr, filled.nbytes))
        ctx._ck(ctx.lib.tpuhip_upload(ctx.h, x.ptr, host.ctypes.data, filled.nbytes))
        filled.free()
        call()
        want = O.pool_avg_i8(data, O.make_pool_desc(s, s[2:], (1, 1), (0, 0, 0, 0)), 13,
                             min(255, int(4428 / (s[2] * s[3]) ** 0.5)))
        assert np.array_equal(ctx.to_nchw(y), want)
        assert not ctx.raw(y)[..., s[1]:].any()

    _, x, y, plain = pool(shape)
    _, x2, y2, larger = pool(other)
    host = np.empty(max(x.nbytes, x2.nbytes), np.int8)
    check(shape, x, y, plain)              # the workspace is there
    graph = Graph(ctx.h)
    with graph.recording():
        plain()
    assert graph.nodes() == 1              # no second launch that adds up partial sums in the workspace
    for k in range(3):
        check(shape, x, y, graph.replay)
        check(other, x2, y2, larger)       # outgrows it
        check(shape, x, y, plain)
    graph.close()
    for t in (x, y, x2, y2):
        t.free()
    ctx.close()
