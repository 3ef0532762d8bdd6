"""Tables that are a leaky ReLU's line are computed behind a conv instead of looked up: every kernel that takes a table, for
slopes at the ends of what the 16-bit form holds, and for tables that are a line but for one entry."""
import numpy as np
import pytest

import oracle_lib as O
from gpu_helpers import conv_desc, f2i32
from tpu_compiler_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


def _line(m, r, wrong_at=None):
    y = np.arange(256).astype(np.int8).astype(np.int64)
    t = np.maximum(y, (y * m + (1 << r >> 1)) >> r)
    if wrong_at is not None:
        t[wrong_at] -= 1
    return t.astype(np.int8)


TABLES = {"0.1": _line(13, 7), "102/1024": _line(102, 10), "nothing": _line(1, 9), "one": _line(1, 0), "half": _line(1, 1),
          "steepest": _line(127, 7), "most bits": _line(253, 9), "too many bits": _line(1021, 12),
          "one below": _line(13, 7, 200), "last": _line(13, 7, 128), "positive": _line(13, 7, 100), "zero": _line(13, 7, 0)}
# algorithm or tile name, channels, kernel
FORMS = [("mfma_p_64x64", 48, 72, 3), ("mfma_pw_64x128_k64", 64, 72, 1), ("mfma_patch2_64x128", 64, 72, 3),
         ("mfma_patch3_32x128", 64, 40, 3), ("mfma_rows_64x192", 128, 72, 3), ("mfma_rows_128x160_c64", 64, 72, 3),
         ("mfma_rows_256x256", 128, 290, 3), ("mfma_rows_64x256_c32", 32, 72, 3), ("mfma_ksplit_32x32_w8", 48, 41, 3), ("depthwise", 40, 40, 3),
         ("depthwise_dot", 40, 40, 3), ("depthwise", 24, 24, 5), ("stem", 3, 33, 3)]


@pytest.mark.parametrize("table", sorted(TABLES))
@pytest.mark.parametrize("form", FORMS, ids=lambda f: "%s_%d" % (f[0], f[1]))
def test_conv_with_a_line_behind_it(ctx, form, table):
    name, ic, oc, k = form
    dw = name.startswith("depthwise")
    tiles = {ctx.lib.tpuhip_conv2d_tile_name(t).decode(): t for t in range(256) if ctx.lib.tpuhip_conv2d_tile_name(t)}
    algo = {"depthwise": capi.ALGO_DEPTHWISE, "depthwise_dot": capi.ALGO_DEPTHWISE_DOT, "stem": 5}.get(name, 16 + tiles.get(name, 0))
    rng = np.random.default_rng(ic + k)
    x = rng.integers(-128, 128, (2, ic, 13, 11)).astype(np.int8)
    w = np.clip(np.rint(rng.normal(0, 32, (oc, 1 if dw else ic, k, k))), -127, 127).astype(np.int8)
    bias, mult = rng.integers(-4096, 4097, oc).astype(np.float32), (rng.integers(1 << 23, 1 << 24, oc) * 128).astype(np.float32)
    # sums of spread 74 * 32 * sqrt(K), times 3/4 on average, onto a spread of about 80
    rsh = np.full(oc, np.rint(np.log2(74 * 32 * (w[0].size ** 0.5) * 0.75 / 80)), np.float32)
    p, g = k // 2, ic if dw else 1
    y_ref = O.conv2d_i8(x, w, bias, rsh, mult, O.make_conv_desc(x.shape, w.shape, g, (1, 1), (p,) * 4, (1, 1), (0, 0), False, True, None))
    assert len(np.unique(y_ref)) == 256      # every entry of the table is met
    t = TABLES[table]
    t_ref = O.lut_i8(y_ref, t)
    wh = ctx.conv_prepack(conv_desc(x.shape, w.shape, g=g, pads=(p,) * 4, algo=algo), w, f2i32(bias), f2i32(mult), f2i32(rsh))
    assert ctx.conv_algo_name(wh) == name
    xt, yt, tt = ctx.from_nchw(x), ctx.tensor(y_ref.shape), ctx.tensor(y_ref.shape)
    for keep in (True, False):
        for v in (yt, tt):
            ctx._ck(ctx.lib.tpuhip_memset(ctx.h, v.ptr, 0x55, v.nbytes))
        ctx.conv_post(wh, xt, yt if keep else None, t, tt)
        assert np.array_equal(ctx.to_nchw(tt), t_ref)
        if t[0] == 0:
            assert not ctx.raw(tt)[..., oc:].any()
        assert np.array_equal(ctx.to_nchw(yt), y_ref) if keep else (ctx.raw(yt) == 0x55).all()
    ctx.conv_weights_destroy(wh)
    for v in (xt, yt, tt):
        v.free()


def test_a_module_finds_lines_of_more_bits():
    """a leaky ReLU of multiplier 102, right shift 10, which no line of 7 bits equals, fused behind a conv of a loaded network"""
    import oracle_graph
    from tpu_compiler_amd import graphs, module
    rng = np.random.default_rng(2)
    one = lambda v: np.array([v], np.float32)
    g = graphs.Graph("line", 1)
    g.add(graphs.Op("tpu.input", "x", [], (1, 64, 40, 41)))
    w = np.clip(np.rint(rng.normal(0, 32, (72, 64, 3, 3))), -127, 127).astype(np.float32)
    attrs = dict(kernel_h=3, kernel_w=3, stride_h=1, stride_w=1, dilation_h=1, dilation_w=1, padding_t=1, padding_b=1, padding_l=1,
                 padding_r=1, group=1, is_dw=0, with_bias=1, do_relu=0, pad_value=0)
    g.add(graphs.Op("tpu.conv_2d", "conv", ["x"], (1, 72, 40, 41), attrs,
                    dict(filter=w, bias=rng.integers(-4096, 4097, 72).astype(np.float32), rshift=np.full(72, 9, np.float32),
                         multiplier=(rng.integers(1 << 23, 1 << 24, 72) * 128.0).astype(np.float32)), "RSHIFT_AND_M_I32"))
    g.add(graphs.Op("tpu.leaky_relu", "leaky", ["conv"], (1, 72, 40, 41), dict(negative_slope=0.1),
                    dict(rshift_pos=one(0), multiplier_pos=one(1), rshift_neg=one(10), multiplier_neg=one(102)), "RSHIFT_AND_M_I8"))
    g.outputs = ["leaky"]
    x = rng.integers(-128, 128, (1, 64, 40, 41)).astype(np.int8)
    want = oracle_graph.run(g, input_data=x)
    for keep in (1, 0):
        m = module()
        m.set_option("keep_all_tensors", keep)
        m.load(g)
        for _ in range(2):
            m.set_tensor_i8("x", x)
            m.invoke()
            assert np.array_equal(m.get_tensor_i8("leaky"), want["leaky"])
            assert not keep or np.array_equal(m.get_tensor_i8("conv"), want["conv"])
        m.close()


def test_a_tile_is_chosen_apart_for_a_line_and_another_table(ctx):
    """a computed line and a lookup are other epilogues: what timing chose for a shape with one is not taken for the other"""
    rng = np.random.default_rng(5)
    x = rng.integers(-128, 128, (1, 64, 19, 23)).astype(np.int8)
    w = rng.integers(-60, 61, (88, 64, 1, 1)).astype(np.int8)
    mult, rsh = np.full(88, 1 << 30, np.int32), np.full(88, 8, np.int32)
    d = conv_desc(x.shape, w.shape, with_bias=False)
    xt, yt, tt = ctx.from_nchw(x), ctx.tensor((1, 88, 19, 23)), ctx.tensor((1, 88, 19, 23))
    other = rng.integers(-128, 128, 256).astype(np.int8)
    y_ref = O.conv2d_i8(x, w, None, rsh.astype(np.float32), mult.astype(np.float32),
                        O.make_conv_desc(x.shape, w.shape, 1, (1, 1), (0, 0, 0, 0), (1, 1), (0, 0), False, False, None))
    known = ctx.lib.tpuhip_conv2d_tiles_known()
    for table, new in ((TABLES["0.1"], 1), (other, 1), (TABLES["half"], 0), (TABLES["one below"], 0), (None, 1)):
        wh = ctx.conv_prepack(d, w, None, mult, rsh)
        if table is None:
            ctx.conv(wh, xt, tt)
        else:
            ctx.conv_post(wh, xt, yt, table, tt)
        assert np.array_equal(ctx.to_nchw(tt), y_ref if table is None else O.lut_i8(y_ref, table))
        known += new
        assert ctx.lib.tpuhip_conv2d_tiles_known() == known
        ctx.conv_weights_destroy(wh)
    for t in (xt, yt, tt):
        t.free()
