"""K split over waves with blocks of 16 x 16 outputs, every variant: input as a patch in LDS and straight from memory, maps that
leave slots, rows, columns and channel blocks over, more and fewer slices of K than waves, everything that rides behind a conv."""
import numpy as np
import pytest

import oracle_lib as O
from gpu_helpers import conv_desc, f2i32
from tpu_compiler_amd import capi

pytestmark = pytest.mark.gpu


def _name(t):
    n = capi.bind().tpuhip_conv2d_tile_name(t)
    return n.decode() if n else ""


SPLIT_TILES = [t for t in range(128) if _name(t).startswith("mfma_split_")]


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


# n, ic, ih, iw, oc, (kh, kw), (sh, sw), (pt, pb, pl, pr), (dh, dw), relu
CASES = [
    (1, 64, 7, 7, 40, (3, 3), (1, 1), (1, 1, 1, 1), (1, 1), True),          # one slice or none per wave
    (1, 512, 13, 13, 33, (3, 3), (1, 1), (1, 1, 1, 1), (1, 1), False),      # nine per wave, rows left over
    (2, 320, 5, 9, 48, (3, 3), (1, 1), (1, 1, 1, 1), (1, 1), True),         # 45 slices: rounds with a rest
    (1, 128, 9, 150, 20, (3, 3), (2, 2), (1, 1, 1, 1), (1, 1), True),       # part of a row per tile, every second pixel
    (1, 64, 3, 131, 16, (3, 3), (1, 1), (1, 1, 1, 1), (1, 1), False),       # columns left over
    (1, 128, 12, 11, 70, (5, 5), (2, 2), (2, 2, 2, 2), (1, 1), False),
    (2, 64, 10, 14, 32, (3, 3), (1, 1), (2, 2, 2, 2), (2, 2), True),        # dilated
    (1, 192, 6, 5, 17, (2, 4), (1, 2), (0, 1, 3, 0), (2, 1), False),
    (3, 1024, 2, 2, 50, (3, 3), (1, 1), (1, 1, 1, 1), (1, 1), True),        # 18 per wave: two rounds of nine
    (1, 1024, 9, 11, 30, (5, 5), (1, 1), (2, 2, 2, 2), (1, 1), False),      # a patch that fewer rows, or columns, bring into LDS
    (1, 64, 1, 1, 16, (3, 3), (1, 1), (1, 1, 1, 1), (1, 1), False),         # one pixel, one column
    (2, 64, 40, 1, 16, (3, 1), (1, 1), (1, 1, 0, 0), (1, 1), True),         # columns of one
    (1, 1024, 14, 14, 70, (1, 1), (1, 1), (0, 0, 0, 0), (1, 1), False),     # straight from memory
    (2, 256, 9, 7, 130, (1, 1), (2, 2), (0, 0, 0, 0), (1, 1), True),
    (1, 96, 11, 5, 24, (3, 3), (1, 1), (1, 1, 1, 1), (1, 1), True),         # slices that straddle taps
    (2, 100, 9, 13, 40, (3, 3), (1, 1), (1, 1, 1, 1), (1, 1), False),       # 63 groups of 16 bytes: one past the end of K
    (1, 37, 20, 21, 50, (5, 5), (2, 2), (2, 2, 2, 2), (1, 1), True),        # 75 groups
    (1, 250, 8, 30, 48, (3, 3), (1, 1), (1, 1, 1, 1), (1, 1), True), (2, 16, 12, 7, 20, (2, 4), (1, 1), (1, 0, 2, 1), (2, 1), False),
    (1, 290, 9, 11, 33, (3, 3), (1, 1), (1, 1, 1, 1), (1, 1), False), (2, 64, 9, 9, 20, (7, 7), (1, 1), (3, 3, 3, 3), (1, 1), True),
    (1, 130, 30, 9, 24, (7, 1), (1, 1), (3, 3, 0, 0), (1, 1), True),
    (3, 16, 5, 6, 33, (1, 1), (1, 1), (0, 0, 0, 0), (1, 1), False), (1, 3, 8, 9, 40, (3, 3), (2, 2), (1, 1, 1, 1), (1, 1), True),
]


def _layer(case, seed):
    n, ic, ih, iw, oc, k, s, pads, dil, relu = case
    rng = np.random.default_rng(seed)
    x = rng.integers(-128, 128, (n, ic, ih, iw)).astype(np.int8)
    w = np.clip(np.rint(rng.normal(0, 14, (oc, ic) + k)), -127, 127).astype(np.int8)
    bias, mult = rng.integers(-4096, 4097, oc).astype(np.float32), (rng.integers(1 << 23, 1 << 24, oc) * 128).astype(np.float32)
    rsh = np.resize(np.array([8, 9, 10, 11, 12], np.float32), oc)
    return rng, x, w, bias, mult, rsh


@pytest.mark.parametrize("tile", SPLIT_TILES, ids=_name)
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:5])))
@pytest.mark.parametrize("post", ["plain", "table_add", "sum_only"])
def test_against_the_oracle(ctx, tile, case, post):
    n, ic, ih, iw, oc, k, s, pads, dil, relu = case
    rng, x, w, bias, mult, rsh = _layer(case, ic + oc)
    d = conv_desc(x.shape, w.shape, stride=s, pads=pads, dil=dil, do_relu=relu, algo=16 + tile)
    y_ref = O.conv2d_i8(x, w, bias, rsh, mult, O.make_conv_desc(x.shape, w.shape, 1, s, pads, dil, (0, 0), relu, True, None))
    xt, other = ctx.from_nchw(x), rng.integers(-128, 128, y_ref.shape).astype(np.int8)
    ot, yt, tt, zt = ctx.from_nchw(other), ctx.tensor(y_ref.shape), ctx.tensor(y_ref.shape), ctx.tensor(y_ref.shape)
    for t in (yt, tt, zt):
        ctx._ck(ctx.lib.tpuhip_memset(ctx.h, t.ptr, 0x55, t.nbytes))
    wh = ctx.conv_prepack(d, w, f2i32(bias), f2i32(mult), f2i32(rsh))
    table = rng.integers(-128, 128, 256).astype(np.int8)
    table[0] = 77                                  # pad channels must stay 0 all the same
    t_ref = O.lut_i8(y_ref, table)
    if post == "plain":
        ctx.conv(wh, xt, yt)
        checks = [(yt, y_ref)]
    elif post == "table_add":
        ctx.conv_post(wh, xt, yt, table, tt, (ot, zt, 37, 51, 5, False))
        checks = [(yt, y_ref), (tt, t_ref), (zt, O.eltwise_add_i8([other, t_ref], [37, 51], [5], False))]
    else:
        ctx.conv_post(wh, xt, None, None, None, (ot, zt, 61, -47, 6, True))
        checks = [(zt, O.eltwise_add_i8([other, y_ref], [61, -47], [6], True))]
    for t, ref in checks:
        assert np.array_equal(ctx.to_nchw(t), ref) and not ctx.raw(t)[..., oc:].any()
    ctx.conv_weights_destroy(wh)
    for t in (xt, ot, yt, tt, zt):
        t.free()


@pytest.mark.parametrize("tile", SPLIT_TILES, ids=_name)
@pytest.mark.parametrize("case", [CASES[0], CASES[1], CASES[12], CASES[14]], ids=lambda c: "x".join(map(str, c[:5])))
@pytest.mark.parametrize("relu_first", [0, 1])
def test_shifts_of_zero_and_a_relu_in_front(ctx, tile, case, relu_first):
    """the requantisation that may overflow, without the patch; a ReLU on the sum"""
    n, ic, ih, iw, oc, k, s, pads, dil, _ = case
    rng, x, w, bias, mult, rsh = _layer(case, ic * 3 + oc)
    if not relu_first:
        rsh[::5] = 0
    d = conv_desc(x.shape, w.shape, stride=s, pads=pads, dil=dil, do_relu=True, relu_first=relu_first, algo=16 + tile)
    od = O.make_conv_desc(x.shape, w.shape, 1, s, pads, dil, (0, 0), True, True, None)
    want = O.conv2d_i8(x, w, bias, rsh, mult, od)   # a rounding shift of a sum below zero is not above it: the same result
    xt, yt = ctx.from_nchw(x), ctx.tensor(want.shape)
    wh = ctx.conv_prepack(d, w, f2i32(bias), f2i32(mult), f2i32(rsh))
    ctx.conv(wh, xt, yt)
    assert np.array_equal(ctx.to_nchw(yt), want) and not ctx.raw(yt)[..., oc:].any()
    ctx.conv_weights_destroy(wh)
    xt.free()
    yt.free()


# n, ic, ih, iw, oc_a, oc_b, stride, dilation: 36 to 72 slices, which all variants take as a patch; the second result's channels end
# within a block of 16, at its end, in a block of 32 whose second half is past them, and after several blocks
@pytest.mark.parametrize("tile", SPLIT_TILES, ids=_name)
@pytest.mark.parametrize("pair", [(1, 256, 13, 11, 128, 40, 1, 1), (2, 256, 9, 15, 256, 16, 2, 1), (1, 512, 7, 7, 128, 24, 1, 1),
                                  (1, 256, 14, 14, 128, 130, 1, 2)], ids=lambda c: "x".join(map(str, c[:6])))
@pytest.mark.parametrize("relus", [(True, False), (False, True)])
def test_a_pair_of_which_the_input_lies_in_a_patch(ctx, tile, pair, relus):
    n, ic, ih, iw, oca, ocb, stride, dil = pair
    parts, refs = [], []
    for oc, relu in zip((oca, ocb), relus):
        case = (n, ic, ih, iw, oc, (3, 3), (stride, stride), (dil,) * 4, (dil, dil), relu)
        rng, x, w, bias, mult, rsh = _layer(case, oca + ocb)
        if parts:
            w, bias, mult = w[::-1].copy(), -bias, mult[::-1].copy()
        d = conv_desc(x.shape, w.shape, stride=case[6], pads=case[7], dil=case[8], do_relu=relu, algo=16 + tile)
        parts.append((d, (w, f2i32(bias), f2i32(mult), f2i32(rsh))))
        refs.append(O.conv2d_i8(x, w, bias, rsh, mult, O.make_conv_desc(x.shape, w.shape, 1, case[6], case[7], case[8], (0, 0), relu, True, None)))
    wh = ctx.conv_prepack_pair(parts[0][0], parts[1][0], parts[0][1], parts[1][1])
    xt, ys = ctx.from_nchw(x), [ctx.tensor(r.shape) for r in refs]
    for t in ys:
        ctx._ck(ctx.lib.tpuhip_memset(ctx.h, t.ptr, 0x55, t.nbytes))
    ctx.conv_pair(wh, xt, ys[0], ys[1])
    for t, ref in zip(ys, refs):
        assert np.array_equal(ctx.to_nchw(t), ref) and not ctx.raw(t)[..., ref.shape[1]:].any()
    ctx.conv_weights_destroy(wh)
    for t in [xt] + ys:
        t.free()


@pytest.mark.parametrize("tile", SPLIT_TILES, ids=_name)
@pytest.mark.parametrize("case", [CASES[0], CASES[1], CASES[12]], ids=lambda c: "x".join(map(str, c[:5])))
@pytest.mark.parametrize("stride", [65520, 65536, 65552])
def test_an_input_stride_given_behind_the_choice(ctx, tile, case, stride):
    """strides on both sides of 16 bits, set once the layer is packed: a part of a wide tensor's channels"""
    n, ic, ih, iw, oc, k, s, pads, dil, relu = case
    rng, x, w, bias, mult, rsh = _layer(case, ic + stride)
    d = conv_desc(x.shape, w.shape, stride=s, pads=pads, dil=dil, do_relu=relu, algo=16 + tile)
    want = O.conv2d_i8(x, w, bias, rsh, mult, O.make_conv_desc(x.shape, w.shape, 1, s, pads, dil, (0, 0), relu, True, None))
    wh = ctx.conv_prepack(d, w, f2i32(bias), f2i32(mult), f2i32(rsh))
    ctx.conv_set_input_stride(wh, stride)
    xt, yt = ctx.from_nchw(x, stride), ctx.tensor(want.shape)
    ctx.conv(wh, xt, yt)
    assert np.array_equal(ctx.to_nchw(yt), want) and not ctx.raw(yt)[..., oc:].any()
    ctx.conv_weights_destroy(wh)
    xt.free()
    yt.free()


def test_a_timed_layer_takes_any_input_stride(ctx):
    case = CASES[0]
    n, ic, ih, iw, oc, k, s, pads, dil, relu = case
    rng, x, w, bias, mult, rsh = _layer(case, 3)
    want = O.conv2d_i8(x, w, bias, rsh, mult, O.make_conv_desc(x.shape, w.shape, 1, s, pads, dil, (0, 0), relu, True, None))
    wh = ctx.conv_prepack(conv_desc(x.shape, w.shape, stride=s, pads=pads, dil=dil, do_relu=relu), w, f2i32(bias), f2i32(mult), f2i32(rsh))
    yt = ctx.tensor(want.shape)
    for stride in (64, 1 << 16, 1 << 21):
        ctx.conv_set_input_stride(wh, stride)
        xt = ctx.from_nchw(x, stride)
        ctx.conv(wh, xt, yt)
        assert np.array_equal(ctx.to_nchw(yt), want), stride
        xt.free()
    ctx.conv_weights_destroy(wh)
    yt.free()
