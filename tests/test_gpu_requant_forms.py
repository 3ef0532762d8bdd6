"""The requantisation whose last steps run on packed int16, at the ends of what it takes and beyond them (a layer with one channel
that does not fit runs the other forms), in every kernel that knows it, against the oracle."""
import numpy as np
import pytest

import oracle_lib as O
from gpu_helpers import conv_desc, f2i32, pool_desc
from tpu_compiler_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


def _tile(ctx, name):
    return next(16 + t for t in range(256) if ctx.lib.tpuhip_conv2d_tile_name(t) == name.encode())


# multipliers with the trailing zeros of a float (1.0, the smallest and largest normal ones, a power of two that makes ties),
# small ones, none, the one that wraps; and with too few zeros for a right shift of 10
MULTS = [1 << 30, (1 << 30) + 128, (1 << 31) - 128, 5 << 28, 3 << 29, 128, 0, 1 << 31]
# right shifts: the smallest, around the one (9) from which on the multiplier is divided, the largest for 7 zeros
SHIFTS = {"fits": [2, 3, 8, 9, 10, 11, 15, 16], "one": [1, 2, 9, 9, 10, 11, 15, 16], "beyond": [2, 3, 8, 9, 10, 11, 16, 17],
          "zeros": [10] * 8}
FORMS = [("mfma_p_64x64", 64, 3), ("mfma_64x64_k128", 48, 1), ("mfma_64x128_k128", 80, 3), ("mfma_p_32x128", 3, 3),
         ("mfma_pw_64x128_k64", 64, 1), ("mfma_pw_128x64_k256_w8", 256, 1), ("mfma_patch2_64x128", 64, 3),
         ("mfma_patch3_32x128", 64, 3), ("depthwise", 64, 3), ("depthwise", 64, 1)]
# these run no other form: a layer with a channel that does not fit is refused (test_gpu_conv_rows)
NARROW_ONLY = [("mfma_rows_128x128_c64", 64, 3), ("mfma_rows_64x192", 128, 3), ("mfma_rows_64x320_c32", 32, 3)]


def _layer(ic, oc, k, dw, shifts, seed):
    """every multiplier with every right shift, weights and biases that make sums around where results end, exact halves among
    them"""
    rng = np.random.default_rng(seed)
    rsh = np.resize(np.array(SHIFTS[shifts]), oc).astype(np.float32)
    mult = np.array([MULTS[(i // 8 + i) % 8] for i in range(oc)], np.float32)
    if shifts == "zeros":
        mult = np.full(oc, (1 << 30) + 64, np.float32)     # 2^30 + 64 rounds to a float with 7 zeros: set as an integer below
    taps = (1 if dw else ic) * k * k
    # spread of the weights for results of spread 60 where the multiplier is about 2^30: sums of 60 * 2^(r + 1)
    sigma = np.minimum(60.0 * 2.0 ** (rsh + 1) / (74 * taps ** 0.5), 60.0)
    w = np.clip(np.rint(rng.normal(0, 1, (oc, 1 if dw else ic, k, k)) * np.maximum(sigma, 0.7)[:, None, None, None]), -127, 127)
    bias = rng.integers(-300, 300, oc) * 2.0 ** np.maximum(rsh - 6, 0)
    return w.astype(np.int8), bias.astype(np.float32), rsh, mult


@pytest.mark.parametrize("form,shifts", [(f, s) for f in FORMS for s in sorted(SHIFTS)] + [(f, "fits") for f in NARROW_ONLY],
                         ids=lambda f: "%s_%d_%d" % f if isinstance(f, tuple) else f)
@pytest.mark.parametrize("relu", [False, True])
def test_rounding_and_saturation(ctx, form, relu, shifts):
    name, ic, k = form
    dw = name == "depthwise"
    oc, g = (ic, ic) if dw else (72, 1)
    w, bias, rsh, mult = _layer(ic, oc, k, dw, shifts, ic + k)
    x = np.random.default_rng(3).integers(-128, 128, (2, ic, 12, 10)).astype(np.int8)
    p = k // 2
    mi = f2i32(mult)
    if shifts == "zeros":
        mi[:] = (1 << 30) + 64      # 6 zeros and a right shift of 10 fit, the last channel's 2^30 + 1 does not
        mi[-1] = (1 << 30) + 1
        mult = mi.astype(np.float64)
    d = conv_desc(x.shape, w.shape, g=g, pads=(p,) * 4, do_relu=relu, algo=capi.ALGO_DEPTHWISE if dw else _tile(ctx, name))
    wh = ctx.conv_prepack(d, w, f2i32(bias), mi, f2i32(rsh))
    general = shifts == "one" and "_pw_" not in name and "patch" not in name
    assert ctx.conv_algo_name(wh) == name or general
    xt, yt = ctx.from_nchw(x), ctx.tensor((2, oc, 12, 10))
    ctx._ck(ctx.lib.tpuhip_memset(ctx.h, yt.ptr, 0x55, yt.nbytes))
    ctx.conv(wh, xt, yt)
    acc = _sums(x, w, bias, p, g)
    want = _requantised(acc, mi, rsh.astype(np.int64), relu)
    assert np.array_equal(ctx.to_nchw(yt), want)
    assert yt.cs == oc or not ctx.raw(yt)[..., oc:].any()
    if shifts != "zeros":   # (the oracle takes multipliers as floats)
        assert np.array_equal(want, O.conv2d_i8(x, w, bias, rsh, mult, O.make_conv_desc(x.shape, w.shape, g, (1, 1), (p,) * 4, (1, 1),
                                                                                        (0, 0), relu, True, None)))
        assert {127, 0 if relu else -128} <= set(np.unique(want))   # (a shift of 10 alone leaves small layers within the range)
    ctx.conv_weights_destroy(wh)
    for t in (xt, yt):
        t.free()


def _sums(x, w, bias, p, g):
    n, ic, ih, iw = x.shape
    k = w.shape[2]
    xp = np.pad(x.astype(np.int64), ((0, 0), (0, 0), (p, p), (p, p)))
    out = np.zeros((n, w.shape[0], ih, iw), np.int64) + bias.astype(np.int64)[None, :, None, None]
    for i in range(k):
        for j in range(k):
            part, tap = xp[:, :, i:i + ih, j:j + iw], w[:, :, i, j].astype(np.int64)
            out += part * tap[:, 0][None, :, None, None] if g > 1 else np.tensordot(tap, part, (1, 1)).transpose(1, 0, 2, 3)
    return out


def _requantised(acc, mult, rsh, relu):
    """QuantizationArithmetic.cpp:487-539 in exact integers"""
    m, r = mult.astype(np.int64)[None, :, None, None], rsh[None, :, None, None]
    v = (acc * m + (1 << 30)) >> 31
    mask = (1 << r) - 1
    y = (v >> r) + ((v & mask) > (mask >> 1) + (v < 0))
    return np.clip(y, 0 if relu else -128, 127).astype(np.int8)


@pytest.mark.parametrize("shifts", ["fits", "one", "beyond"])
def test_stem_and_pool(ctx, shifts):
    w, bias, rsh, mult = _layer(3, 64, 7, False, shifts, 5)
    x = np.random.default_rng(4).integers(-128, 128, (2, 3, 30, 30)).astype(np.int8)
    want = O.conv2d_i8(x, w, bias, rsh, mult, O.make_conv_desc(x.shape, w.shape, 1, (2, 2), (3,) * 4, (1, 1), (0, 0), True, True, None))
    d = conv_desc(x.shape, w.shape, stride=(2, 2), pads=(3,) * 4, do_relu=True)
    wh = ctx.conv_prepack(d, w, f2i32(bias), f2i32(mult), f2i32(rsh))
    xt, yt = ctx.from_nchw(x), ctx.tensor(want.shape)
    pd = pool_desc(want.shape, (3, 3), (2, 2), (0, 1, 0, 1), (7, 7))
    pt = ctx.tensor((2, 64, 7, 7))
    ctx.conv_post(wh, xt, yt, pool=(pd, pt))
    assert np.array_equal(ctx.to_nchw(yt), want)
    padded = np.pad(want, ((0, 0), (0, 0), (0, 1), (0, 1)), constant_values=-128)
    best = np.max([padded[:, :, i:i + 13:2, j:j + 13:2] for i in range(3) for j in range(3)], axis=0)
    assert np.array_equal(ctx.to_nchw(pt), best)
    ctx.conv_weights_destroy(wh)


@pytest.mark.parametrize("shifts", [("fits", "fits"), ("fits", "one"), ("one", "fits"), ("beyond", "fits")])
@pytest.mark.parametrize("triple", [(64, 256, 64), (128, 512, 128)])
@pytest.mark.parametrize("form", ["residual", "kept", "no add"])
def test_two_convs_in_one_launch(ctx, triple, shifts, form):
    """a pointwise conv, an add and another pointwise conv: each conv requantises in its own form"""
    ic, oc1, oc2 = triple
    n, h, w_ = 2, 9, 11
    (wa, ba, ra, ma), (wb, bb, rb, mb) = _layer(ic, oc1, 1, False, shifts[0], ic), _layer(oc1, oc2, 1, False, shifts[1], oc1)
    # of every eight channels the multipliers move on by one with the shifts: all of SHIFTS are in either conv
    assert {int(v) for v in ra} == set(SHIFTS[shifts[0]]) and {int(v) for v in rb} == set(SHIFTS[shifts[1]])
    relu_a, relu_b = form == "kept", form != "kept"
    pw = lambda x, w, b, r, m, relu: O.conv2d_i8(x, w, b, r, m, O.make_conv_desc(x.shape, w.shape, 1, (1, 1), (0,) * 4, (1, 1), (0, 0),
                                                                                 relu, True, None))
    rng = np.random.default_rng(oc1 + 1)
    x = rng.integers(-128, 128, (n, ic, h, w_)).astype(np.int8)
    other = rng.integers(-128, 128, (n, oc1, h, w_)).astype(np.int8)
    ya = pw(x, wa, ba, ra, ma, relu_a)
    mid = ya if form == "no add" else O.eltwise_add_i8([other, ya], [61, 47], [6], True)
    yb = pw(mid, wb, bb, rb, mb, relu_b)
    assert {127, 0 if relu_a else -128} <= set(np.unique(ya)) and {127, 0 if relu_b else -128} <= set(np.unique(yb))
    ch = ctx.conv_chain_prepack(conv_desc(x.shape, wa.shape, do_relu=relu_a), conv_desc(ya.shape, wb.shape, do_relu=relu_b),
                                (wa, f2i32(ba), f2i32(ma), f2i32(ra)), (wb, f2i32(bb), f2i32(mb), f2i32(rb)))
    xt, ot, yat, zt, ybt = ctx.from_nchw(x), ctx.from_nchw(other), ctx.tensor(ya.shape), ctx.tensor(ya.shape), ctx.tensor(yb.shape)
    for t in (yat, zt, ybt):
        ctx._ck(ctx.lib.tpuhip_memset(ctx.h, t.ptr, 0x55, t.nbytes))
    ctx.conv_chain(ch, xt, ybt, yat if form == "kept" else None, None if form == "no add" else (ot, zt, 61, 47, 6, True))
    assert np.array_equal(ctx.to_nchw(ybt), yb)
    assert form != "kept" or np.array_equal(ctx.to_nchw(yat), ya)
    assert form == "no add" or np.array_equal(ctx.to_nchw(zt), mid)
    ctx.conv_chain_destroy(ch)
    for t in (xt, ot, yat, zt, ybt):
        t.free()
