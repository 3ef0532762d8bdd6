"""The stem kernel of layers that requantise on packed int16: images whose rows are and are not whole 16-byte chunks, pixels of 4
and 16 bytes, kernels up to 7 x 8, paddings up to the patch's own, ragged last tiles, one row and one column of results, and the
layers that stay with the other stem kernel (a right shift of 1)."""
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


# n, ic, ih, iw, oc, (kh, kw), (sh, sw), pads (t, b, l, r), x_cs, relu
CASES = [
    (2, 3, 24, 32, 32, (3, 3), (1, 1), (1, 1, 1, 1), 4, True),
    (40, 3, 30, 32, 32, (3, 3), (1, 1), (1, 1, 1, 1), 4, True), (70, 3, 34, 32, 32, (3, 3), (2, 2), (1, 1, 1, 1), 4, False),
    (70, 3, 19, 45, 24, (3, 3), (1, 1), (1, 1, 1, 1), 4, False), (140, 3, 19, 45, 24, (3, 3), (2, 2), (0, 1, 0, 1), 16, True),
    (70, 4, 17, 30, 64, (7, 7), (2, 2), (3, 3, 3, 3), 4, True), (70, 4, 31, 36, 33, (7, 8), (3, 2), (3, 3, 8, 7), 4, False),
    (40, 1, 40, 28, 7, (5, 5), (1, 1), (2, 2, 2, 2), 16, True), (70, 2, 9, 300, 40, (1, 4), (1, 1), (0, 0, 0, 3), 4, False),
    (1200, 3, 3, 32, 16, (3, 3), (1, 1), (0, 0, 1, 1), 4, True), (40, 3, 40, 3, 16, (3, 3), (1, 1), (1, 1, 0, 0), 4, True),
    (150, 3, 8, 2, 16, (3, 2), (1, 1), (1, 1, 1, 0), 4, False), (70, 3, 64, 64, 32, (3, 3), (2, 2), (1, 1, 1, 1), 4, True),
    (40, 3, 60, 61, 64, (7, 7), (2, 2), (3, 3, 3, 3), 4, False), (9, 3, 130, 257, 20, (3, 3), (1, 1), (1, 1, 1, 1), 4, True),
    (11, 3, 8, 1700, 64, (7, 7), (1, 1), (3, 3, 3, 3), 4, True),
]
# few tiles, one column of results, and a patch of one row that passes its share of LDS
OTHER_KERNEL = [CASES[0], CASES[10], (11, 3, 8, 2400, 64, (7, 7), (1, 1), (3, 3, 3, 3), 4, True)]
CASES += OTHER_KERNEL[2:]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:5])))
@pytest.mark.parametrize("post", ["plain", "leaky", "table", "shift_1"])
def test_against_the_oracle(ctx, case, post):
    n, ic, ih, iw, oc, k, s, pads, x_cs, relu = case
    rows = case not in OTHER_KERNEL and post != "shift_1"
    rng = np.random.default_rng(ic + ih * 3 + oc + k[0] * 7)
    x = rng.integers(-128, 128, (n, ic, ih, iw)).astype(np.int8)
    w = np.clip(np.rint(rng.normal(0, 40, (oc, ic, *k))), -127, 127).astype(np.int8)
    bias, mult = rng.integers(-4096, 4097, oc).astype(np.float32), (rng.integers(1 << 23, 1 << 24, oc) * 128).astype(np.float32)
    rsh = np.resize(np.array([2, 7, 8, 9, 10, 11, 16], np.float32), oc)
    if post == "shift_1":
        rsh[0] = 1
    d = conv_desc(x.shape, w.shape, stride=s, pads=pads, do_relu=relu, x_cs=x_cs)
    want = O.conv2d_i8(x, w, bias, rsh, mult, O.make_conv_desc(x.shape, w.shape, 1, s, pads, (1, 1), (0, 0), relu, True, None))
    xt, yt, tt = ctx.from_nchw(x, x_cs), ctx.tensor(want.shape), ctx.tensor(want.shape)
    for t in (yt, tt):
        ctx._ck(ctx.lib.tpuhip_memset(ctx.h, t.ptr, 0x55, t.nbytes))
    wh = ctx.conv_prepack(d, w, f2i32(bias), f2i32(mult), f2i32(rsh))
    assert ctx.conv_algo_name(wh) == "stem" and (ctx.lib.tpuhip_conv2d_stem_rows(wh) > 0) == rows
    if post == "leaky":
        table = ctx.leaky_relu_table(0, 1, 10, 102)
        ctx.conv_post(wh, xt, yt, table, tt)
        checks = [(yt, want), (tt, O.lut_i8(want, table))]
    elif post == "table":
        table = rng.integers(-128, 128, 256).astype(np.int8)
        table[0] = 77                                  # pad channels must stay 0 all the same
        ctx.conv_post(wh, xt, None, table, tt)
        checks = [(tt, O.lut_i8(want, table))]
    else:
        ctx.conv(wh, xt, yt)
        checks = [(yt, want)]
    for t, ref in checks:
        assert np.array_equal(ctx.to_nchw(t), ref) and not ctx.raw(t)[..., oc:].any()
    ctx.conv_weights_destroy(wh)
    for t in (xt, yt, tt):
        t.free()
