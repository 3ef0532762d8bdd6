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
         ("mfma_patch3_32x128", 64, 40, 3), ("mfma_ksplit_32x32_w8", 48, 41, 3), ("depthwise", 40, 40, 3),
         ("depthwise_dot", 40, 40, 3), ("depthwise", 24, 24, 5), ("stem", 3, 33, 3)]


@pytest.mark.parametrize("table", sorted(TABLES))
@pytest.mark.parametrize("form", FORMS, ids=lambda f: "%s_%d" % (f[0], f[1]))
def test_conv_with_a_line_behind_it(ctx, form, table):
    name, ic, oc, k = form
    dw = name.startswith("depthwise")
    tiles = {ctx.lib.tpuhip_conv2d_tile_name(t).decode(): t for t in range(64) if ctx.lib.tpuhip_conv2d_tile_name(t)}
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
