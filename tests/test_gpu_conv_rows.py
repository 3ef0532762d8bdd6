"""The fourth form of the row-patch kernel, every variant: stride 1 and 2, maps that leave slots, rows and channel blocks over,
maps as wide as the tile, patches of more than one pass, with an add, a table, and a leaky ReLU that is computed behind them."""
import numpy as np
import pytest

import oracle_lib as O
from gpu_helpers import conv_desc, f2i32
from tpu_compiler_amd import capi

pytestmark = pytest.mark.gpu


def _name(t):
    n = capi.bind().tpuhip_conv2d_tile_name(t)
    return n.decode() if n else ""


ROWS_TILES = [t for t in range(128) if _name(t).startswith("mfma_rows_")]


def _bn(t):
    return int(_name(t).split("_")[2].split("x")[1])


def _channels(t):
    """what the input channels are a multiple of"""
    return {"c32": 32, "c64": 64}.get(_name(t).split("_")[-1][:3], 128)


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


# n, ic, ih, iw, oc, stride, relu
CASES = [
    (2, 64, 13, 11, 70, 1, True), (2, 64, 13, 11, 70, 2, False), (1, 32, 9, 128, 64, 1, False), (1, 32, 7, 127, 33, 2, True),
    (3, 128, 5, 38, 40, 1, True), (1, 256, 6, 26, 130, 1, False), (1, 512, 4, 19, 33, 2, False), (1, 1024, 3, 7, 20, 1, True),
    (1, 32, 1, 1, 16, 1, True), (2, 64, 2, 1, 16, 2, False), (1, 64, 1, 40, 290, 1, False), (1, 128, 17, 64, 300, 2, True),
    (1, 64, 40, 76, 64, 1, False), (9, 64, 3, 3, 48, 1, True), (2, 128, 13, 11, 70, 2, False), (9, 128, 3, 3, 48, 1, True),
    (1, 128, 40, 76, 129, 1, False), (1, 128, 1, 1, 16, 1, True), (1, 256, 9, 19, 100, 2, True),
]
WIDE = {160: [(1, 64, 3, 160, 40, 1, True), (1, 32, 5, 319, 40, 2, False)], 256: [(1, 64, 4, 256, 40, 1, False)],
        384: [(1, 128, 3, 384, 40, 1, True)], 192: [(1, 128, 6, 190, 40, 1, False)], 320: [(1, 32, 3, 320, 64, 1, True), (1, 64, 5, 304, 64, 1, False), (1, 32, 5, 608, 64, 2, False)],
        640: [(1, 32, 2, 640, 64, 1, False), (1, 64, 3, 304, 70, 1, True)]}


@pytest.mark.parametrize("tile,case", [(t, c) for t in ROWS_TILES for c in CASES + WIDE.get(_bn(t), []) if -(-c[3] // c[5]) <= _bn(t) and c[1] % _channels(t) == 0],
                         ids=lambda v: _name(v) if isinstance(v, int) else "x".join(map(str, v)))
@pytest.mark.parametrize("post", ["plain", "add", "table_add", "line", "line_add"])
def test_against_the_oracle(ctx, tile, case, post):
    n, ic, ih, iw, oc, s, relu = case
    rng = np.random.default_rng(ic + ih * 3 + oc + s)
    x = rng.integers(-128, 128, (n, ic, ih, iw)).astype(np.int8)
    w = np.clip(np.rint(rng.normal(0, 14, (oc, ic, 3, 3))), -127, 127).astype(np.int8)
    bias, mult = rng.integers(-4096, 4097, oc).astype(np.float32), (rng.integers(1 << 23, 1 << 24, oc) * 128).astype(np.float32)
    rsh = np.resize(np.array([2, 8, 9, 10, 11, 12, 16], np.float32), oc)
    d = conv_desc(x.shape, w.shape, stride=(s, s), pads=(1,) * 4, do_relu=relu, algo=16 + tile)
    y_ref = O.conv2d_i8(x, w, bias, rsh, mult, O.make_conv_desc(x.shape, w.shape, 1, (s, s), (1,) * 4, (1, 1), (0, 0), relu, True, None))
    xt, other = ctx.from_nchw(x), rng.integers(-128, 128, y_ref.shape).astype(np.int8)
    ot, yt, tt, zt = ctx.from_nchw(other), ctx.tensor(y_ref.shape), ctx.tensor(y_ref.shape), ctx.tensor(y_ref.shape)
    for t in (yt, tt, zt):
        ctx._ck(ctx.lib.tpuhip_memset(ctx.h, t.ptr, 0x55, t.nbytes))
    wh = ctx.conv_prepack(d, w, f2i32(bias), f2i32(mult), f2i32(rsh))
    checks = [(yt, y_ref)]
    try:
        if post == "plain":
            ctx.conv(wh, xt, yt)
        elif post == "add":
            ctx.conv_add(wh, xt, yt, ot, zt, 61, -47, 6, True)
            checks.append((zt, O.eltwise_add_i8([other, y_ref], [61, -47], [6], True)))
        elif post == "table_add":
            table = rng.integers(-128, 128, 256).astype(np.int8)
            table[0] = 77                                  # pad channels must stay 0 all the same
            t_ref = O.lut_i8(y_ref, table)
            ctx.conv_post(wh, xt, yt, table, tt, (ot, zt, 37, 51, 5, False))
            checks += [(tt, t_ref), (zt, O.eltwise_add_i8([other, t_ref], [37, 51], [5], False))]
        else:
            v = np.arange(256).astype(np.int8).astype(int)
            table = np.maximum(v, (v * 13 + 64) >> 7).astype(np.int8)      # leaky ReLU of 13 / 128: computed
            t_ref = O.lut_i8(y_ref, table)
            if post == "line":
                ctx.conv_post(wh, xt, None, table, tt)
                checks = [(tt, t_ref)]
            else:            # the residual blocks of a detector: only the sum is kept
                ctx.conv_post(wh, xt, None, table, None, (ot, zt, 37, 51, 5, False))
                checks = [(zt, O.eltwise_add_i8([other, t_ref], [37, 51], [5], False))]
    except capi.TpuHipError as e:     # a row of the patch beyond the LDS
        assert "tile variant" in str(e) and (s + 2) * iw * (ic + 16) > 140 << 10, str(e)
        checks = []
    for t, ref in checks:
        assert np.array_equal(ctx.to_nchw(t), ref) and not ctx.raw(t)[..., oc:].any()
    ctx.conv_weights_destroy(wh)
    for t in (xt, ot, yt, tt, zt):
        t.free()


@pytest.mark.parametrize("tile", ROWS_TILES)
def test_other_layers_are_refused(ctx, tile):
    """96 channels, 1x1, another padding, a map wider than the tile, a right shift of 1, dilation"""
    for shape, wshape, kw, shift in [((1, 96, 8, 8), (64, 96, 3, 3), dict(pads=(1,) * 4), 8), ((1, 128, 8, 8), (64, 128, 1, 1), {}, 8),
                                     ((1, 128, 8, 8), (64, 128, 3, 3), {}, 8), ((1, 128, 8, 700), (64, 128, 3, 3), dict(pads=(1,) * 4), 8),
                                     ((1, 128, 8, 8), (64, 128, 3, 3), dict(pads=(1,) * 4), 1),
                                     ((1, 128, 8, 8), (64, 128, 3, 3), dict(pads=(1,) * 4, dil=(2, 2)), 8)]:
        d = conv_desc(shape, wshape, algo=16 + tile, **kw)
        wh = ctx.conv_prepack(d, np.zeros(wshape, np.int8), None, np.full(64, 1 << 30, np.int32), np.full(64, shift, np.int32))
        xt, yt = ctx.tensor(shape), ctx.tensor((d.n, d.oc, d.oh, d.ow))
        with pytest.raises(capi.TpuHipError, match="tile variant"):
            ctx.conv(wh, xt, yt)
        ctx.conv_weights_destroy(wh)
        xt.free()
        yt.free()
