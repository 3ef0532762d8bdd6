"""FullyConnected of few rows, every split of its outputs over workgroups, and batches of products in the forms that the
requantisation and the columns per workgroup take."""
import numpy as np
import pytest

import oracle_lib as O
import test_gpu_ops as ops
from gpu_helpers import f2i32
from tpu_compiler_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


# rows, K, columns: blocks of 16 x 16, 16 channels x 32 rows, 32 x 32 and 32 x 64, rows and channels over, pad channels in a block
# of their own, fewer and more slices than the waves hold at once; K on both sides of what four waves hold; few channels of many rows
@pytest.mark.parametrize("m,k,n,relu", [(16, 64, 24, False), (17, 130, 1000, True), (100, 2100, 1000, False), (129, 70, 2070, True),
                                        (250, 192, 4090, False), (256, 2050, 90, True), (1, 5000, 40, False), (300, 4200, 17, True),
                                        (5, 1024, 33, True), (16, 1025, 24, False), (100, 1024, 1000, False), (32, 960, 4090, True),
                                        (250, 1024, 4090, True), (129, 1030, 2070, False), (1111, 4150, 10, True), (261, 4200, 300, False)])
def test_fully_connected_blocks(ctx, m, k, n, relu):
    ops.test_fully_connected(ctx, m, k, n, relu)


@pytest.mark.parametrize("shift", [0, 9])
def test_fully_connected_of_a_shift_of_zero(ctx, shift):
    rng = np.random.default_rng(shift)
    m, k, n = 33, 200, 70
    x, w = ops.rnd_i8(rng, (m, k)), ops.rnd_w(rng, (n, k), 20)
    bias, mult, rsh = rng.integers(-3000, 3000, n).astype(np.float32), np.float32(1 << (30 if shift else 23)), np.float32(shift)
    want = O.fc_i8(x, w, bias, [rsh], [mult], 1, m, k, n, False)[0]
    xt, yt = ctx.from_nchw(x.reshape(m, k, 1, 1)), ctx.tensor((m, n, 1, 1))
    wh = ctx.fc_prepack(m, k, n, xt.cs, yt.cs, False, w, f2i32(bias), f2i32([mult])[0], f2i32([rsh])[0])
    ctx._ck(ctx.lib.tpuhip_memset(ctx.h, yt.ptr, 0x55, yt.nbytes))
    ctx.fc(wh, xt, yt)
    assert np.array_equal(ctx.to_nchw(yt).reshape(m, n), want) and not ctx.raw(yt)[..., n:].any()
    ctx.conv_weights_destroy(wh)


# batch_high, batch_low, rows, K, columns, transposes: one to five blocks of columns in one and two workgroups, K steps around
# those in flight and around a pass through LDS, rows left over; enough products for two blocks a wave, which differs with the views
# and with one or several pairs (300 and 600 workgroups of one block)
@pytest.mark.parametrize("bh,bl,m,k,n,lt,ot", [(2, 3, 40, 128, 97, 1, 1), (1, 3, 33, 129, 129, 0, 0), (2, 2, 31, 33, 160, 1, 0),
                                               (2, 2, 64, 545, 20, 0, 1), (8, 40, 70, 40, 150, 1, 1),
                                               (1, 3, 33, 20, 70, 0, 0), (2, 2, 40, 96, 100, 1, 1), (4, 25, 90, 70, 161, 0, 1),
                                               (4, 25, 90, 70, 161, 1, 0)])
@pytest.mark.parametrize("form", ["one pair", "pairs", "shift of zero"])
def test_batched_products(ctx, bh, bl, m, k, n, lt, ot, form):
    rng = np.random.default_rng(m + k + n)
    batch = bh * bl
    x_shape = (bh, m, bl, k) if lt else (bh, bl, m, k)
    y_shape = (bh, m, bl, n) if ot else (bh, bl, m, n)
    x, w = ops.rnd_i8(rng, x_shape), ops.rnd_w(rng, (batch, n, k), 20)
    bias = rng.integers(-3000, 3000, (batch, n)).astype(np.float32)
    mult = (rng.integers(1 << 23, 1 << 24, batch) * 128).astype(np.float32)
    rsh = rng.integers(6, 11, batch).astype(np.float32)
    if form == "one pair":
        mult[:], rsh[:] = mult[0], 8
    if form == "shift of zero":
        mult[0], rsh[0] = 1 << 22, 0
    if bh == 1 and not lt and not ot:
        x_shape, y_shape = x_shape[1:], y_shape[1:]
    want = O.fc_batched_i8(x.reshape(x_shape), w, bias, rsh, mult, bh, bl, m, k, n, lt, ot, False).reshape(y_shape)
    xv, yv = ops._view4(x_shape), ops._view4(y_shape)
    xt, yt = ctx.from_nchw(x.reshape(xv)), ctx.tensor(yv)
    ctx._ck(ctx.lib.tpuhip_memset(ctx.h, yt.ptr, 0, yt.nbytes))
    d = capi.FcBatchedDesc(bh, bl, m, k, n, lt, ot, 0, xv[1], xv[2], xv[3], xt.cs, yv[1], yv[2], yv[3], yt.cs)
    wh = ctx.fc_batched_prepack(d, w, f2i32(bias), f2i32(mult), f2i32(rsh))
    ctx.fc_batched(wh, xt, yt)
    assert np.array_equal(ctx.to_nchw(yt).reshape(y_shape), want)
    assert not ctx.raw(yt)[..., yv[1]:].any()
    ctx.fc_batched_destroy(wh)
    xt.free()
    yt.free()
