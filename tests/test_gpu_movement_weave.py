"""Channel shuffles whose groups are woven in registers, and permutes through tiles of 64 and of 128 channels, at their edges."""
import numpy as np
import pytest

import oracle_lib as O
from tpu_compiler_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


def _check(ctx, kind, shape, params):
    x = np.random.default_rng(sum(shape) + len(params)).integers(-128, 128, shape).astype(np.int8)
    want = O.move_i8(kind, x, params, None)
    xt, yt = ctx.from_nchw(x), ctx.tensor(want.shape)
    ctx._ck(ctx.lib.tpuhip_memset(ctx.h, yt.ptr, 0x55, yt.nbytes))
    ctx.move(O.MOVE_KINDS.index(kind), xt, yt, params)
    assert np.array_equal(ctx.to_nchw(yt), want) and not ctx.raw(yt)[..., want.shape[1]:].any()
    xt.free()
    yt.free()


# whole groups of 16 channels, a rest, groups that begin at any byte
@pytest.mark.parametrize("groups", [2, 4])
@pytest.mark.parametrize("c", [4, 16, 20, 36, 64, 100, 132])
def test_channel_shuffle(ctx, c, groups):
    _check(ctx, "shuffle_channel", (2, c, 5, 7), [groups])


@pytest.mark.parametrize("c", [1, 63, 64, 65, 127, 128, 130, 200])
@pytest.mark.parametrize("order", [[0, 2, 3, 1], [0, 3, 1, 2], [1, 0, 2, 3]])
def test_permute(ctx, c, order):
    _check(ctx, "permute", (3, c, 66, 61), order)


# dimensions that end within tiles of j and of channels, in the runs of tiles that an XCD takes and in a grid; few of j (up to 16 and
# 32 after padding) with planes enough for wide tiles, and just not; channels in whole rounds of the XCDs
@pytest.mark.parametrize("shape,order", [((1, 66, 40, 37), [1, 0, 2, 3]), ((2, 200, 23, 31), [1, 0, 2, 3]), ((17, 130, 22, 21), [1, 0, 2, 3]),
                                         ((33, 130, 22, 21), [1, 0, 2, 3]), ((1, 1000, 9, 13), [1, 0, 2, 3]), ((3, 1030, 7, 15), [1, 0, 2, 3]),
                                         ((1, 66, 31, 16), [1, 0, 2, 3]), ((5, 192, 3, 70), [0, 2, 3, 1]), ((2, 129, 67, 5), [0, 3, 2, 1]),
                                         ((1, 65, 9, 200), [0, 3, 1, 2]), ((2, 64, 5, 130), [0, 3, 1, 2]), ((60000, 65, 1, 1), [1, 0, 2, 3]),
                                         ((1, 3, 300, 280), [1, 0, 2, 3])])
def test_permute_tiles(ctx, shape, order):
    _check(ctx, "permute", shape, order)
