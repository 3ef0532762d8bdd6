"""The stem with its max pool where the input patch ends at or beside a load of the whole workgroup (512 dwords), and average
pools whose windows eight lanes share, at the least and most positions, with ragged channels, pads and the last lanes idle."""
import numpy as np
import pytest

import oracle_graph
import oracle_lib as O
from gpu_helpers import pool_desc
from tpu_compiler_amd import capi, module
from tpu_compiler_amd.graphs import BASE_SEED, Builder

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


# one tile's patch: 11 rows of 2 * (conv columns - 1) + 8 dwords, rounded to 4: 5632 = 11 loads, then 12, then 5 and 1
# -- and batches whose tiles are of two, three (the last of two rows) and more pooled rows
@pytest.mark.parametrize("n,h,w", [(2, 22, 505), (2, 22, 507), (2, 13, 503), (2, 30, 224), (2, 9, 11),
                                   (40, 33, 20), (70, 33, 20), (100, 41, 12), (257, 13, 9)])
def test_stem_with_pool_tiles(n, h, w):
    b = Builder("stem", BASE_SEED + w, n, (6, 16))
    x = b.input("input", 3, h, w)
    c = b.conv("conv", x, 64, 7, stride=2, pad=3, relu=True)
    p = b.pool_max("pool", c, 3, 2, (0, 1, 0, 1))
    g = b.finish([p])
    want = oracle_graph.run(g)
    for keep in (1, 0):
        m = module()
        m.set_option("keep_all_tensors", keep)
        m.load(g)
        assert dict(m.kernels())["conv"] == "stem"
        m.set_tensor("input", g.input_op().data.astype(np.float32))
        m.invoke()
        for name in ("pool", "conv")[:1 + keep]:
            assert np.array_equal(m.get_tensor_i8(name), want[name].reshape(g.by_name[name].shape)), (keep, name)
        m.close()


@pytest.mark.parametrize("k,s,pads", [((4, 4), (1, 1), (0, 0, 0, 0)), ((1, 17), (1, 3), (0, 0, 0, 0)), ((7, 9), (2, 2), (3, 3, 4, 4)),
                                      ((8, 8), (8, 8), (0, 0, 0, 0)), ((8, 8), (3, 1), (4, 3, 5, 2))])
@pytest.mark.parametrize("n,c", [(1, 1), (3, 15), (2, 17), (1, 300)])
@pytest.mark.parametrize("mult,rs", [(85, 12), (255, 3)])      # (255, 3): every sum but the smallest saturates
def test_average_of_windows_that_eight_lanes_share(ctx, k, s, pads, n, c, mult, rs):
    shape = (n, c, 19, 18)
    x = np.random.default_rng(c + k[1]).integers(-128, 128, shape).astype(np.int8)
    want = O.pool_avg_i8(x, O.make_pool_desc(shape, k, s, pads), rs, mult)
    d = pool_desc(shape, k, s, pads)
    xt, yt = ctx.from_nchw(x), ctx.tensor(want.shape)
    ctx._ck(ctx.lib.tpuhip_memset(ctx.h, yt.ptr, 0x55, yt.nbytes))
    ctx.pool_avg(d, xt, yt, mult, rs)
    assert np.array_equal(ctx.to_nchw(yt), want) and not ctx.raw(yt)[..., c:].any()
    xt.free()
    yt.free()
