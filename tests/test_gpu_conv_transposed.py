"""Transposed convs of eight 32-byte slices or more per output (zeros between the input's pixels): phases that differ in size
and in taps or have none, strides and dilations against the zeros, odd numbers of 16-channel groups, ragged tiles and channel
blocks, patches past 64 KB, and both sides of the rule that takes a layer to the patch kernel."""
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


PLAIN, PATCH = 1, 2   # tpuhip_conv2d_gather_form on 256 CUs
# n, ic, ih, iw, oc, (kh, kw), stride, pads (t, b, l, r), dil, ins, relu, relu_first, kernel
CASES = [
    (2, 128, 13, 11, 70, (4, 4), (1, 1), (2, 2, 2, 2), (1, 1), (1, 1), True, 0, PATCH),
    (1, 64, 9, 33, 33, (4, 4), (1, 1), (2, 2, 2, 2), (1, 1), (1, 1), False, 1, PATCH),             # eight slices; relu before
    (1, 48, 9, 33, 33, (4, 4), (1, 1), (2, 2, 2, 2), (1, 1), (1, 1), False, 0, PLAIN),             # six: the other kernel
    (3, 80, 6, 7, 16, (4, 4), (1, 1), (2, 1, 1, 2), (1, 1), (1, 1), True, 0, PLAIN),               # 5 groups of 16, odd result sizes
    (3, 80, 6, 7, 70, (4, 4), (1, 1), (2, 1, 1, 2), (1, 1), (1, 1), True, 0, PATCH),               # of more than one channel block
    (1, 136, 5, 6, 100, (3, 3), (1, 1), (1, 2, 1, 2), (1, 1), (1, 1), False, 0, PATCH),            # taps 1, 2, 2, 4; odd counts of entries
    (1, 144, 20, 40, 40, (3, 3), (1, 1), (1, 2, 1, 2), (1, 1), (1, 1), False, 0, PATCH),           # likewise, many channels a slice
    (2, 272, 4, 9, 40, (3, 3), (1, 1), (0, 0, 0, 0), (1, 1), (1, 1), True, 0, PATCH),              # 17 groups of 16
    (1, 256, 6, 5, 40, (2, 2), (1, 1), (0, 1, 0, 1), (1, 1), (2, 2), True, 0, PLAIN),              # phases without a tap
    (1, 128, 7, 6, 20, (4, 3), (1, 1), (2, 2, 1, 1), (1, 1), (1, 0), False, 0, PATCH),             # two phases
    (1, 64, 7, 8, 64, (5, 4), (3, 3), (3, 2, 2, 2), (1, 1), (1, 1), True, 0, PATCH),               # stride 3 against the zeros
    (1, 64, 8, 9, 33, (4, 4), (1, 2), (3, 3, 3, 3), (2, 1), (2, 2), False, 0, PLAIN),              # nine phases, stride and dilation
    (2, 512, 1, 1, 40, (4, 4), (1, 1), (3, 3, 3, 3), (1, 1), (1, 1), True, 0, PATCH),              # one pixel to 4 x 4
    (1, 512, 2, 1, 24, (2, 3), (1, 1), (0, 0, 1, 1), (1, 1), (1, 1), False, 0, PATCH),             # a single result column
    (1, 256, 1, 1, 40, (3, 3), (1, 1), (1, 1, 1, 1), (1, 1), (1, 1), False, 0, PLAIN),             # one phase of results: the other kernel
    (3, 256, 5, 1, 70, (3, 3), (1, 1), (1, 1, 1, 1), (1, 1), (0, 1), True, 0, PLAIN),              # likewise, of one column
    (2, 384, 1, 6, 24, (3, 3), (1, 1), (1, 1, 1, 1), (1, 1), (1, 0), False, 1, PLAIN),             # and of one row
    (1, 256, 5, 101, 40, (4, 4), (1, 1), (2, 2, 2, 2), (1, 1), (1, 1), True, 0, PATCH),            # three rows of patch: 84 KB
    (1, 256, 3, 250, 36, (4, 4), (1, 1), (2, 2, 2, 2), (1, 1), (1, 1), True, 0, PLAIN),            # no patch: the other kernel
    (1, 64, 201, 200, 8, (4, 4), (1, 1), (2, 2, 2, 2), (1, 1), (1, 1), True, 0, PATCH),
    (1, 64, 200, 200, 8, (4, 4), (1, 1), (2, 2, 2, 2), (1, 1), (1, 1), False, 0, PATCH),
    (1, 64, 340, 340, 8, (4, 4), (1, 1), (2, 2, 2, 2), (1, 1), (1, 1), True, 0, PLAIN),            # many outputs: the other kernel
    (1, 80, 96, 96, 16, (4, 4), (1, 1), (2, 2, 2, 2), (1, 1), (1, 1), True, 0, PATCH),             # one channel block: 36864 outputs
    (1, 80, 96, 95, 16, (4, 4), (1, 1), (2, 2, 2, 2), (1, 1), (1, 1), False, 0, PLAIN),            # fewer: the other kernel
    (2, 256, 33, 32, 70, (2, 2), (1, 1), (0, 1, 0, 1), (1, 1), (2, 2), True, 0, PATCH),            # nine phases, some without a tap
    (4, 128, 24, 49, 33, (4, 4), (1, 2), (3, 3, 3, 3), (2, 1), (2, 2), False, 0, PATCH),           # nine phases, stride and dilation
    (2, 112, 40, 35, 70, (6, 6), (1, 1), (4, 4, 4, 4), (1, 1), (2, 2), True, 0, PLAIN),            # fewer than 128 channels
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:5])))
@pytest.mark.parametrize("smallest_shift", [0, 1])
def test_against_the_oracle(ctx, case, smallest_shift):
    n, ic, ih, iw, oc, k, stride, pads, dil, ins, relu, relu_first, kernel = case
    rng = np.random.default_rng(ic + ih * 3 + oc + k[0])
    x = rng.integers(-128, 128, (n, ic, ih, iw)).astype(np.int8)
    w = np.clip(np.rint(rng.normal(0, 16, (oc, ic, *k))), -127, 127).astype(np.int8)
    bias, mult = rng.integers(-4096, 4097, oc).astype(np.float32), (rng.integers(1 << 23, 1 << 24, oc) * 128).astype(np.float32)
    rsh = rng.integers(7, 12, oc).astype(np.float32)
    rsh[::7] = smallest_shift                       # 0: the form of the requantisation that may overflow
    if relu_first:   # relu before the requantisation with multipliers above 0 is relu after it
        relu = True
    want = O.conv2d_i8(x, w, bias, rsh, mult, O.make_conv_desc(x.shape, w.shape, 1, stride, pads, dil, ins, relu, True, None))
    d = conv_desc(x.shape, w.shape, stride=stride, pads=pads, dil=dil, ins=ins, do_relu=relu, relu_first=relu_first)
    assert ctx.lib.tpuhip_conv2d_gather_form(d, 256, None) == kernel
    xt, yt = ctx.from_nchw(x), ctx.tensor(want.shape)
    ctx._ck(ctx.lib.tpuhip_memset(ctx.h, yt.ptr, 0x55, yt.nbytes))
    wh = ctx.conv_prepack(d, w, f2i32(bias), f2i32(mult), f2i32(rsh))
    ctx.conv(wh, xt, yt)
    assert np.array_equal(ctx.to_nchw(yt), want) and not ctx.raw(yt)[..., oc:].any()
    assert len(np.unique(want)) > 8
    ctx.conv_weights_destroy(wh)
    xt.free()
    yt.free()
