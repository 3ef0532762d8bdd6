"""How transposed convs are laid out for the patch kernel (host code): whatever the shape, its fragment reads stay within the
patch, and a workgroup has the two waves or more that fetch its parameters."""
import ctypes as C
import random

import pytest

from gpu_helpers import conv_desc
from tpu_compiler_amd import capi

LIB = capi.bind()


def form(x_shape, w_shape, num_cu=256, **kw):
    reach = (C.c_int * 5)()
    f = LIB.tpuhip_conv2d_gather_form(conv_desc(x_shape, w_shape, **kw), num_cu, reach)
    return f, list(reach)


def check(f, reach):
    patch, first, end, lds, threads = reach
    if f == 2:
        assert patch <= first and end <= lds <= 160 * 1024, (patch, first, end, lds)
        assert 128 <= threads <= 1024 and threads % 64 == 0
    return f


@pytest.mark.parametrize("ic,ih,iw,oc,k,pads,ins", [
    # an odd number of 16-channel groups times an odd number of taps: the last 32-byte slice is half empty
    (144, 20, 40, 40, (3, 3), (1, 2, 1, 2), (1, 1)), (136, 5, 6, 100, (3, 3), (1, 2, 1, 2), (1, 1)),
    (272, 4, 9, 40, (3, 3), (0, 0, 0, 0), (1, 1)), (176, 9, 30, 70, (5, 5), (2, 2, 2, 2), (1, 1)),
    (240, 30, 20, 70, (3, 4), (2, 1, 3, 1), (1, 1)), (336, 47, 47, 64, (5, 3), (4, 3, 2, 2), (2, 2)),
])
def test_a_half_empty_slice_reads_within_the_patch(ic, ih, iw, oc, k, pads, ins):
    assert check(*form((1, ic, ih, iw), (oc, ic, *k), pads=pads, ins=ins)) == 2


def test_drawn_layers_read_within_the_patch():
    rng = random.Random(20)
    seen = [0, 0, 0]
    for _ in range(4000):
        ins = (rng.randint(0, 3), rng.randint(0, 3))
        k = (rng.randint(1, 6), rng.randint(1, 6))
        dil = (rng.choice((1, 1, 1, 2, 3)), rng.choice((1, 1, 1, 2, 3)))
        stride = (rng.choice((1, 1, 2, 3)), rng.choice((1, 1, 2, 3)))
        pads = tuple(rng.randint(0, dil[i // 2] * (k[i // 2] - 1)) for i in range(4))
        ic, oc = rng.choice((32, 48, 64, 80, 100, 128, 144, 256, 272, 512)), rng.randint(1, 200)
        ih, iw = rng.choice((1, 1, 2, 5, 9, 20, 33, 60)), rng.choice((1, 1, 2, 7, 12, 31, 53, 90))
        d = dict(stride=stride, pads=pads, dil=dil, ins=ins)
        if conv_desc((1, ic, ih, iw), (oc, ic, *k), **d).oh <= 0 or conv_desc((1, ic, ih, iw), (oc, ic, *k), **d).ow <= 0:
            continue
        seen[check(*form((rng.choice((1, 2, 8)), ic, ih, iw), (oc, ic, *k), num_cu=rng.choice((256, 256, 64)), **d))] += 1
    assert seen[1] > 300 and seen[2] > 300, seen
