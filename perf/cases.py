"""The work that is timed: what a user of the INT8 interpreter has it do, through its public entry points.

Whole networks go through `tpu_compiler_amd.module` the way pymlir's users drive it (load once, then host array
in, host array out, per batch); single ops go through `tpu_compiler_amd.capi.Context` on tensors in device
memory, the way a host that swaps single kernels calls them.  All tensors are int8 or float-stored integers, so
every result is exact.

Kinds of case and the ranges draw() takes them from:
  net    a whole network: residual bottleneck classifier, inverted-residual classifier, or one-stage detector;
         1 to 64 images (1 to 8 for the detector), sides of 96 to 288 (320 to 608) pixels, float or int8 at the
         host, every tensor kept or the outputs only
  dump   a residual backbone whose every tensor is read back, as accuracy comparisons do
  file   the tool flow: model and weights from files, one input file in, one output file out
  conv   one conv, or a depthwise and a pointwise conv behind each other: 1 to 16 images of 7 to 112 pixels a side
  zoo    the convs that are not plain: grouped, dilated, transposed, large kernel with stride
  mix    the elementwise, table, pooling and joining ops of a feature map
  move   the data-movement ops
  fc     a classifier matrix product and a batch of transposed ones
"""
import os
import tempfile

import numpy as np
import torch

from tpu_compiler_amd import capi, graphs, mlir_text, module

SIGMA = 32.0     # spread of the int8 weights
LEVEL = 40.0     # root mean square the requantisation shifts aim at


def listed():
    return [
        # the smallest call there is: one 3x3 conv of one image, tensors resident
        dict(name="conv_one_image", kind="conv", form="dense", n=1, ic=64, oc=64, k=3, h=56, w=56),
        # a classifier on one image, host to host: latency of ~50 dependent layers
        dict(name="classifier_one_image", kind="net", net="bottleneck", batch=1, side=224, io="f32", keep=True),
        # the same serving batches of bytes, outputs only: the repository's headline configuration
        dict(name="classifier_batch_32", kind="net", net="bottleneck", batch=32, side=224, io="i8", keep=False),
        # the light classifier on large float batches
        dict(name="light_classifier_batch_64", kind="net", net="inverted", batch=64, side=224, io="f32", keep=True),
        # the detector at its full size and batch: the largest work
        dict(name="detector_batch_8", kind="net", net="detector", batch=8, side=608, io="i8", keep=False),
        # the detector on one smaller image, float maps of three heads back to the host
        dict(name="detector_one_image", kind="net", net="detector", batch=1, side=416, io="f32", keep=True),
        # every tensor of a backbone to the host, odd side: comparing layer by layer
        dict(name="backbone_dump", kind="dump", blocks=7, batch=2, side=193),
        # from files to a file: what a command-line run pays for, loading included
        dict(name="file_run", kind="file", net="inverted", batch=1, side=160),
        # feature-map ops on a ragged map and channel count
        dict(name="map_ops", kind="mix", n=4, c=120, h=75, w=75),
        # data movement on a ragged map
        dict(name="movement_ops", kind="move", n=4, c=96, h=78, w=66),
        # matrix products
        dict(name="matrix_products", kind="fc", m=100, k=2048, n=1000, bh=4, bl=8, bm=160, bk=64, bn=160),
        # grouped, dilated, transposed and large-kernel convs
        dict(name="conv_variants", kind="zoo", n=4, c=128, h=45, w=53),
    ]


def _log(rng, lo, hi):
    return int(round(2.0 ** rng.uniform(np.log2(lo), np.log2(hi))))


def draw(rng):
    kind = rng.choice(["net", "net", "net", "dump", "file", "conv", "conv", "zoo", "mix", "move", "fc"])
    if kind == "net":
        net = rng.choice(["bottleneck", "inverted", "detector"])
        if net == "detector":
            side, batch = 32 * rng.randint(10, 19), _log(rng, 1, 8)
        else:
            side, batch = rng.randint(96, 288), _log(rng, 1, 64)
            while batch * side * side > 64 * 224 * 224:
                batch -= 1
        return dict(kind="net", net=net, batch=batch, side=side, io=rng.choice(["f32", "i8"]),
                    keep=rng.random() < 0.5)
    if kind == "dump":
        return dict(kind="dump", blocks=rng.randint(3, 10), batch=rng.randint(1, 4), side=rng.randint(96, 224))
    if kind == "file":
        return dict(kind="file", net="inverted", batch=rng.randint(1, 4), side=rng.randint(96, 224))
    if kind == "conv":
        n = _log(rng, 1, 16)
        h, w = _log(rng, 7, 112), _log(rng, 7, 112)
        if rng.random() < 0.4:
            return dict(kind="conv", form="separable", n=n, ic=rng.randint(2, 40) * 8, oc=rng.randint(2, 48) * 8,
                        k=3, h=h, w=w)
        return dict(kind="conv", form="dense", n=n, ic=_log(rng, 16, 512), oc=_log(rng, 16, 512),
                    k=rng.choice([1, 3]), h=h, w=w)
    n = _log(rng, 1, 16)
    h, w = rng.randint(10, 112), rng.randint(10, 112)
    if kind == "zoo":
        return dict(kind="zoo", n=min(n, 8), c=32 * rng.randint(1, 8), h=h // 2 + 4, w=w // 2 + 4)
    if kind == "mix":
        return dict(kind="mix", n=n, c=rng.randint(8, 400), h=h, w=w)
    if kind == "move":
        return dict(kind="move", n=n, c=8 * rng.randint(1, 40), h=2 * (h // 2), w=2 * (w // 2))
    return dict(kind="fc", m=_log(rng, 1, 256), k=_log(rng, 64, 8192), n=_log(rng, 10, 4096), bh=rng.randint(1, 8),
                bl=rng.randint(1, 12), bm=_log(rng, 8, 384), bk=rng.randint(2, 16) * 8, bn=_log(rng, 8, 384))


# -- networks ---------------------------------------------------------------------------------------------------------

#: int8 values of N(0, SIGMA) at 65536 evenly spaced quantiles: a uniform 16-bit draw indexes it
_NORMAL = np.clip(np.rint(torch.special.ndtri((torch.arange(65536, dtype=torch.float64) + 0.5) / 65536).numpy() * SIGMA),
                  -127, 127).astype(np.float32)


class _Net:
    """Appends quantised ops to a graph; the shifts keep every activation near LEVEL, estimated from the weights."""

    def __init__(self, name):
        self.g = graphs.Graph(name, 1)
        self.rng = np.random.default_rng(20)
        self.rms = {}
        self.flops = 0
        self.weights = 0

    def _op(self, op, rms):
        self.g.add(op)
        self.rms[op.name] = rms
        return op.name

    def shape(self, src):
        return self.g.by_name[src].shape

    def input(self, n, c, h, w):
        return self._op(graphs.Op("tpu.input", "input", [], (n, c, h, w)), 73.9)

    def conv(self, name, src, oc, k, stride=1, groups=1, relu=False):
        n, ic, ih, iw = self.shape(src)
        p = k // 2
        oh, ow = (ih + 2 * p - k) // stride + 1, (iw + 2 * p - k) // stride + 1
        w = _NORMAL[self.rng.integers(0, 65536, (oc, ic // groups, k, k), dtype=np.uint16)]
        mult = self.rng.integers(1 << 23, 1 << 24, oc) * 128.0
        acc = self.rms[src] * np.sqrt((w.reshape(oc, -1) ** 2).sum(1)) * mult / 2.0 ** 31
        attrs = dict(kernel_h=k, kernel_w=k, stride_h=stride, stride_w=stride, dilation_h=1, dilation_w=1, padding_t=p,
                     padding_b=p, padding_l=p, padding_r=p, group=groups, is_dw=int(groups > 1), with_bias=1,
                     do_relu=int(relu), pad_value=0)
        weights = dict(filter=w if groups == 1 else w.reshape(groups, oc // groups, ic // groups, k, k),
                       bias=self.rng.integers(-4096, 4097, oc).astype(np.float32),
                       rshift=np.clip(np.rint(np.log2(np.maximum(acc, 1.0) / LEVEL)), 1, 18).astype(np.float32),
                       multiplier=mult.astype(np.float32))
        self.flops += 2 * n * oc * oh * ow * (ic // groups) * k * k
        self.weights += w.size + 12 * oc
        return self._op(graphs.Op("tpu.conv_2d", name, [src], (n, oc, oh, ow), attrs, weights, "RSHIFT_AND_M_I32"),
                        LEVEL * (0.7 if relu else 1.0))

    def add(self, name, a, b, relu):
        m = self.rng.integers(40, 101, 2)
        rms = np.sqrt((m[0] * self.rms[a]) ** 2 + (m[1] * self.rms[b]) ** 2)
        r = int(np.clip(np.rint(np.log2(rms / LEVEL)), 0, 14))
        return self._op(graphs.Op("tpu.eltwise_add", name, [a, b], self.shape(a), dict(do_relu=int(relu)),
                                  dict(rshift=np.array([r], np.float32), multiplier=m.astype(np.float32)),
                                  "RSHIFT_AND_M_I8"), LEVEL * (0.7 if relu else 1.0))

    def leaky(self, src):
        one = lambda v: np.array([v], np.float32)
        return self._op(graphs.Op("tpu.leaky_relu", src + "_leaky", [src], self.shape(src), dict(negative_slope=0.1),
                                  dict(rshift_pos=one(0), multiplier_pos=one(1), rshift_neg=one(7),
                                       multiplier_neg=one(13)), "RSHIFT_AND_M_I8"), 0.71 * self.rms[src])

    def max_pool(self, name, src):
        n, c, h, w = self.shape(src)
        oh, ow = -(-(h - 3) // 2) + 1, -(-(w - 3) // 2) + 1
        return self._op(graphs.Op("tpu.pool_max_2d", name, [src], (n, c, oh, ow),
                                  dict(kernel_h=3, kernel_w=3, stride_h=2, stride_w=2, padding_t=0,
                                       padding_b=(oh - 1) * 2 + 3 - h, padding_l=0, padding_r=(ow - 1) * 2 + 3 - w,
                                       do_relu=0, count_include_pad=0, pad_value=0)), 1.4 * self.rms[src])

    def classify(self, src, classes):
        n, c, h, w = self.shape(src)
        mult = int(np.clip(np.rint(2.0 ** 13 * LEVEL / (h * w * 18.0)), 1, 255))
        src = self._op(graphs.Op("tpu.pool_avg_2d", "pool", [src], (n, c, 1, 1),
                                 dict(kernel_h=h, kernel_w=w, stride_h=1, stride_w=1, padding_t=0, padding_b=0,
                                      padding_l=0, padding_r=0, do_relu=0, count_include_pad=1, pad_value=0),
                                 dict(rshift=np.array([13], np.float32), multiplier=np.array([mult], np.float32)),
                                 "RSHIFT_AND_M_I8"), LEVEL)
        src = self._op(graphs.Op("tpu.reshape", "pool_flat", [src], (n, c)), LEVEL)
        w = _NORMAL[self.rng.integers(0, 65536, (classes, c), dtype=np.uint16)]
        r = int(np.rint(np.log2(LEVEL * SIGMA * c ** 0.5 * 0.75 / LEVEL)))
        self.flops += 2 * n * c * classes
        self.weights += w.size + 4 * classes
        return self._op(graphs.Op("tpu.fully_connected", "fc", [src], (n, classes), dict(do_relu=0),
                                  dict(filter=w, bias=self.rng.integers(-2048, 2049, classes).astype(np.float32),
                                       rshift=np.array([r], np.float32),
                                       multiplier=np.array([3 << 29], np.float32)), "RSHIFT_AND_M_I32"), LEVEL)

    def upsample(self, name, src):
        n, c, h, w = self.shape(src)
        return self._op(graphs.Op("tpu.upsample", name, [src], (n, c, 2 * h, 2 * w), dict(scale_h=2, scale_w=2)),
                        self.rms[src])

    def concat(self, name, a, b):
        n, c, h, w = self.shape(a)
        return self._op(graphs.Op("tpu.concat", name, [a, b], (n, c + self.shape(b)[1], h, w),
                                  dict(axis=1, do_relu=0)), self.rms[a])

    def done(self, outputs):
        self.g.outputs = list(outputs)
        self.outputs = sum(int(np.prod(self.shape(o))) for o in outputs)
        return self


def _bottleneck(batch, side, blocks=16, classify=True):
    net = _Net("bottleneck")
    x = net.input(batch, 3, side, side)
    x = net.conv("conv1", x, 64, 7, stride=2, relu=True)
    x = net.max_pool("pool1", x)
    done = 0
    for stage, (count, mid) in enumerate(((3, 64), (4, 128), (6, 256), (3, 512))):
        for b in range(min(count, blocks - done)):
            p, stride = "res%d%s" % (stage + 2, "abcdef"[b]), 2 if b == 0 and stage else 1
            sc = net.conv(p + "_branch1", x, mid * 4, 1, stride=stride) if b == 0 else x
            y = net.conv(p + "_branch2a", x, mid, 1, stride=stride, relu=True)
            y = net.conv(p + "_branch2b", y, mid, 3, relu=True)
            y = net.conv(p + "_branch2c", y, mid * 4, 1)
            x = net.add(p, sc, y, True)
        done = min(blocks, done + count)
    return net.done([net.classify(x, 1000) if classify else x])


def _inverted(batch, side):
    net = _Net("inverted")
    x = net.input(batch, 3, side, side)
    x = net.conv("conv1", x, 32, 3, stride=2, relu=True)
    cin, idx = 32, 0
    for t, c, count, s in ((1, 16, 1, 1), (6, 24, 2, 2), (6, 32, 3, 2), (6, 64, 4, 2), (6, 96, 3, 1), (6, 160, 3, 2),
                           (6, 320, 1, 1)):
        for i in range(count):
            idx, stride, y = idx + 1, s if i == 0 else 1, x
            p = "block%d" % idx
            if t != 1:
                y = net.conv(p + "_expand", y, cin * t, 1, relu=True)
            y = net.conv(p + "_dw", y, cin * t, 3, stride=stride, groups=cin * t, relu=True)
            y = net.conv(p + "_project", y, c, 1)
            x = net.add(p + "_add", x, y, False) if stride == 1 and cin == c else y
            cin = c
    return net.done([net.classify(net.conv("conv_last", x, 1280, 1, relu=True), 1000)])


def _detector(batch, side):
    net = _Net("detector")
    count = [0]

    def cbl(x, oc, k, stride=1):
        count[0] += 1
        return net.leaky(net.conv("conv%d" % count[0], x, oc, k, stride=stride))

    x = cbl(net.input(batch, 3, side, side), 32, 3)
    routes = []
    for oc, blocks in ((64, 1), (128, 2), (256, 8), (512, 8), (1024, 4)):
        x = cbl(x, oc, 3, stride=2)
        for _ in range(blocks):
            x = net.add("res%d" % count[0], x, cbl(cbl(x, oc // 2, 1), oc, 3), False)
        routes.append(x)
    outs = []
    for mid, route in ((512, None), (256, 3), (128, 2)):
        if route is not None:
            x = net.concat("route%d" % mid, net.upsample("up%d" % mid, cbl(x, mid, 1)), routes[route])
        for _ in range(2):
            x = cbl(cbl(x, mid, 1), mid * 2, 3)
        x = cbl(x, mid, 1)
        outs.append(net.conv("head%d" % mid, cbl(x, mid * 2, 3), 255, 1))
    return net.done(outs)


_NETS = {"bottleneck": _bottleneck, "inverted": _inverted, "detector": _detector}
_kept = {}       # what a user's program loads once: modules, packed weights


def _once(case, make):
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    if key not in _kept:
        _kept[key] = make()
    return _kept[key]


def _build(case):
    if case["kind"] == "dump":
        return _bottleneck(case["batch"], case["side"], case["blocks"], classify=False)
    return _NETS[case["net"]](case["batch"], case["side"])


def _load(case):
    net = _build(case)
    m = module()
    m.set_option("keep_all_tensors", int(case.get("keep", True)))
    m.load(net.g)
    return m, net.g.outputs


def _write_files(case):
    folder = tempfile.TemporaryDirectory(prefix="tpuhip_case_")
    net = _build(case)
    mlir_text.write_mlir(net.g, os.path.join(folder.name, "model.mlir"))
    return folder, net.g.outputs


# -- single ops -------------------------------------------------------------------------------------------------------

_ctx = []


def _context():
    if not _ctx:
        _ctx.append(capi.Context(0))
    return _ctx[0]


class _Map(capi.DeviceTensor):
    """A channels-last tensor of the library in memory that torch holds."""

    def __init__(self, shape, fill=None):
        n, c, h, w = shape
        cs = capi.channel_stride(c)
        self.store = torch.zeros(n * h * w * cs + 256, dtype=torch.int8, device="cuda")
        self.view = self.store[:n * h * w * cs].view(n, h, w, cs)
        if fill is not None:
            self.view[..., :c] = torch.randint(-128, 128, (n, h, w, c), dtype=torch.int8, device="cuda", generator=fill)
        super().__init__(_context(), shape, cs, ptr=self.store.data_ptr(), owner=False)


def _pack(rng, oc, icg, k, ic, hw_in, hw_out, n, stride=1, pads=(0, 0, 0, 0), dil=1, groups=1, ins=0, relu=True):
    w = _NORMAL[rng.integers(0, 65536, (oc, icg, k, k), dtype=np.uint16)].astype(np.int8)
    mult = (rng.integers(1 << 23, 1 << 24, oc) * 128).astype(np.int32)
    live = icg * k * k / float((1 + ins) ** 2)
    r = np.rint(np.log2(73.9 * SIGMA * live ** 0.5 * mult / 2.0 ** 31 / LEVEL))
    d = capi.ConvDesc(n, ic, hw_in[0], hw_in[1], oc, hw_out[0], hw_out[1], groups, k, k, stride, stride, *pads, dil, dil,
                      ins, ins, int(relu), 1, capi.channel_stride(ic), capi.channel_stride(oc), 0, 0)
    return _context().conv_prepack(d, w, rng.integers(-4096, 4097, oc).astype(np.int32), mult,
                                   np.maximum(r, 1).astype(np.int32))


def _conv_handles(case):
    rng = np.random.default_rng(21)
    n, hw, k = case["n"], (case["h"], case["w"]), case["k"]
    p = k // 2
    if case["form"] == "dense":
        return (_pack(rng, case["oc"], case["ic"], k, case["ic"], hw, hw, n, pads=(p,) * 4),)
    return (_pack(rng, case["ic"], 1, k, case["ic"], hw, hw, n, pads=(p,) * 4, groups=case["ic"]),
            _pack(rng, case["oc"], case["ic"], 1, case["ic"], hw, hw, n))


def _zoo_shapes(case):
    """(input side pair, output side pair, kernel, stride, pads, dilation, groups, inserted zeros) per conv"""
    h, w = case["h"], case["w"]
    return [((h, w), (h, w), 3, 1, (1,) * 4, 1, 32, 0),                                # grouped
            ((h, w), (h, w), 3, 1, (2,) * 4, 2, 1, 0),                                 # dilated
            ((h, w), (2 * h, 2 * w), 4, 1, (2,) * 4, 1, 1, 1),                         # transposed, doubles the map
            ((h, w), ((h + 1) // 2, (w + 1) // 2), 5, 2, (2,) * 4, 1, 1, 0)]           # large kernel, stride


def _zoo_handles(case):
    rng, c = np.random.default_rng(22), case["c"]
    return [_pack(rng, c, c // g, k, c, i, o, case["n"], s, pads, dil, g, ins)
            for i, o, k, s, pads, dil, g, ins in _zoo_shapes(case)]


def _fc_handles(case):
    rng, ctx = np.random.default_rng(23), _context()
    shift = lambda k: int(max(1, np.rint(np.log2(73.9 * SIGMA * k ** 0.5 * 0.75 / LEVEL))))
    m, k, n = case["m"], case["k"], case["n"]
    normal = lambda *s: _NORMAL[rng.integers(0, 65536, s, dtype=np.uint16)].astype(np.int8)
    one = ctx.fc_prepack(m, k, n, capi.channel_stride(k), capi.channel_stride(n), 0, normal(n, k),
                         rng.integers(-2048, 2049, n), 3 << 29, shift(k))
    bh, bl, m, k, n = (case["b" + v] for v in "hlmkn")
    # input and result laid out [bh, m, bl, k] and [bh, m, bl, n]: heads between rows and features
    d = capi.FcBatchedDesc(bh, bl, m, k, n, 1, 1, 0, m, bl, k, capi.channel_stride(m), m, bl, n, capi.channel_stride(m))
    many = ctx.fc_batched_prepack(d, normal(bh * bl, n, k), rng.integers(-2048, 2049, (bh * bl, n)),
                                  np.full(bh * bl, 3 << 29, np.int32), np.full(bh * bl, shift(k), np.int32))
    return one, many


def _mix_shapes(case):
    n, c, h, w = case["n"], case["c"], case["h"], case["w"]
    return dict(add=(n, c, h, w), gate=(n, c, h, w), top=(n, c, h, w), leaky=(n, c, h, w), table=(n, c, h, w),
                joined=(n, 2 * c, h, w), scaled=(n, 2 * c, h, w), big=(n, c, 2 * h, 2 * w),
                pooled=(n, c, (h - 1) // 2 + 1, (w - 1) // 2 + 1), mean=(n, c, h // 2, w // 2), all=(n, c, 1, 1))


def _pool(x, y, k, s, p):
    (n, c, ih, iw), (_, _, oh, ow) = x.shape, y.shape
    return capi.PoolDesc(n, c, ih, iw, oh, ow, k[0], k[1], s, s, p, p, p, p, x.cs, y.cs)


_TABLE = np.clip(np.rint(127 * np.tanh(np.arange(256).astype(np.int8) / 40.0)), -128, 127).astype(np.int8)

#: (kind, parameters, result shape) of each data-movement op on (n, c, h, w)
_MOVES = [
    (capi.MOVE_PAD_CONST, [0, 0, 1, 2, 0, 0, 3, 1], lambda n, c, h, w: (n, c, h + 4, w + 3)),
    (capi.MOVE_PAD_EDGE, [0, 0, 2, 2, 0, 0, 2, 2], lambda n, c, h, w: (n, c, h + 4, w + 4)),
    (capi.MOVE_CROP, [0, 0, 1, 3, 1, 1, 1, 1], lambda n, c, h, w: (n, c, h - 3, w - 5)),
    (capi.MOVE_PERMUTE, [0, 2, 3, 1], lambda n, c, h, w: (n, h, w, c)),
    (capi.MOVE_PERMUTE, [0, 1, 3, 2], lambda n, c, h, w: (n, c, w, h)),
    (capi.MOVE_REORG, [2], lambda n, c, h, w: (n, c * 4, h // 2, w // 2)),
    (capi.MOVE_SHUFFLE_CHANNEL, [4], lambda n, c, h, w: (n, c, h, w)),
    (capi.MOVE_DEPTH_TO_SPACE, [2, 0], lambda n, c, h, w: (n, c // 4, 2 * h, 2 * w)),
    (capi.MOVE_REVERSE, [3], lambda n, c, h, w: (n, c, h, w)),
    (capi.MOVE_TILE, [1, 2], lambda n, c, h, w: (n, 2 * c, h, w)),
]


# -- the four functions that are called per case ------------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind in ("net", "dump", "file"):
        rng = np.random.default_rng(seed)
        x = rng.integers(-128, 128, (case["batch"], 3, case["side"], case["side"]), dtype=np.int8)
        if kind == "file":
            folder, outputs = _once(case, lambda: _write_files(case))
            at = os.path.join(folder.name, "in_%d.npz" % seed)
            np.savez(at, input=x.astype(np.float32))
            return dict(case=case, folder=folder.name, input=at, outputs=outputs)
        m, outputs = _once(case, lambda: _load(case))
        return dict(case=case, m=m, outputs=outputs, x=x if case.get("io") == "i8" else x.astype(np.float32))
    fill = torch.Generator(device="cuda")
    fill.manual_seed(seed)
    n = case["n"]
    if kind == "conv":
        handles = _once(case, lambda: _conv_handles(case))
        x = _Map((n, case["ic"], case["h"], case["w"]), fill)
        ys = [_Map((n, c, case["h"], case["w"])) for c in ((case["ic"], case["oc"])[2 - len(handles):])]
        return dict(case=case, handles=handles, x=x, ys=ys)
    if kind == "zoo":
        handles = _once(case, lambda: _zoo_handles(case))
        return dict(case=case, handles=handles, x=_Map((n, case["c"], case["h"], case["w"]), fill),
                    ys=[_Map((n, case["c"]) + s[1]) for s in _zoo_shapes(case)])
    if kind == "fc":
        handles = _once(case, lambda: _fc_handles(case))
        return dict(case=case, handles=handles,
                    xs=[_Map((case["m"], case["k"], 1, 1), fill),
                        _Map((case["bh"], case["bm"], case["bl"], case["bk"]), fill)],
                    ys=[_Map((case["m"], case["n"], 1, 1)), _Map((case["bh"], case["bm"], case["bl"], case["bn"]))])
    shape = (n, case["c"], case["h"], case["w"])
    if kind == "mix":
        return dict(case=case, a=_Map(shape, fill), b=_Map(shape, fill), g=_Map((n, case["c"], 1, 1), fill),
                    ys={k: _Map(s) for k, s in _mix_shapes(case).items()})
    return dict(case=case, x=_Map(shape, fill), ys=[_Map(s(*shape)) for _, _, s in _MOVES])


def run(state):
    kind = state["case"]["kind"]
    if kind == "net":
        m = state["m"]
        if state["case"]["io"] == "f32":
            return m.run(state["x"])
        m.set_tensor_i8("input", state["x"])
        m.invoke()
        return {name: m.get_tensor_i8(name) for name in state["outputs"]}
    if kind == "dump":
        state["m"].run(state["x"])
        return state["m"].get_all_tensor()
    if kind == "file":
        out = os.path.join(state["folder"], "out.npz")
        m = module()
        m.interpret_files(os.path.join(state["folder"], "model.mlir"), state["input"], out)
        m.close()
        f = capi.TensorFile(out)
        got = {name: f.read(name) for name in state["outputs"]}
        f.close()
        return got
    ctx = _context()
    if kind == "conv":
        x = state["x"]
        for h, y in zip(state["handles"], state["ys"]):
            ctx.conv(h, x, y)
            x = y
    elif kind == "zoo":
        for h, y in zip(state["handles"], state["ys"]):
            ctx.conv(h, state["x"], y)
    elif kind == "fc":
        ctx.fc(state["handles"][0], state["xs"][0], state["ys"][0])
        ctx.fc_batched(state["handles"][1], state["xs"][1], state["ys"][1])
    elif kind == "mix":
        a, b, g, ys = state["a"], state["b"], state["g"], state["ys"]
        ctx.eltwise_add([a, b], [50, 60], 7, True, ys["add"])
        ctx.binary(capi.BIN_MUL, a, g, ys["gate"], multiplier=3 << 29, rshift=6)
        ctx.binary(capi.BIN_MAX, a, b, ys["top"], m0=60, m1=70, rshift=6)
        ctx.leaky_relu(a, ys["leaky"], 0, 1, 7, 13)
        ctx.lut(b, ys["table"], _TABLE)
        ctx.concat([a, b], 1, ys["joined"])
        ctx.concat([a, b], 1, ys["scaled"], rshift=[6, 7], mult=[70, 90])
        ctx.upsample(a, ys["big"], 2, 2)
        ctx.pool_max(_pool(a, ys["pooled"], (3, 3), 2, 1), a, ys["pooled"])
        ctx.pool_avg(_pool(a, ys["mean"], (2, 2), 2, 0), a, ys["mean"], 64, 8)
        h, w = a.shape[2:]
        ctx.pool_avg(_pool(a, ys["all"], (h, w), 1, 0), a, ys["all"], min(255, int(4428 / (h * w) ** 0.5)), 13)
        return {k: y.view for k, y in ys.items()}
    else:
        for (kind, params, _), y in zip(_MOVES, state["ys"]):
            ctx.move(kind, state["x"], y, params)
    return [y.view for y in state["ys"]]


def work(case):
    size = lambda s: int(np.prod(s))
    kind = case["kind"]
    if kind in ("net", "dump", "file"):
        net = _build(case)
        word = 1 if case.get("io") == "i8" else 4
        back = net.outputs if kind != "dump" else sum(size(op.shape) for op in net.g.ops)
        return dict(bytes=word * (size(net.shape("input")) + back) + net.weights * (4 if kind == "file" else 1),
                    flops=net.flops)
    n = case["n"]
    if kind == "conv":
        pix, ic, oc, k = n * case["h"] * case["w"], case["ic"], case["oc"], case["k"]
        if case["form"] == "dense":
            return dict(bytes=pix * (ic + oc) + oc * (ic * k * k + 12), flops=2 * pix * oc * ic * k * k)
        return dict(bytes=pix * (2 * ic + oc) + ic * 21 + oc * (ic + 12), flops=2 * pix * ic * (k * k + oc))
    if kind == "zoo":
        c, total = case["c"], dict(bytes=n * case["c"] * case["h"] * case["w"], flops=0)
        for _, (oh, ow), k, _, _, _, g, ins in _zoo_shapes(case):
            total["bytes"] += n * c * oh * ow + c * (c // g * k * k + 12)
            total["flops"] += 2 * n * c * oh * ow * (c // g) * k * k // (1 + ins) ** 2
        return total
    if kind == "fc":
        m, k, n = case["m"], case["k"], case["n"]
        batch, bm, bk, bn = case["bh"] * case["bl"], case["bm"], case["bk"], case["bn"]
        return dict(bytes=m * k + n * k + 4 * n + m * n + batch * (bm * bk + bn * bk + 4 * bn + bm * bn),
                    flops=2 * (m * k * n + batch * bm * bk * bn))
    shape = (n, case["c"], case["h"], case["w"])
    if kind == "mix":
        return dict(bytes=2 * size(shape) + n * case["c"] + sum(size(s) for s in _mix_shapes(case).values()), flops=0)
    return dict(bytes=size(shape) + sum(size(s(*shape)) for _, _, s in _MOVES), flops=0)


def tolerance(case):
    return "exact"        # int8 results of integer arithmetic
