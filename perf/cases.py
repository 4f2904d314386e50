"""The work whose speed is looked after, as cases that can be prepared, run and compared.

A case is one pass of a piece of a convolutional network through the public entry points (`cunn_amd.THNN`), on
tensors that the caller keeps: the forward call of one module or of a short chain of modules, and for training also
the two backward calls of each module, with the flat gradient buffer cleared first as a training step does. All
tensors are fp32 NCHW, the only layout and type the library has. Sizes are those of `bench.py`'s workloads and of the
layer tables of this repository; `draw` spreads over the ranges that those sizes stand for.

Chains that are trained contain a ReLU only in front of the first convolution whose sums have more than a few terms:
behind one, an element within rounding of zero could have its gradient switched on or off by another order of
summation, and two correct results could not be compared element by element.
"""
import math

import torch

from cunn_amd import CudaLongTensor, CudaTensor, THNN

BN_MOMENTUM, BN_EPS = 0.1, 1e-5


def listed():
    return [
        # One image through a depthwise-separable block with evaluation-mode BatchNormalization: what a deployed
        # network does per image and layer. Four short calls; launches and host time are all there is.
        dict(name="block_infer_1x512x14", op="block_infer", n=1, c=512, k=512, h=14, w=14, stride=1),
        # The same kind of block in training at the size of the metric's depthwise layer: depthwise 3x3 stride 2,
        # BatchNormalization + ReLU, 1x1 convolution, BatchNormalization (linear projection), forward and backward.
        dict(name="block_train_64x128x56", op="block_train", n=64, c=128, k=128, h=56, w=56, stride=2),
        # The metric's layer by itself: depthwise 3x3 stride 2, forward, gradInput and weight gradient.
        dict(name="dw_train_64x128x56s2", op="dw_train", n=64, c=128, m=1, h=56, w=56, k=3, stride=2),
        # Depthwise planes of an odd width, where no row starts on a vector boundary.
        dict(name="dw_train_32x128x147", op="dw_train", n=32, c=128, m=1, h=147, w=147, k=3, stride=1),
        # BatchNormalization in training behind a middle layer: a channel fits one compute unit.
        dict(name="bn_train_64x256x28", op="bn_train", n=64, c=256, h=28, w=28, relu=False),
        # BatchNormalization + ReLU (fused entry points) behind a first layer: few channels of large planes.
        dict(name="bnrelu_train_32x64x112", op="bn_train", n=32, c=64, h=112, w=112, relu=True),
        # Pooling behind a first layer: max 3x3 stride 2 with indices and average 2x2, forward and backward.
        dict(name="pool_train_64x64x112", op="pool_train", n=64, c=64, h=112, w=112, mk=3, ms=2, mp=1, ak=2, as_=2, ap=0, ceil=False),
        # The largest: a 3x3 convolution of a residual stage, forward, gradInput and weight gradient.
        dict(name="conv_train_64x256x28", op="conv_train", n=64, cin=256, cout=256, h=28, w=28, k=3, stride=1, pad=1, dil=1),
        # The first layer of a network on photographs: three input planes, 7x7 stride 2.
        dict(name="conv_train_32x3x224s2", op="conv_train", n=32, cin=3, cout=64, h=224, w=224, k=7, stride=2, pad=3, dil=1),
        # A ragged one: channel counts that are no powers of two, odd planes, no padding.
        dict(name="conv_train_32x80x73", op="conv_train", n=32, cin=80, cout=192, h=73, w=73, k=3, stride=1, pad=0, dil=1),
        # The branch of a bottleneck block at a small batch, forward only: 1x1 + ReLU, 3x3 + ReLU, 1x1.
        dict(name="bottleneck_infer_8x256x56", op="bottleneck_infer", n=8, c=256, k=64, h=56, w=56),
        # The doubling transposed convolution of a decoder in training.
        dict(name="fullconv_train_64x256x14", op="fullconv_train", n=64, cin=256, cout=128, h=14, w=14, k=4, stride=2, pad=1),
    ]


# ---------------------------------------------------------------------------------------------- ranges --------

def _log(rng, lo, hi):
    """A whole number from lo to hi, spread evenly over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _channels(rng, lo, hi):
    """Channel counts: multiples of 8 mostly, any number now and then."""
    c = _log(rng, lo, hi)
    return c if rng.random() < 0.3 or c < 16 else (c + 4) // 8 * 8


def _plane(rng, lo, hi):
    h = _log(rng, lo, hi)
    return h, h if rng.random() < 0.75 else _log(rng, max(lo, h * 2 // 3), min(hi, h * 3 // 2))


def _one(rng):
    op = rng.choice(["block_infer", "block_train", "dw_train", "dw_train", "bn_train", "bn_train", "pool_train", "conv_train",
                     "conv_train", "conv_train", "bottleneck_infer", "fullconv_train"])
    if op in ("block_infer", "block_train"):
        h, w = _plane(rng, 7, 112)
        n = _log(rng, 1, 8) if op == "block_infer" else _log(rng, 16, 128)
        return dict(op=op, n=n, c=_channels(rng, 32, 1024), k=_channels(rng, 32, 1024), h=h, w=w, stride=rng.choice([1, 2]))
    if op == "dw_train":
        h, w = _plane(rng, 7, 150)
        return dict(op=op, n=_log(rng, 4, 128), c=_channels(rng, 16, 1024), m=rng.choice([1, 1, 1, 2]), h=h, w=w, k=rng.choice([3, 3, 5]),
                    stride=rng.choice([1, 2]))
    if op == "bn_train":
        h, w = _plane(rng, 7, 150)
        return dict(op=op, n=_log(rng, 4, 128), c=_channels(rng, 16, 1024), h=h, w=w, relu=rng.random() < 0.5)
    if op == "pool_train":
        h, w = _plane(rng, 14, 150)
        mk, ms, mp = rng.choice([(3, 2, 1), (2, 2, 0), (3, 2, 0)])
        ak, as_, ap = rng.choice([(2, 2, 0), (3, 1, 1)])
        return dict(op=op, n=_log(rng, 4, 128), c=_channels(rng, 16, 512), h=h, w=w, mk=mk, ms=ms, mp=mp, ak=ak, as_=as_, ap=ap,
                    ceil=rng.random() < 0.3)
    if op == "conv_train":
        h, w = _plane(rng, 7, 224)
        k, dil = rng.choice([(1, 1), (3, 1), (3, 1), (3, 2), (5, 1), (7, 1)])
        cin = 3 if rng.random() < 0.15 else _channels(rng, 16, 1024)
        stride = 1 if dil > 1 else rng.choice([1, 1, 2])
        pad = dil * (k // 2) if rng.random() < 0.8 else 0
        return dict(op=op, n=_log(rng, 4, 64), cin=cin, cout=_channels(rng, 16, 1024), h=h, w=w, k=k, stride=stride, pad=pad, dil=dil)
    if op == "bottleneck_infer":
        h, w = _plane(rng, 7, 56)
        k = _channels(rng, 32, 256)
        return dict(op=op, n=_log(rng, 1, 16), c=4 * k, k=k, h=h, w=w)
    h, w = _plane(rng, 7, 64)
    k, stride, pad = rng.choice([(4, 2, 1), (2, 2, 0), (3, 1, 1)])
    return dict(op=op, n=_log(rng, 4, 64), cin=_channels(rng, 16, 512), cout=_channels(rng, 16, 512), h=h, w=w, k=k, stride=stride, pad=pad)


def draw(rng):
    while True:
        case = _one(rng)
        if case["op"] == "conv_train" and min(case["h"], case["w"]) + 2 * case["pad"] < case["dil"] * (case["k"] - 1) + 1:
            continue
        w = work(case)
        # within the largest listed case's time, and not all but empty
        if w["bytes"] / 4.0e12 + w["flops"] / 60e12 < 1.2e-3 and w["bytes"] > 1e5:
            return case


# ------------------------------------------------------------------------------------------ shapes, work ------

def _out(h, k, stride, pad, dil=1):
    return (h + 2 * pad - dil * (k - 1) - 1) // stride + 1


def _pooled(h, k, s, p, ceil):
    o = (h + 2 * p - k + (s - 1 if ceil else 0)) // s + 1
    return o - 1 if (ceil or p) and (o - 1) * s >= h + p else o


def _extent(case):
    """(output height, output width) of the case's strided module."""
    op, h, w = case["op"], case["h"], case["w"]
    if op in ("block_infer", "block_train"):
        return _out(h, 3, case["stride"], 1), _out(w, 3, case["stride"], 1)
    if op == "dw_train":
        return _out(h, case["k"], case["stride"], case["k"] // 2), _out(w, case["k"], case["stride"], case["k"] // 2)
    if op == "conv_train":
        return tuple(_out(v, case["k"], case["stride"], case["pad"], case["dil"]) for v in (h, w))
    if op == "fullconv_train":
        return tuple((v - 1) * case["stride"] - 2 * case["pad"] + case["k"] for v in (h, w))
    return h, w


def work(case):
    """Bytes: every input of the pass once, every output once (4-byte elements, 8-byte indices). Flops: the products
    of the convolutions; what normalisation and pooling add is small and not counted."""
    op, n, h, w = case["op"], case["n"], case["h"], case["w"]
    oh, ow = _extent(case)
    if op == "block_infer":
        c, k = case["c"], case["k"]
        return dict(bytes=4 * (n * c * h * w + n * k * oh * ow + 10 * c + c * k + k), flops=2 * n * oh * ow * c * (9 + k))
    if op == "block_train":
        c, k = case["c"], case["k"]
        acts = 2 * n * c * h * w + 2 * n * k * oh * ow          # x, its gradient; the block's output, the arriving gradient
        return dict(bytes=4 * (acts + 2 * n * oh * ow * (c + k) + 2 * c * k), flops=6 * n * oh * ow * c * (9 + k))
    if op == "dw_train":
        c, m, k = case["c"], case["m"], case["k"]
        return dict(bytes=4 * (2 * n * c * h * w + 2 * n * c * m * oh * ow), flops=6 * n * c * m * oh * ow * k * k)
    if op == "bn_train":
        return dict(bytes=4 * 4 * n * case["c"] * h * w, flops=0)
    if op == "pool_train":
        c, ce = case["c"], case["ceil"]
        m = [_pooled(v, case["mk"], case["ms"], case["mp"], ce) for v in (h, w)]
        a = [_pooled(v, case["ak"], case["as_"], case["ap"], ce) for v in (h, w)]
        return dict(bytes=n * c * (4 * 3 * h * w + (4 + 4 + 8) * m[0] * m[1] + 8 * a[0] * a[1]), flops=0)
    if op == "conv_train":
        ci, co, k = case["cin"], case["cout"], case["k"]
        return dict(bytes=4 * (2 * n * ci * h * w + 2 * n * co * oh * ow + 2 * co * ci * k * k), flops=6 * n * oh * ow * co * ci * k * k)
    if op == "bottleneck_infer":
        c, k = case["c"], case["k"]
        return dict(bytes=4 * (2 * n * c * h * w + 2 * c * k + 9 * k * k), flops=2 * n * h * w * (2 * c * k + 9 * k * k))
    ci, co, k = case["cin"], case["cout"], case["k"]
    return dict(bytes=4 * (2 * n * ci * h * w + 2 * n * co * oh * ow + 2 * co * ci * k * k), flops=6 * n * h * w * co * ci * k * k)


def tolerance(case):
    """About four times the largest error of any output against the same pass in 64 bits, over the listed cases and some
    drawn ones. Max-pooling indices are the same, always."""
    op = case["op"]
    if op in ("dw_train", "bn_train"):
        return {"rel": 6e-7, "max": 3e-6}
    if op == "pool_train":
        return {"rel": 4e-7, "max": 2e-6}
    if op == "block_infer":
        return {"rel": 6.4e-7, "max": 6e-6}
    if op == "block_train":      # the gradients of the first normalisation's parameters are sums that nearly cancel
        return {"rel": 8e-6, "max": 3e-5}
    if op == "bottleneck_infer":
        return {"rel": 1.2e-6, "max": 1e-5}
    # convolutions: the error grows with the root of the number of terms of the longest sum, 8.4e-7 at 2304
    rel = max(2e-6, 7.5e-8 * math.sqrt(max(case["cin"], case["cout"]) * case["k"] ** 2))
    return {"rel": rel, "max": 9 * rel}


# --------------------------------------------------------------------------------------------- the passes -----

class _Maker:
    """Tensors of one state: torch tensors on the GPU, and the library's handles on the same memory."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed * 2654435761 % (1 << 62) + 17)
        self.t, self.h = {}, {}

    def put(self, name, tensor, kind=CudaTensor):
        self.t[name], self.h[name] = tensor, kind.from_torch(tensor)

    def normal(self, name, *shape, std=1.0, mean=0.0):
        self.put(name, torch.randn(shape, generator=self.gen, device="cuda").mul_(std).add_(mean))

    def uniform(self, name, lo, hi, *shape):
        self.put(name, torch.rand(shape, generator=self.gen, device="cuda").mul_(hi - lo).add_(lo))

    def result(self, name, *shape):
        self.put(name, torch.zeros(shape, device="cuda"))

    def gradients(self, **shapes):
        """Parameter gradients as views of one flat buffer, which a training step clears in one go."""
        self.put("grads", torch.zeros(sum(math.prod(s) for s in shapes.values()), device="cuda"))
        at = 0
        for name, shape in shapes.items():
            self.put(name, self.t["grads"][at:at + math.prod(shape)].view(shape))
            at += math.prod(shape)

    def buffers(self, *names):
        """Work buffers that the library sizes (a module's finput, fgradInput ...)."""
        for name in names:
            self.h[name] = CudaTensor()

    def norm(self, tag, c, trained=True):
        """Parameters and running statistics of a BatchNormalization over c channels."""
        self.uniform("g" + tag, 0.5, 1.5, c)
        self.normal("b" + tag, c, std=0.1)
        if trained:
            self.put("rm" + tag, torch.zeros(c, device="cuda"))
            self.put("rv" + tag, torch.ones(c, device="cuda"))
        else:
            self.normal("rm" + tag, c, std=0.1)
            self.uniform("rv" + tag, 0.5, 1.5, c)
        self.result("sm" + tag, c)
        self.result("ss" + tag, c)

    def conv(self, tag, cout, cin, k):
        self.normal("w" + tag, cout, cin * k * k, std=math.sqrt(2.0 / (cin * k * k)))
        self.uniform("b" + tag, -0.02, 0.02, cout)


def prepare(case, seed):
    m = _Maker(seed)
    op, n, h, w = case["op"], case["n"], case["h"], case["w"]
    oh, ow = _extent(case)
    if op in ("block_infer", "block_train"):
        c, k = case["c"], case["k"]
        m.normal("x", n, c, h, w)
        m.uniform("wd", -0.8, 0.8, 1, c, 3, 3)
        m.uniform("bd", -1 / 3, 1 / 3, 1, c)
        m.conv("p", k, c, 1)
        if op == "block_train":      # a convolution in front of a trained normalisation has no bias: it would be removed again
            m.h["bd"] = m.h["bp"] = None
        m.norm("1", c, op == "block_train")
        m.norm("2", k, op == "block_train")
        for name, planes in (("y1", c), ("a1", c), ("y2", k), ("a2", k)):
            m.result(name, n, planes, oh, ow)
        m.buffers("cd", "od", "cp", "op")
        if op == "block_train":
            m.normal("ga2", n, k, oh, ow)
            m.result("gy2", n, k, oh, ow)
            m.result("ga1", n, c, oh, ow)
            m.result("gy1", n, c, oh, ow)
            m.result("gx", n, c, h, w)
            m.gradients(gwd=(1, c, 3, 3), gg1=(c,), gb1=(c,), gwp=(k, c), gg2=(k,), gb2=(k,))
            m.buffers("gcp")
    elif op == "dw_train":
        c, mm, k = case["c"], case["m"], case["k"]
        m.normal("x", n, c, h, w)
        m.normal("gy", n, c * mm, oh, ow)
        m.uniform("wt", -math.sqrt(6) / k, math.sqrt(6) / k, mm, c, k, k)
        m.uniform("b", -1 / k, 1 / k, mm, c)
        m.result("y", n, c * mm, oh, ow)
        m.result("gx", n, c, h, w)
        m.gradients(gw=(mm, c, k, k), gb=(mm, c))
        m.buffers("cols", "ones")
    elif op == "bn_train":
        c = case["c"]
        m.normal("x", n, c, h, w, std=2.0, mean=0.5)
        m.normal("gy", n, c, h, w)
        m.norm("", c)
        m.result("y", n, c, h, w)
        m.result("gx", n, c, h, w)
        m.gradients(gg=(c,), gb=(c,))
    elif op == "pool_train":
        c, ce = case["c"], case["ceil"]
        mo = [_pooled(v, case["mk"], case["ms"], case["mp"], ce) for v in (h, w)]
        ao = [_pooled(v, case["ak"], case["as_"], case["ap"], ce) for v in (h, w)]
        # activations behind a ReLU-like layer tie often: values in steps of 1/64
        m.put("x", torch.rand((n, c, h, w), generator=m.gen, device="cuda").mul_(128).round_().div_(64).sub_(1))
        m.normal("gym", n, c, *mo)
        m.normal("gya", n, c, *ao)
        m.result("ym", n, c, *mo)
        m.put("idx", torch.zeros((n, c, *mo), dtype=torch.int64, device="cuda"), CudaLongTensor)
        m.result("ya", n, c, *ao)
        m.result("gxm", n, c, h, w)
        m.result("gxa", n, c, h, w)
    elif op in ("conv_train", "fullconv_train"):
        ci, co, k = case["cin"], case["cout"], case["k"]
        m.normal("x", n, ci, h, w)
        m.normal("gy", n, co, oh, ow)
        shape = (ci, co, k, k) if op == "fullconv_train" else (co, ci * k * k) if case["dil"] == 1 else (co, ci, k, k)
        m.normal("wt", *shape, std=math.sqrt(2.0 / (ci * k * k)))
        m.uniform("b", -0.02, 0.02, co)
        m.result("y", n, co, oh, ow)
        m.result("gx", n, ci, h, w)
        m.gradients(gw=shape, gb=(co,))
        m.buffers("cols", "gcols", "ones")
    else:
        c, k = case["c"], case["k"]
        m.normal("x", n, c, h, w)
        m.conv("1", k, c, 1)
        m.conv("2", k, k, 3)
        m.conv("3", c, k, 1)
        m.result("a1", n, k, h, w)
        m.result("a2", n, k, h, w)
        m.result("y", n, c, h, w)
        m.buffers("c1", "c2", "c3", "ones")
    return dict(case=case, t=m.t, h=m.h)


def run(state):
    case, t, h = state["case"], state["t"], state["h"]
    op = case["op"]
    if op == "block_infer":
        s = case["stride"]
        THNN.SpatialDepthWiseConvolution_updateOutput(h["x"], h["y1"], h["wd"], h["bd"], h["cd"], h["od"], 3, 3, s, s, 1, 1)
        THNN.BatchNormalizationReLU_updateOutput(h["y1"], h["a1"], h["g1"], h["b1"], h["rm1"], h["rv1"], h["sm1"], h["ss1"],
                                                 False, BN_MOMENTUM, BN_EPS)
        THNN.SpatialConvolutionMM_updateOutput(h["a1"], h["y2"], h["wp"], h["bp"], h["cp"], h["op"], 1, 1, 1, 1, 0, 0)
        THNN.BatchNormalizationReLU_updateOutput(h["y2"], h["a2"], h["g2"], h["b2"], h["rm2"], h["rv2"], h["sm2"], h["ss2"],
                                                 False, BN_MOMENTUM, BN_EPS)
        return dict(y1=t["y1"], a1=t["a1"], y2=t["y2"], a2=t["a2"])
    if op == "block_train":
        s = case["stride"]
        h["grads"].fill(0.0)
        THNN.SpatialDepthWiseConvolution_updateOutput(h["x"], h["y1"], h["wd"], h["bd"], h["cd"], h["od"], 3, 3, s, s, 1, 1)
        THNN.BatchNormalizationReLU_updateOutput(h["y1"], h["a1"], h["g1"], h["b1"], h["rm1"], h["rv1"], h["sm1"], h["ss1"],
                                                 True, BN_MOMENTUM, BN_EPS)
        THNN.SpatialConvolutionMM_updateOutput(h["a1"], h["y2"], h["wp"], h["bp"], h["cp"], h["op"], 1, 1, 1, 1, 0, 0)
        THNN.BatchNormalization_updateOutput(h["y2"], h["a2"], h["g2"], h["b2"], h["rm2"], h["rv2"], h["sm2"], h["ss2"],
                                             True, BN_MOMENTUM, BN_EPS)
        THNN.BatchNormalization_backward(h["y2"], h["ga2"], h["gy2"], h["gg2"], h["gb2"], h["g2"], h["rm2"], h["rv2"],
                                         h["sm2"], h["ss2"], True, 1.0, BN_EPS)
        THNN.SpatialConvolutionMM_updateGradInput(h["a1"], h["gy2"], h["ga1"], h["wp"], h["gcp"], h["op"], 1, 1, 1, 1, 0, 0)
        THNN.SpatialConvolutionMM_accGradParameters(h["a1"], h["gy2"], h["gwp"], None, h["cp"], h["op"], 1, 1, 1, 1, 0, 0, 1.0)
        THNN.BatchNormalizationReLU_backward(h["y1"], h["ga1"], h["gy1"], h["gg1"], h["gb1"], h["g1"], h["b1"], h["rm1"], h["rv1"],
                                             h["sm1"], h["ss1"], True, 1.0, BN_EPS)
        THNN.SpatialDepthWiseConvolution_updateGradInput(h["x"], h["gy1"], h["gx"], h["wd"], h["cd"], h["od"], 3, 3, s, s, 1, 1)
        THNN.SpatialDepthWiseConvolution_accGradParameters(h["x"], h["gy1"], h["gwd"], None, h["cd"], h["od"], 3, 3, s, s, 1, 1, 1.0)
        return {k: t[k] for k in ("y1", "a1", "y2", "a2", "gy2", "ga1", "gy1", "gx", "gwd", "gwp", "gg1", "gb1", "gg2", "gb2",
                                  "rm1", "rv1", "rm2", "rv2", "sm1", "ss1", "sm2", "ss2")}
    if op == "dw_train":
        g = (case["k"], case["k"], case["stride"], case["stride"], case["k"] // 2, case["k"] // 2)
        h["grads"].fill(0.0)
        THNN.SpatialDepthWiseConvolution_updateOutput(h["x"], h["y"], h["wt"], h["b"], h["cols"], h["ones"], *g)
        THNN.SpatialDepthWiseConvolution_updateGradInput(h["x"], h["gy"], h["gx"], h["wt"], h["cols"], h["ones"], *g)
        THNN.SpatialDepthWiseConvolution_accGradParameters(h["x"], h["gy"], h["gw"], h["gb"], h["cols"], h["ones"], *g, 1.0)
        return {k: t[k] for k in ("y", "gx", "gw", "gb")}
    if op == "bn_train":
        h["grads"].fill(0.0)
        if case["relu"]:
            THNN.BatchNormalizationReLU_updateOutput(h["x"], h["y"], h["g"], h["b"], h["rm"], h["rv"], h["sm"], h["ss"], True,
                                                     BN_MOMENTUM, BN_EPS)
            THNN.BatchNormalizationReLU_backward(h["x"], h["gy"], h["gx"], h["gg"], h["gb"], h["g"], h["b"], h["rm"], h["rv"],
                                                 h["sm"], h["ss"], True, 1.0, BN_EPS)
        else:
            THNN.BatchNormalization_updateOutput(h["x"], h["y"], h["g"], h["b"], h["rm"], h["rv"], h["sm"], h["ss"], True,
                                                 BN_MOMENTUM, BN_EPS)
            THNN.BatchNormalization_backward(h["x"], h["gy"], h["gx"], h["gg"], h["gb"], h["g"], h["rm"], h["rv"], h["sm"], h["ss"],
                                             True, 1.0, BN_EPS)
        return {k: t[k] for k in ("y", "gx", "gg", "gb", "rm", "rv", "sm", "ss")}
    if op == "pool_train":
        mx = (case["mk"], case["mk"], case["ms"], case["ms"], case["mp"], case["mp"], case["ceil"])
        av = (case["ak"], case["ak"], case["as_"], case["as_"], case["ap"], case["ap"], case["ceil"], True)
        THNN.SpatialMaxPooling_updateOutput(h["x"], h["ym"], h["idx"], *mx)
        THNN.SpatialMaxPooling_updateGradInput(h["x"], h["gym"], h["gxm"], h["idx"], *mx)
        THNN.SpatialAveragePooling_updateOutput(h["x"], h["ya"], *av)
        THNN.SpatialAveragePooling_updateGradInput(h["x"], h["gya"], h["gxa"], *av)
        return {k: t[k] for k in ("ym", "idx", "gxm", "ya", "gxa")}
    if op == "conv_train":
        g = (case["k"], case["k"], case["stride"], case["stride"], case["pad"], case["pad"])
        h["grads"].fill(0.0)
        if case["dil"] == 1:
            THNN.SpatialConvolutionMM_updateOutput(h["x"], h["y"], h["wt"], h["b"], h["cols"], h["ones"], *g)
            THNN.SpatialConvolutionMM_updateGradInput(h["x"], h["gy"], h["gx"], h["wt"], h["gcols"], h["ones"], *g)
            THNN.SpatialConvolutionMM_accGradParameters(h["x"], h["gy"], h["gw"], h["gb"], h["cols"], h["ones"], *g, 1.0)
        else:
            g += (case["dil"], case["dil"])
            THNN.SpatialDilatedConvolution_updateOutput(h["x"], h["y"], h["wt"], h["b"], h["cols"], h["ones"], *g)
            THNN.SpatialDilatedConvolution_updateGradInput(h["x"], h["gy"], h["gx"], h["wt"], h["gcols"], *g)
            THNN.SpatialDilatedConvolution_accGradParameters(h["x"], h["gy"], h["gw"], h["gb"], h["cols"], h["ones"], *g, 1.0)
        return {k: t[k] for k in ("y", "gx", "gw", "gb")}
    if op == "fullconv_train":
        g = (case["k"], case["k"], case["stride"], case["stride"], case["pad"], case["pad"], 0, 0)
        h["grads"].fill(0.0)
        THNN.SpatialFullConvolution_updateOutput(h["x"], h["y"], h["wt"], h["b"], h["cols"], h["ones"], *g)
        THNN.SpatialFullConvolution_updateGradInput(h["x"], h["gy"], h["gx"], h["wt"], h["gcols"], *g)
        THNN.SpatialFullConvolution_accGradParameters(h["x"], h["gy"], h["gw"], h["gb"], h["cols"], h["ones"], *g, 1.0)
        return {k: t[k] for k in ("y", "gx", "gw", "gb")}
    THNN.SpatialConvolutionMMReLU_updateOutput(h["x"], h["a1"], h["w1"], h["b1"], h["c1"], h["ones"], 1, 1, 1, 1, 0, 0)
    THNN.SpatialConvolutionMMReLU_updateOutput(h["a1"], h["a2"], h["w2"], h["b2"], h["c2"], h["ones"], 3, 3, 1, 1, 1, 1)
    THNN.SpatialConvolutionMM_updateOutput(h["a2"], h["y"], h["w3"], h["b3"], h["c3"], h["ones"], 1, 1, 1, 1, 0, 0)
    return {k: t[k] for k in ("a1", "a2", "y")}
