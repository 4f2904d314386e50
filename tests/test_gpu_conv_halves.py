"""Convolution passes on half-precision parts (three fp16 products per fp32 product, half_parts.h) wherever
they can be forced: tile shapes and their edges, ragged channels, strides (phases), dilation, K split over workgroups, a
smaller last group of positions; operands of all sizes, infinities and NaNs, images, channels and corners of very
different size, on fp16 parts, on bf16 parts where those do not hold an image or a weight row, and both in one call. Bounds: those of test_gpu_conv_split.py (a chain of K fp32 additions); element by element, K fp32
additions of what the terms of the element add up to in magnitude."""
import numpy as np
import pytest

import cunn_amd
from test_gpu_conv_split import SIZES, _check_error, _check_non_finite, _check_sizes, _passes, _tensors

from oracle import oracle as O

pytestmark = pytest.mark.gpu

# N, Cin, Cout, H, W, k, stride, pad
CASES = [
    (2, 64, 128, 12, 12, 3, 1, 1),    # 128 x 128 tiles, 64 x 128 in gradInput
    (3, 36, 70, 9, 11, 3, 2, 1),      # ragged groups of channels, 96-row tiles, four phases
    (2, 20, 40, 14, 10, 5, 1, 0),     # no border in the forward pass
    (4, 512, 136, 7, 8, 1, 1, 0),     # 1x1
    (2, 17, 30, 16, 15, 3, 1, 1),     # 32-row tiles, one channel in the last group
    (1, 24, 300, 30, 28, 7, 2, 3),
    (9, 256, 96, 13, 15, 3, 1, 1),    # K split over workgroups
    (2, 40, 64, 9, 10, 2, 2, 0),
    (1, 16, 33, 5, 4, 4, 1, 2),       # fewer positions than a tile
    # 16-byte and transposed gathers, k-tiles inside an image or not (the weight gradient's large tiles: LARGE)
    (2, 64, 120, 16, 16, 3, 2, 1),
    (3, 64, 120, 9, 12, 3, 1, 1),
    (2, 64, 128, 25, 25, 3, 2, 1),
    (2, 28, 60, 16, 16, 3, 1, 1),
    (3, 28, 60, 13, 14, 3, 1, 1),
]


@pytest.fixture(autouse=True)
def _forced():
    cunn_amd.set_switch("THCUNN_CONV_HALVES", "1")
    yield
    cunn_amd.set_switch("THCUNN_CONV_HALVES", None)


@pytest.mark.parametrize("case", CASES)
def test_operands_of_all_kinds(case):
    for kind in ("normal", "one-signed", "scaled", "tiny", "smallest"):
        print("case", case, kind, flush=True)
        _check_error(case, kind)
    for sizes in SIZES:
        print("case", case, sizes, flush=True)
        _check_sizes(case, *sizes)
    _check_non_finite(case)


@pytest.mark.parametrize("case", CASES)
def test_large_and_non_finite_weights(case):
    """Blocks that are computed again with weights whose bf16 parts overflow (2^104 and more), infinities, NaNs and subnormal ones: as the
    oracle gives them (gradInput, where zeros beyond gradOutput meet the weights, without the infinities and NaNs). Bound for an
    element: two chains of K fp32 additions, ours and the oracle's, each rounded by 2^-24 of what it adds up to at most, and, where sums are
    subnormal, by 2^-150 (products of the subnormal row are smaller than that)."""
    N, Ci, Co, H, W, k, st, pad = case
    x, w, gy = _tensors(case, "normal", 7)
    x, gy = x * np.float32(1e-4), gy * np.float32(1e-4)
    w[3, 1], w[4, 2], w[5], w[Co - 1, Ci * k * k - 1] = 3e38, -2.0 ** 104, w[5] * 1e-42, 2.0 ** 110
    g = (k, k, st, st, pad, pad)
    for special in (False, True):
        if special:
            w[0, 3], w[1, 0], w[2, Ci * k * k - 2], x[0, 1, 2, 3] = np.inf, np.nan, -np.inf, np.inf
        got = _passes(case, x, w, gy, gy)
        with np.errstate(all="ignore"):
            refs = (O.convmm_updateOutput(x, w, None, *g), O.convmm_updateGradInput(x.shape, gy, w, *g))
            sums = (O.convmm_updateOutput(np.abs(x), np.abs(w), None, *g), O.convmm_updateGradInput(x.shape, np.abs(gy), np.abs(w), *g))
        for name, here, ref, total, K in list(zip(("output", "gradInput"), got, refs, sums, (Ci * k * k, Co * k * k)))[:1 if special else 2]:
            print(case, name, special, flush=True)
            for f in (np.isnan, np.isposinf, np.isneginf):
                assert np.array_equal(f(here), f(ref)), f.__name__
            fine = np.isfinite(ref)
            bound = 2 * K * (2.0 ** -24 * total[fine].astype(np.float64) + 2.0 ** -150)
            worst = (np.abs(here[fine].astype(np.float64) - ref[fine]) / bound).max()
            print("worst element at %.3g of its bound" % worst, flush=True)
            assert worst <= 1


@pytest.mark.parametrize("case", CASES)
def test_forced_passes_run_these_kernels(case):
    """Other last bits than with the switch off, in the output and (1x1 windows aside) in gradInput; the weight gradient: LARGE."""
    x, w, gy = _tensors(case, "normal")
    here = _passes(case, x, w, gy, gy)
    cunn_amd.set_switch("THCUNN_CONV_HALVES", "0")
    other = _passes(case, x, w, gy, gy)
    assert not np.array_equal(here[0], other[0])
    assert case[5] == 1 or not np.array_equal(here[1], other[1])


def _terms(x, w, dil):
    """sum and sum of magnitudes of the terms of every output of a stride-1 convolution without padding"""
    k = w.shape[2]
    span = dil * (k - 1) + 1
    col = np.lib.stride_tricks.sliding_window_view(x.astype(np.float64), (span, span), axis=(2, 3))[..., ::dil, ::dil]
    w = w.astype(np.float64)
    return np.einsum("ncijkl,ockl->noij", col, w), np.einsum("ncijkl,ockl->noij", np.abs(col), np.abs(w))


@pytest.mark.parametrize("dil", [1, 2])
@pytest.mark.parametrize("where", ["image", "channel", "corner", "few", "one"])
def test_very_different_sizes(where, dil):
    print("case", where, dil, flush=True)
    rng = np.random.default_rng(3)
    N, Ci, Co, H, W, k = 3, 24, 40, 15, 18, 3
    x = np.maximum(rng.standard_normal((N, Ci, H, W)), 0)
    w = rng.standard_normal((Co, Ci, k, k))
    if where == "image":
        x[1] *= 1e-20
    elif where == "channel":                       # small elements with large weights
        x[:, 5] *= 1e-12
        w[:, 5] *= 1e12
    elif where == "corner":
        x[:, :, :7, :8] *= 1e-15
    elif where == "few":                           # neighbours in a group of channels are zero
        x[0, :, 2:9, 2:9] = 0
        x[0, 3, 5, 5] = 1e-14
    else:                                          # everything else is small beside one element
        x[2, 1, 4, 4] = 1e15
    x, w, b = x.astype(np.float32), w.astype(np.float32), rng.standard_normal(Co).astype(np.float32) * (where in ("few", "one"))
    b = b.astype(np.float32)
    CT, y = cunn_amd.CudaTensor, cunn_amd.CudaTensor()
    cunn_amd.THNN.SpatialDilatedConvolution_updateOutput(CT.from_numpy(x), y, CT.from_numpy(w), CT.from_numpy(b), CT(), CT(),
                                                         k, k, 1, 1, 0, 0, dil, dil)
    ref, terms = _terms(x, w, dil)
    ref, terms = ref + b[None, :, None, None], terms + np.abs(b)[None, :, None, None]
    assert (np.abs(y.numpy() - ref) <= Ci * k * k * 2.0 ** -24 * terms + 2.0 ** -149).all()


@pytest.mark.parametrize("Ci, k", [(16, 224), (16, 215), (9, 200)])
def test_windows_beyond_the_index_arithmetic(Ci, k):
    """(groups of channels) x taps x taps at and beyond 2^32, where the division that takes (group, tap) apart is no longer exact:
    every weight of such a window counts. One channel of large weights and elements, so a wrong one would show."""
    print("case", Ci, k, flush=True)
    rng = np.random.default_rng(k)
    Co = 2
    x = rng.standard_normal((1, Ci, k + 1, k + 1)).astype(np.float32)
    w = np.zeros((Co, Ci, k, k), np.float32)
    w[:, :, -1, -3:] = rng.standard_normal((Co, Ci, 3))   # the last taps of every channel
    w[:, :, 0, :3] = rng.standard_normal((Co, Ci, 3))
    ref = np.zeros((1, Co, 2, 2))
    for i in range(2):
        for j in range(2):
            ref[0, :, i, j] = (w.astype(np.float64) * x[0, :, i:i + k, j:j + k]).sum((1, 2, 3))
    CT, y = cunn_amd.CudaTensor, cunn_amd.CudaTensor()
    cunn_amd.THNN.SpatialConvolutionMM_updateOutput(CT.from_numpy(x), y, CT.from_numpy(w.reshape(Co, -1)), None, CT(), CT(),
                                                    k, k, 1, 1, 0, 0)
    # at most 96 terms of size 1 that are not zero
    assert np.abs(y.numpy() - ref).max() <= 96 * 2.0 ** -24 * 96


def _grad_input(gy, w, dil, stride, H, W):
    """gradInput of a convolution without padding in 64 bits, and the sum of the magnitudes of its terms"""
    import torch
    f = lambda a, b: torch.nn.functional.conv_transpose2d(torch.from_numpy(a).double(), torch.from_numpy(b).double(), stride=stride,
                                                          dilation=dil).numpy()
    out = []
    for a, b in ((gy, w), (np.abs(gy), np.abs(w))):
        full, padded = f(a, b), np.zeros(gy.shape[:1] + w.shape[1:2] + (H, W))
        padded[:, :, :full.shape[2], :full.shape[3]] = full
        out.append(padded)
    return out


def _forward_and_grad_input(x, gy, w, dil, stride):
    """Both passes without padding against 64 bits, element by element: K fp32 additions of the element's own terms."""
    CT, y, gx = cunn_amd.CudaTensor, cunn_amd.CudaTensor(), cunn_amd.CudaTensor()
    Co, Ci, k, _ = w.shape
    a = (k, k, stride, stride, 0, 0, dil, dil)
    cunn_amd.THNN.SpatialDilatedConvolution_updateOutput(CT.from_numpy(x), y, CT.from_numpy(w), None, CT(), CT(), *a)
    ref, terms = _terms(x, w, dil)
    ref, terms = ref[:, :, ::stride, ::stride], terms[:, :, ::stride, ::stride]
    worst = np.abs(y.numpy() - ref) / (Ci * k * k * 2.0 ** -24 * terms + 2.0 ** -149)
    print("forward: worst element at %.3g of its bound" % worst.max(), flush=True)
    assert worst.max() <= 1
    cunn_amd.THNN.SpatialDilatedConvolution_updateGradInput(CT.from_numpy(x), CT.from_numpy(gy), gx, CT.from_numpy(w), CT(), *a)
    ref, terms = _grad_input(gy, w, dil, stride, x.shape[2], x.shape[3])
    worst = np.abs(gx.numpy() - ref) / (Co * k * k * 2.0 ** -24 * terms + 2.0 ** -149)
    print("gradInput: worst element at %.3g of its bound" % worst.max(), flush=True)
    assert worst.max() <= 1


# 2^power apart: within reach of two parts, at the edge of it, at half the bits, lost altogether
POWERS = [20, 27, 28, 29, 40, 44, 48, 52, 60]


@pytest.mark.parametrize("dil, stride", [(1, 1), (2, 1), (1, 2)])
@pytest.mark.parametrize("power", POWERS)
def test_large_weights_that_meet_zeros(power, dil, stride):
    """The rest of a weight row decides the output where the plane that its large weights meet is zero."""
    print("case", power, dil, stride, flush=True)
    rng = np.random.default_rng(power)
    N, Ci, Co, H, W, k = 3, 40, 48, 15, 18, 3
    f = lambda *s: rng.standard_normal(s).astype(np.float32)
    span = dil * (k - 1) + 1
    x, w, gy = f(N, Ci, H, W), f(Co, Ci, k, k), f(N, Co, (H - span) // stride + 1, (W - span) // stride + 1)
    wx = w.copy()
    x[:, 5] = 0
    wx[:, 5] *= np.float32(2.0 ** power)
    gy[:, 7] = 0
    wx[7] *= np.float32(2.0 ** power)
    wx[7, 5] = w[7, 5]
    _forward_and_grad_input(x, gy, wx, dil, stride)


@pytest.mark.parametrize("dil, stride", [(1, 1), (2, 1), (1, 2)])
@pytest.mark.parametrize("power", POWERS)
def test_small_elements_that_weights_pick_out(power, dil, stride):
    """Rows of one weight each: an output is one element of the image, also one that is small beside all its neighbours."""
    print("case", power, dil, stride, flush=True)
    rng = np.random.default_rng(power)
    N, Ci, Co, H, W, k = 3, 40, 40, 15, 18, 3
    f = lambda *s: rng.standard_normal(s).astype(np.float32)
    span = dil * (k - 1) + 1
    x, gy = f(N, Ci, H, W), f(N, Co, (H - span) // stride + 1, (W - span) // stride + 1)
    for t in (x, gy):
        few = rng.random(t.shape) < 0.02
        few[1] = False                              # an image that is ordinary throughout
        t[few] *= np.float32(2.0 ** -power)
    w = np.zeros((Co, Ci, k, k), np.float32)
    for o in range(Co):
        w[o, o, o % 3, o // 3 % 3] = rng.standard_normal()
    _forward_and_grad_input(x, gy, w, dil, stride)


@pytest.mark.parametrize("case", [(40, 24, 40, 3, 3, 3), (9, 24, 136, 5, 4, 3), (300, 20, 30, 1, 2, 1), (2, 16, 70, 40, 39, 2)])
def test_images_of_both_kinds_in_a_tile(case):
    """Every third image holds elements far below its largest: tiles of many images, tiles inside one, 1x1 planes."""
    print("case", case, flush=True)
    N, Ci, Co, H, W, k = case
    rng = np.random.default_rng(N)
    f = lambda *s: rng.standard_normal(s).astype(np.float32)
    x, w, gy = f(N, Ci, H, W), f(Co, Ci, k, k) * np.float32(0.1), f(N, Co, H - k + 1, W - k + 1) if k <= min(H, W) else None
    for t in (x, gy):
        t[::3, ::5] *= np.float32(2.0 ** -50)
    w[:3] *= (rng.random((3, Ci, k, k)) < 0.1).astype(np.float32)
    _forward_and_grad_input(x, gy, w, 1, 1)


def test_more_images_than_a_grid_dimension_holds():
    """70000 images of one position each: 256 of them in a tile, of both kinds; all three passes."""
    rng = np.random.default_rng(9)
    N, Ci, Co, k = 70000, 16, 8, 2
    x, w, gy = (rng.standard_normal(s).astype(np.float32) for s in ((N, Ci, k, k), (Co, Ci, k, k), (N, Co, 1, 1)))
    x[::1000, :5] *= np.float32(1e-20)
    x[1::1000, 5:] = 0
    gy[2::1000, 1:] *= np.float32(1e-20)
    CT, y, gx = cunn_amd.CudaTensor, cunn_amd.CudaTensor(), cunn_amd.CudaTensor()
    THNN, tw, a = cunn_amd.THNN, CT.from_numpy(w.reshape(Co, -1)), (k, k, 1, 1, 0, 0)
    THNN.SpatialConvolutionMM_updateOutput(CT.from_numpy(x), y, tw, None, CT(), CT(), *a)
    THNN.SpatialConvolutionMM_updateGradInput(CT.from_numpy(x), CT.from_numpy(gy), gx, tw, CT(), CT(), *a)
    xd, wd, gd = (v.astype(np.float64) for v in (x.reshape(N, -1), w.reshape(Co, -1), gy.reshape(N, Co)))
    for got, p, q in ((y.numpy().reshape(N, Co), xd, wd.T), (gx.numpy().reshape(N, -1), gd, wd),
                      (_weight_gradient(x, gy, k, 1, 0), gd.T, xd)):
        assert (np.abs(got - p @ q) <= p.shape[1] * 2.0 ** -24 * (np.abs(p) @ np.abs(q)) + 2.0 ** -149).all()


@pytest.mark.parametrize("relu", [False, True])
def test_bias_relu_and_buffers(relu):
    """Bias and clamp in the epilogue; a buffer tensor that is too small and cannot grow leaves the call to the other kernels."""
    import torch
    N, Ci, Co, H, W, k = 2, 32, 72, 11, 13, 3
    rng = np.random.default_rng(4)
    x, w, b = (rng.standard_normal(s).astype(np.float32) for s in ((N, Ci, H, W), (Co, Ci * k * k), (Co,)))
    THNN, CT = cunn_amd.THNN, cunn_amd.CudaTensor
    f = THNN.SpatialConvolutionMMReLU_updateOutput if relu else THNN.SpatialConvolutionMM_updateOutput
    ref = torch.nn.functional.conv2d(*(torch.from_numpy(v).double() for v in (x, w.reshape(Co, Ci, k, k), b)), padding=1).numpy()
    if relu:
        ref = np.maximum(ref, 0)
    for buffer in (CT(), None):
        y = CT()
        f(CT.from_numpy(x), y, CT.from_numpy(w), CT.from_numpy(b), buffer, CT(), k, k, 1, 1, 1, 1)
        assert np.linalg.norm(y.numpy() - ref) <= (2.0 ** -25 * np.sqrt(Ci * k * k) + 2.0 ** -24) * np.linalg.norm(ref)


@pytest.mark.parametrize("case", [(2, 40, 24, 7, 9, 4, 2, 1), (3, 16, 72, 6, 6, 3, 1, 1), (1, 33, 20, 9, 5, 2, 2, 0)])
def test_transposed(case):
    import torch
    print("case", case, flush=True)
    N, Ci, Co, H, W, k, st, pad = case
    rng = np.random.default_rng(5)
    x, w, b = (rng.standard_normal(s).astype(np.float32) for s in ((N, Ci, H, W), (Ci, Co, k, k), (Co,)))
    d = [torch.from_numpy(v).double() for v in (x, w, b)]
    ref = torch.nn.functional.conv_transpose2d(*d, stride=st, padding=pad).numpy()
    CT, y = cunn_amd.CudaTensor, cunn_amd.CudaTensor()
    cunn_amd.THNN.SpatialFullConvolution_updateOutput(CT.from_numpy(x), y, CT.from_numpy(w), CT.from_numpy(b), CT(), CT(),
                                                      k, k, st, st, pad, pad, 0, 0)
    assert np.linalg.norm(y.numpy() - ref) <= (2.0 ** -25 * np.sqrt(Ci * k * k) + 2.0 ** -24) * np.linalg.norm(ref)


@pytest.mark.parametrize("which", ["x image", "gy image", "row", "column", "both"])
@pytest.mark.parametrize("case", [(4, 64, 128, 16, 16, 3, 1, 1), (4, 28, 60, 13, 14, 3, 1, 1)])
def test_weight_gradient_of_very_different_sizes(case, which):
    """Images, gradOutput rows and columns that are small throughout, alone or against large partners."""
    import torch
    print("case", case, which, flush=True)
    N, Ci, Co, H, W, k, st, pad = case
    rng = np.random.default_rng(7)
    x, gy = rng.standard_normal((N, Ci, H, W)), rng.standard_normal((N, Co, H, W))
    if which == "x image":
        x[1] *= 1e-14
        gy[1] *= 1e14
    elif which == "gy image":
        gy[2] *= 1e-20
    elif which == "row":
        gy[:, 3] *= 1e-25
    elif which == "column":
        x[:, 5] *= 1e-25
    else:
        gy[:, 3] *= 1e-16
        x[:, 5] *= 1e16
    x, gy = x.astype(np.float32), gy.astype(np.float32)
    THNN, CT = cunn_amd.THNN, cunn_amd.CudaTensor
    gw = CT.from_numpy(np.zeros((Co, Ci * k * k), np.float32))
    THNN.SpatialConvolutionMM_accGradParameters(CT.from_numpy(x), CT.from_numpy(gy), gw, None, CT(), CT(), k, k, st, st, pad, pad, 1.0)
    f = lambda a, b: torch.nn.grad.conv2d_weight(torch.from_numpy(a).double(), (Co, Ci, k, k), torch.from_numpy(b).double(),
                                                 stride=st, padding=pad).numpy().reshape(Co, -1)
    terms = f(np.abs(x), np.abs(gy))
    assert (np.abs(gw.numpy() - f(x, gy)) <= N * H * W * 2.0 ** -24 * terms + 2.0 ** -149).all()


# Layers whose weight gradient runs on large tiles (the short reductions above take small ones): every instance of the kernel - 128 x 128
# and 64 x 256 tiles, k-tiles inside an image or not, 16-byte or transposed gathers.
LARGE = [
    (16, 64, 128, 24, 24, 3, 1, 1),
    (18, 64, 128, 48, 48, 3, 2, 1),
    (20, 64, 128, 23, 24, 3, 1, 1),
    (20, 64, 128, 23, 23, 3, 1, 1),
    (32, 28, 60, 24, 24, 3, 1, 1),
    (36, 28, 60, 47, 47, 3, 2, 1),
    (33, 28, 60, 23, 24, 3, 1, 1),
    (36, 28, 60, 23, 23, 3, 1, 1),
]


def _weight_gradient(x, gy, k, st, pad):
    THNN, CT = cunn_amd.THNN, cunn_amd.CudaTensor
    gw = CT.from_numpy(np.zeros((gy.shape[1], x.shape[1] * k * k), np.float32))
    THNN.SpatialConvolutionMM_accGradParameters(CT.from_numpy(x), CT.from_numpy(gy), gw, None, CT(), CT(), k, k, st, st, pad, pad, 1.0)
    return gw.numpy()


def _weight_gradient_exact(x, gy, k, st, pad):
    """in 64 bits; and the sum of the magnitudes of the terms"""
    import torch
    out = []
    for a, b in ((x, gy), (np.abs(x), np.abs(gy))):
        col = torch.nn.functional.unfold(torch.from_numpy(a).cuda().double(), k, padding=pad, stride=st)   # N, K, L
        rows = torch.from_numpy(b).cuda().double().flatten(2).transpose(0, 1).flatten(1)                   # Co, N * L
        out.append((rows @ col.transpose(1, 2).flatten(0, 1)).cpu().numpy())
    return out


@pytest.mark.parametrize("case", LARGE)
def test_weight_gradient_on_large_tiles(case):
    """Within the bound of sums of the positions of a split, and not what the other kernels give: these ran."""
    print("case", case, flush=True)
    N, Ci, Co, H, W, k, st, pad = case
    oH, oW = (H + 2 * pad - k) // st + 1, (W + 2 * pad - k) // st + 1
    rng = np.random.default_rng(8)
    x, gy = rng.standard_normal((N, Ci, H, W)).astype(np.float32), rng.standard_normal((N, Co, oH, oW)).astype(np.float32)
    got = _weight_gradient(x, gy, k, st, pad)
    ref, _ = _weight_gradient_exact(x, gy, k, st, pad)
    cunn_amd.set_switch("THCUNN_CONV_HALVES", "0")
    other = _weight_gradient(x, gy, k, st, pad)
    assert not np.array_equal(got, other)
    error, before = (np.linalg.norm(v - ref) / np.linalg.norm(ref) for v in (got, other))
    print("error %.3g, six products %.3g" % (error, before), flush=True)
    assert error <= 2.0 ** -25 * np.sqrt(N * oH * oW) + 2.0 ** -24


@pytest.mark.parametrize("which", ["row", "column", "images", "few"])
@pytest.mark.parametrize("power", [27, 40, 60])
@pytest.mark.parametrize("case", LARGE)
def test_weight_gradient_of_mixed_rows(case, power, which):
    """Rows and columns that hold both sizes, the large elements against zeros: the small ones are the whole sum."""
    print("case", case, power, which, flush=True)
    N, Ci, Co, H, W, k, st, pad = case
    rng = np.random.default_rng(power)
    oH, oW = (H + 2 * pad - k) // st + 1, (W + 2 * pad - k) // st + 1
    x, gy = rng.standard_normal((N, Ci, H, W)), rng.standard_normal((N, Co, oH, oW))
    big = 2.0 ** power
    if which == "row":                    # half of every gradOutput plane is large, no image under its windows
        gy[..., oW // 2:] *= big
        x[..., oW // 2 * st - pad:] = 0
    elif which == "column":               # half of every image plane is large, no gradOutput where windows touch it
        x[..., W // 2:] *= big
        gy[..., max(0, (W // 2 + pad - k) // st + 1):] = 0
    elif which == "images":               # images that only the other operand's zeros keep apart
        x[0], gy[0] = 0, gy[0] * big
        x[3], gy[3] = x[3] * big, 0
    else:                                 # small elements everywhere, and rows of nothing else
        gy[rng.random(gy.shape) < 0.02] /= big
        x[rng.random(x.shape) < 0.02] /= big
        gy[:, :3] /= big
    x, gy = x.astype(np.float32), gy.astype(np.float32)
    ref, terms = _weight_gradient_exact(x, gy, k, st, pad)
    worst = np.abs(_weight_gradient(x, gy, k, st, pad) - ref) / (N * oH * oW * 2.0 ** -24 * terms + 2.0 ** -149)
    print("worst element at %.3g of its bound" % worst.max(), flush=True)
    assert worst.max() <= 1


def test_buffers_of_a_fixed_size():
    """A buffer tensor that cannot grow and holds just what the other kernels need leaves a call to those, bit for bit; one that holds
    what these need does not (the weight gradient on half-precision parts asks for one that can grow)."""
    import torch
    CT, THNN = cunn_amd.CudaTensor, cunn_amd.THNN
    rng = np.random.default_rng(11)
    N, Ci, Co, H, k = 16, 64, 128, 24, 3
    x, w, gy = (CT.from_numpy(rng.standard_normal(s).astype(np.float32)) for s in ((N, Ci, H, H), (Co, Ci * k * k), (N, Co, H, H)))
    a = (k, k, 1, 1, 1, 1)

    def call(which, buffer):
        out = CT.from_numpy(np.zeros(((N, Co, H, H), (N, Ci, H, H), (Co, Ci * k * k))[which], np.float32))
        if which == 0:
            THNN.SpatialConvolutionMM_updateOutput(x, out, w, None, buffer, CT(), *a)
        elif which == 1:
            THNN.SpatialConvolutionMM_updateGradInput(x, gy, out, w, buffer, CT(), *a)
        else:
            THNN.SpatialConvolutionMM_accGradParameters(x, gy, out, None, buffer, CT(), *a, 1.0)
        return out.numpy()

    for which in range(3):
        buffers, results = [], []
        for switch in ("0", "1"):
            cunn_amd.set_switch("THCUNN_CONV_HALVES", switch)
            buffers.append(CT())
            results.append(call(which, buffers[-1]))
        small, large = (b.numpy().size for b in buffers)
        print("pass", which, "floats", small, large, flush=True)
        assert small < large and not np.array_equal(*results)
        for floats, expected in ((small, results[0]), (large, results[0] if which == 2 else results[1])):
            assert np.array_equal(call(which, CT.from_torch(torch.zeros(floats, device="cuda"))), expected)


def test_captured_calls_do_not_allocate():
    """Buffers sized by the other kernels' needs: a captured call takes what fits them (the weight gradient on half-precision
    parts never does: five times the splits); after an eager call has sized them for these kernels, a captured one is theirs."""
    import ctypes
    lib, st = cunn_amd._lib.load(), cunn_amd.tensor.state()
    hip = ctypes.CDLL("libamdhip64.so")
    CT = cunn_amd.CudaTensor
    rng = np.random.default_rng(8)
    f = lambda *s: CT.from_numpy(rng.standard_normal(s).astype(np.float32))
    x, w, gy = f(4, 64, 16, 16), f(128, 64 * 9), f(4, 128, 16, 16)
    y, gx, gw = CT(), CT(), CT.from_numpy(np.zeros((128, 64 * 9), np.float32))
    bufs = [CT() for _ in range(3)]
    ones = CT()

    def step():
        a = (3, 3, 1, 1, 1, 1)
        cunn_amd.THNN.SpatialConvolutionMM_updateOutput(x, y, w, None, bufs[0], ones, *a)
        cunn_amd.THNN.SpatialConvolutionMM_updateGradInput(x, gy, gx, w, bufs[1], ones, *a)
        lib.THCudaTensor_fill(st, gw.handle, 0.0)
        cunn_amd.THNN.SpatialConvolutionMM_accGradParameters(x, gy, gw, None, bufs[2], ones, *a, 1.0)

    def results():
        lib.THCState_synchronize(st)
        return [t.numpy().copy() for t in (y, gx, gw)]

    s = ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(s)) == 0
    lib.THCState_setCurrentStream(st, s)
    try:
        cunn_amd.set_switch("THCUNN_CONV_HALVES", "0")
        step()
        plain = results()
        cunn_amd.set_switch("THCUNN_CONV_HALVES", "1")
        for warm in (False, True):
            print("warm", warm, flush=True)
            if warm:
                step()
                eager = results()
            graph, run = ctypes.c_void_p(), ctypes.c_void_p()
            assert hip.hipStreamBeginCapture(s, 0) == 0
            step()
            assert hip.hipStreamEndCapture(s, ctypes.byref(graph)) == 0
            assert hip.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)) == 0
            for _ in range(3):
                lib.THCudaTensor_fill(st, y.handle, -7.0)
                lib.THCState_synchronize(st)
                assert hip.hipGraphLaunch(run, s) == 0
                got = results()
                if warm:
                    assert all(np.array_equal(a, b) for a, b in zip(got, eager))
                else:
                    assert np.array_equal(got[2], plain[2])
                    # both within 3e-7 of the exact sums' norm
                    assert all(np.linalg.norm(a - b) <= 6e-7 * np.linalg.norm(b) for a, b in zip(got, plain))
                if warm:
                    step()
            assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0
    finally:
        lib.THCState_synchronize(st)
        lib.THCState_setCurrentStream(st, None)
        hip.hipStreamDestroy(s)


# Layers around the lines of the rule that gives a pass to these kernels, and far inside: sums of 900 terms and more, windows that
# mostly lie on the border, K split by the other kernels, strides.
RULE = [
    (43, 109, 120, 57, 36, 3, 1, 1),
    (24, 98, 98, 40, 40, 3, 1, 1),
    (34, 71, 50, 62, 18, 4, 1, 2),
    (28, 186, 26, 18, 36, 7, 1, 0),
    (62, 61, 296, 9, 26, 7, 1, 0),
    (32, 80, 192, 73, 73, 3, 1, 0),
    (16, 128, 128, 56, 56, 3, 1, 1),
    (16, 256, 256, 28, 28, 3, 1, 1),
    (10, 222, 374, 73, 60, 3, 2, 0),
    (39, 56, 329, 10, 62, 7, 2, 3),
]


@pytest.mark.parametrize("zeros", [False, True])
def test_no_less_exact_than_the_other_kernels(zeros):
    """By shape, with ordinary operands and with half of them zero (behind a ReLU): the error against 64 bits is not above that of
    the kernels that these replace (2 %: what another seed changes it by), wherever the rule takes these, which it does at times."""
    import torch
    F = torch.nn.functional
    taken = {"output": 0, "gradInput": 0}
    for case in RULE:
        N, Ci, Co, H, W, k, st, pad = case
        oH, oW = (H + 2 * pad - k) // st + 1, (W + 2 * pad - k) // st + 1
        g = torch.Generator(device="cuda").manual_seed(N)
        x, w, gy = (torch.randn(s, device="cuda", generator=g) for s in ((N, Ci, H, W), (Co, Ci * k * k), (N, Co, oH, oW)))
        if zeros:
            x, gy = x.clamp_min(0), gy * (torch.rand(gy.shape, device="cuda", generator=g) < 0.5)
        THNN, CT = cunn_amd.THNN, cunn_amd.CudaTensor
        results = []
        for switch in (None, "0"):
            cunn_amd.set_switch("THCUNN_CONV_HALVES", switch)
            y, gx = torch.zeros(N, Co, oH, oW, device="cuda"), torch.zeros_like(x)
            tx, tw, a = CT.from_torch(x), CT.from_torch(w), (k, k, st, st, pad, pad)
            THNN.SpatialConvolutionMM_updateOutput(tx, CT.from_torch(y), tw, None, CT(), CT(), *a)
            THNN.SpatialConvolutionMM_updateGradInput(tx, CT.from_torch(gy), CT.from_torch(gx), tw, CT(), CT(), *a)
            torch.cuda.synchronize()
            results.append((y, gx))
        wd, gd = w.double(), gy.double().flatten(2)
        exact = (torch.stack([wd @ F.unfold(x[n:n + 1].double(), k, padding=pad, stride=st)[0] for n in range(N)]).view_as(results[0][0]),
                 torch.cat([F.fold((wd.t() @ gd[n])[None], (H, W), k, padding=pad, stride=st) for n in range(N)]))
        for name, here, other, ref in zip(taken, *results, exact):
            if torch.equal(here, other):
                continue
            taken[name] += 1
            error, before = (float((v.double() - ref).norm() / ref.norm()) for v in (here, other))
            print(case, name, "error %.3g, the other kernels %.3g" % (error, before), flush=True)
            assert error <= 1.02 * before
    assert all(taken.values()), taken


@pytest.mark.parametrize("zeros", ["none", "input", "both"])
def test_weight_gradient_no_less_exact_than_the_other_kernels(zeros):
    """The same for the weight gradient, around its line and inside; one layer each beyond the line, and without the 16-byte fold."""
    import torch
    taken = []
    for case in ((64, 256, 256, 28, 28, 3, 1, 1), (30, 57, 120, 51, 48, 7, 1, 3), (15, 40, 371, 55, 42, 7, 1, 3), (32, 80, 192, 73, 73, 3, 1, 0),
                 (16, 256, 256, 28, 28, 3, 1, 1), (55, 105, 221, 72, 25, 3, 1, 0)):
        N, Ci, Co, H, W, k, st, pad = case
        oH, oW = (H + 2 * pad - k) // st + 1, (W + 2 * pad - k) // st + 1
        g = torch.Generator(device="cuda").manual_seed(N)
        x, gy = (torch.randn(s, device="cuda", generator=g) for s in ((N, Ci, H, W), (N, Co, oH, oW)))
        if zeros != "none":
            x = x.clamp_min(0)
        if zeros == "both":
            gy = gy * (torch.rand(gy.shape, device="cuda", generator=g) < 0.5)
        THNN, CT = cunn_amd.THNN, cunn_amd.CudaTensor
        results = []
        for switch in (None, "0"):
            cunn_amd.set_switch("THCUNN_CONV_HALVES", switch)
            gw = torch.zeros(Co, Ci * k * k, device="cuda")
            THNN.SpatialConvolutionMM_accGradParameters(CT.from_torch(x), CT.from_torch(gy), CT.from_torch(gw), None, CT(), CT(),
                                                        k, k, st, st, pad, pad, 1.0)
            torch.cuda.synchronize()
            results.append(gw)
        if torch.equal(*results):
            continue
        taken.append(case)
        ref = sum(gy[n].double().flatten(1) @ torch.nn.functional.unfold(x[n:n + 1].double(), k, padding=pad, stride=st)[0].t() for n in range(N))
        error, before = (float((v.double() - ref).norm() / ref.norm()) for v in results)
        print(case, zeros, "error %.3g, the other kernels %.3g" % (error, before), flush=True)
        assert error <= 1.02 * before
    assert 1 < len(taken) < 6, taken
