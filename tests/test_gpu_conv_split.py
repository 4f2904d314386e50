"""Convolutions multiply fp32 operands as six products of bf16 parts (SpatialConvolutionMM,
lib/THCUNN/generic/SpatialConvolutionMM.cu:58-486). Checked here: the error against a 64-bit sum stays below what
fp32 additions alone would give, also for one-signed and badly scaled operands and for the smallest floats beside the
largest, and infinities, NaNs and values that would round up to infinity as bf16 come out exactly as an fp32 convolution
gives them (an operand that is not finite must not spread to outputs it does not reach).

Bound of the error: a chain of K fp32 additions rounds K times, each by at most 2^-24 of the partial sum, with random
sign: about 2^-24 sqrt(K) / 2 of the result's norm for operands of mixed sign, and for one-signed operands (partial
sums that grow to the result) less than that."""
import numpy as np
import pytest

import cunn_amd

pytestmark = pytest.mark.gpu

from oracle import oracle as O  # noqa: E402

# N, Cin, Cout, H, W, k, stride, pad
CASES = [
    (2, 64, 128, 12, 12, 3, 1, 1),
    (3, 36, 70, 9, 11, 3, 2, 1),      # strided, ragged rows and columns
    (2, 20, 40, 14, 10, 5, 1, 0),
    (4, 512, 128, 7, 8, 1, 1, 0),     # 1x1 with a long reduction
    (2, 3, 24, 21, 19, 3, 1, 1),      # three input planes
    # the weight gradient's large tiles: 128 x 128 and 64 x 256, k-tiles inside an image or not, 16-byte or transposed gathers
    (2, 64, 120, 16, 16, 3, 2, 1),
    (3, 64, 120, 9, 12, 3, 1, 1),
    (2, 64, 128, 25, 25, 3, 2, 1),
    (2, 28, 60, 16, 16, 3, 1, 1),
    (2, 28, 60, 16, 16, 3, 2, 1),
    (3, 28, 60, 9, 12, 3, 1, 1),
    (3, 28, 60, 13, 14, 3, 1, 1),
    # the weight gradient's small tiles: 2x2, 2x1, 1x2 and 1x1 blocks, images shorter than a k-tile, padded rows of positions
    (3, 3, 64, 30, 28, 7, 2, 3),
    (2, 3, 50, 13, 11, 3, 1, 1),
    (2, 6, 24, 16, 12, 3, 1, 1),
    (5, 8, 32, 4, 4, 1, 1, 0),
    (4, 6, 24, 5, 5, 3, 1, 1),
    # bordered copies in runs: planes of an odd size, larger than a run, smaller with several to a run, wide rows
    (2, 8, 24, 67, 61, 3, 1, 1),
    (33, 64, 8, 37, 35, 3, 1, 1),
    (1, 8, 16, 3, 4500, 3, 1, 1),
    (9, 32, 8, 67, 61, 3, 1, 1),      # the same in longer runs
    (2, 32, 8, 3, 4500, 3, 1, 1),
]


def _tensors(case, kind, seed=5):
    N, Ci, Co, H, W, k, st, pad = case
    rng = np.random.default_rng(seed)
    oH, oW = (H + 2 * pad - k) // st + 1, (W + 2 * pad - k) // st + 1
    x, w, gy = (rng.standard_normal(s) for s in ((N, Ci, H, W), (Co, Ci * k * k), (N, Co, oH, oW)))
    if kind == "one-signed":
        x, w, gy = np.abs(x), np.abs(w), np.abs(gy)
    elif kind == "scaled":
        x *= np.exp2(np.round(rng.standard_normal(x.shape) * 4))
        gy *= np.exp2(np.round(rng.standard_normal(gy.shape) * 4))
    elif kind == "tiny":
        x, w = x * 1e-30, w * 1e-3
    elif kind == "smallest":             # the parts of these would be subnormal as bf16
        x, gy, w = x * 1e-35, gy * 1e-35, w + 2
    return tuple(v.astype(np.float32) for v in (x, w, gy))


def _passes(case, x, w, gy, gyw):
    """(output, gradInput from gy, gradWeight from gyw) of the library"""
    N, Ci, Co, H, W, k, st, pad = case
    THNN, CT = cunn_amd.THNN, cunn_amd.CudaTensor
    g = (k, k, st, st, pad, pad)
    tx, tw, y, gx, gw = CT.from_numpy(x), CT.from_numpy(w), CT(), CT(), CT.from_numpy(np.zeros_like(w))
    THNN.SpatialConvolutionMM_updateOutput(tx, y, tw, None, CT(), CT(), *g)
    THNN.SpatialConvolutionMM_updateGradInput(tx, CT.from_numpy(gy), gx, tw, CT(), CT(), *g)
    THNN.SpatialConvolutionMM_accGradParameters(tx, CT.from_numpy(gyw), gw, None, CT(), CT(), *g, 1.0)
    return y.numpy(), gx.numpy(), gw.numpy()


@pytest.mark.parametrize("kind", ["normal", "one-signed", "scaled", "tiny", "smallest"])
@pytest.mark.parametrize("case", CASES)
def test_error_against_64_bit_sums(case, kind):
    print("case", case, kind, flush=True)
    _check_error(case, kind)


def _check_error(case, kind):
    import torch
    N, Ci, Co, H, W, k, st, pad = case
    x, w, gy = _tensors(case, kind)
    dx, dw = (torch.from_numpy(v).double().requires_grad_() for v in (x, w.reshape(Co, Ci, k, k)))
    y = torch.nn.functional.conv2d(dx, dw, stride=st, padding=pad)
    y.backward(torch.from_numpy(gy).double())
    terms = (Ci * k * k, Co * k * k, N * gy.shape[2] * gy.shape[3])
    gyw = gy if kind != "smallest" else (gy * np.float32(1e35)).astype(np.float32)
    gw = torch.nn.grad.conv2d_weight(dx.detach(), dw.shape, torch.from_numpy(gyw).double(), stride=st, padding=pad)
    for got, ref, n in zip(_passes(case, x, w, gy, gyw), (y.detach(), dx.grad, gw), terms):
        ref = ref.numpy().reshape(got.shape)
        err = np.linalg.norm(got.astype(np.float64) - ref) / np.linalg.norm(ref)
        assert err <= 2.0 ** -25 * np.sqrt(n) + 2.0 ** -24, (err, n)   # + one rounding of the result


@pytest.mark.parametrize("case", CASES)
def test_non_finite_operands(case):
    print("case", case, flush=True)
    _check_non_finite(case)


def _check_non_finite(case, passes=3):
    N, Ci, Co, H, W, k, st, pad = case
    x, w, gy = _tensors(case, "normal", 6)
    w *= 1e-3
    x[0, 1, 2, 3], x[1 % N, 0, 4 % H, 4 % W], x[N - 1, Ci - 1, H - 1, W - 1], x[0, 2, H - 1, 0] = np.inf, np.nan, 3.4e38, -3.4e38
    gy[0, 3, 1, 2], gy[1 % N, 0, 0, 0] = -np.inf, np.nan
    gyw = gy * np.float32(1e-3)          # times 3.4e38 still finite: no sum overflows in one order and not in another
    gy[N - 1, Co - 1, 2, 1] = 3.4e38
    g = (k, k, st, st, pad, pad)
    with np.errstate(all="ignore"):
        gw = np.zeros_like(w)
        ref = (O.convmm_updateOutput(x, w, None, *g), O.convmm_updateGradInput(x.shape, gy, w, *g),
               O.convmm_accGradParameters(x, gyw, gw, None, *g, 1.0)[0])
    for name, got, r in list(zip(("output", "gradInput", "gradWeight"), _passes(case, x, w, gy, gyw), ref))[:passes]:
        print(name)
        assert np.array_equal(np.isnan(got), np.isnan(r)) and np.array_equal(np.isposinf(got), np.isposinf(r))
        assert np.array_equal(np.isneginf(got), np.isneginf(r))
        fine = np.isfinite(r)
        # relative to the largest term: 3.4e38 times a weight
        np.testing.assert_allclose(got[fine], r[fine], rtol=1e-5, atol=max(1e-4, 1e-6 * np.abs(r[fine], dtype=np.float64).max()))


def _same_special(got, ref):
    for f in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(f(got), f(ref)), f.__name__
    fine = np.isfinite(ref)
    np.testing.assert_allclose(got[fine], ref[fine], rtol=1e-5, atol=1e-4)


# A sum whose length is no multiple of the k-tile is filled up with zero weights, and what those are multiplied with is
# some element of the image: an infinity there must not reach outputs that it is no term of, nor turn into NaN where it is.
@pytest.mark.parametrize("direct", ["0", None])
@pytest.mark.parametrize("case", [(2, 8, 40, 13, 12, 3, 2, 0), (2, 6, 36, 11, 15, 5, 3, 1), (1, 8, 24, 9, 9, 2, 3, 0)])
def test_infinities_beside_filled_up_sums(case, direct):
    """Strided gradInput (phases of Cout x taps terms) and the transposed convolution's forward pass: infinities in the first
    plane, which the zero weights meet."""
    print("case", case, direct, flush=True)
    N, Ci, Co, H, W, k, st, pad = case
    _, w, gy = _tensors(case, "normal", 12)
    gy[0, 0, 1, 1], gy[N - 1, 0, 0, 2], gy[0, 0, gy.shape[2] - 1, 0] = np.inf, -np.inf, np.inf
    THNN, CT = cunn_amd.THNN, cunn_amd.CudaTensor
    g = (k, k, st, st, pad, pad)
    cunn_amd.set_switch("THCUNN_CONV_DIRECT", direct)
    try:
        gx, y = CT(), CT()
        THNN.SpatialConvolutionMM_updateGradInput(CT.from_numpy(np.zeros((N, Ci, H, W), np.float32)), CT.from_numpy(gy), gx,
                                                  CT.from_numpy(w), CT(), CT(), *g)
        wf, bias = w.reshape(Co, Ci, k, k), np.arange(Ci, dtype=np.float32)
        THNN.SpatialFullConvolution_updateOutput(CT.from_numpy(gy), y, CT.from_numpy(wf), CT.from_numpy(bias), CT(), CT(), *g, 0, 0)
    finally:
        cunn_amd.set_switch("THCUNN_CONV_DIRECT", None)
    with np.errstate(all="ignore"):
        _same_special(gx.numpy(), O.convmm_updateGradInput((N, Ci, H, W), gy, w, *g))
        _same_special(y.numpy(), O.fullconv_updateOutput(gy, wf, bias, *g))


@pytest.mark.parametrize("relu", [False, True])
@pytest.mark.parametrize("case", [(2, 3, 24, 21, 19, 3, 1, 1), (2, 3, 40, 15, 14, 7, 2, 3), (1, 3, 70, 9, 9, 1, 1, 0), (2, 5, 136, 10, 9, 3, 1, 0)])
def test_infinities_beside_filled_up_sums_forward(case, relu):
    print("case", case, relu, flush=True)
    N, Ci, Co, H, W, k, st, pad = case
    x, w, _ = _tensors(case, "normal", 13)
    x[0, 0, 3, 3], x[N - 1, 0, 0, 4], x[0, 0, H - 1, W - 1] = np.inf, -np.inf, np.inf
    THNN, CT = cunn_amd.THNN, cunn_amd.CudaTensor
    y, g = CT(), (k, k, st, st, pad, pad)
    f = THNN.SpatialConvolutionMMReLU_updateOutput if relu else THNN.SpatialConvolutionMM_updateOutput
    f(CT.from_numpy(x), y, CT.from_numpy(w), None, CT(), CT(), *g)
    with np.errstate(all="ignore"):
        ref = O.convmm_updateOutput(x, w, None, *g)
        if relu:
            ref = np.where(ref > 0, ref, np.float32(0))
    _same_special(y.numpy(), ref)


# Sizes of x and w (of gradOutput and x in the weight gradient): operands so small that a bf16 part of theirs would be
# subnormal, with partners large enough that the sums are ordinary numbers; and operands and sums above the range in which
# products are formed from parts. The bound is the one above: no size of an operand may cost precision.
SIZES = [(1e-33, 1e16), (1e-36, 1e19), (1e19, 1e-36), (1e-38, 1e21), (1e-39, 1e22), (1e30, 1e-39), (1e-39, 1e36), (1e15, 1e17)]


def _check_sizes(case, a, b, passes=3):
    import torch
    N, Ci, Co, H, W, k, st, pad = case
    x, w, gy = _tensors(case, "normal", 8)
    f = lambda v, s: (v.astype(np.float64) * s).astype(np.float32)
    x, w, gyw, gy = f(x, a), f(w, b), f(gy, b), f(gy, a)
    d = lambda v, *s: torch.from_numpy(v.reshape(*s) if s else v).double()
    dw = d(w, Co, Ci, k, k)
    refs = (torch.nn.functional.conv2d(d(x), dw, stride=st, padding=pad),
            torch.nn.grad.conv2d_input(x.shape, dw, d(gy), stride=st, padding=pad),
            torch.nn.grad.conv2d_weight(d(x), dw.shape, d(gyw), stride=st, padding=pad))
    terms = (Ci * k * k, Co * k * k, N * gy.shape[2] * gy.shape[3])
    for name, got, ref, n in list(zip(("output", "gradInput", "gradWeight"), _passes(case, x, w, gy, gyw), refs, terms))[:passes]:
        ref = ref.numpy().reshape(got.shape)
        err = np.linalg.norm(got.astype(np.float64) - ref) / np.linalg.norm(ref)
        assert err <= 2.0 ** -25 * np.sqrt(n) + 2.0 ** -24, (name, err, n)


@pytest.mark.parametrize("sizes", SIZES)
@pytest.mark.parametrize("case", CASES)
def test_small_operands_with_large_partners(case, sizes):
    print("case", case, sizes, flush=True)
    _check_sizes(case, *sizes)


@pytest.mark.parametrize("direct", ["0", "1", "2"])
def test_bias_of_any_size(direct):
    """The sums start from the bias in some kernels and meet it at the end in others: nothing of it may be lost or overflow."""
    case = (2, 32, 40, 9, 8, 3, 1, 1)
    print("direct", direct, flush=True)
    N, Ci, Co, H, W, k, st, pad = case
    x, w, _ = _tensors(case, "normal", 9)
    size = np.array([0, 1e-44, 1e-38, 1e-3, 1, 1e20, 1e26, 3e38])[np.arange(Co) % 8]
    bias = (size * np.where(np.arange(Co) % 3, 1, -1)).astype(np.float32)
    x = (x.astype(np.float64) * np.array([1, 1e-38])[:N, None, None, None]).astype(np.float32)
    cunn_amd.set_switch("THCUNN_CONV_DIRECT", direct)
    try:
        THNN, CT = cunn_amd.THNN, cunn_amd.CudaTensor
        y = CT()
        THNN.SpatialConvolutionMM_updateOutput(CT.from_numpy(x), y, CT.from_numpy(w), CT.from_numpy(bias), CT(), CT(), k, k, st, st, pad, pad)
        got = y.numpy()
    finally:
        cunn_amd.set_switch("THCUNN_CONV_DIRECT", None)
    K = Ci * k * k
    col = np.lib.stride_tricks.sliding_window_view(np.pad(x.astype(np.float64), ((0, 0), (0, 0), (1, 1), (1, 1))), (k, k), axis=(2, 3))
    W64 = w.astype(np.float64).reshape(Co, Ci, k, k)
    ref = np.einsum("ncijkl,ockl->noij", col, W64) + bias.astype(np.float64)[None, :, None, None]
    terms = np.einsum("ncijkl,ockl->noij", np.abs(col), np.abs(W64)) + np.abs(bias.astype(np.float64))[None, :, None, None]
    # K fp32 additions of what the terms add up to in magnitude, and a rounding to the smallest float
    assert (np.abs(got - ref) <= K * 2.0 ** -24 * terms + 2.0 ** -149).all()


# ---- the kernel for short calls: every tile shape, ragged rows and columns, fewer k-steps than waves, uneven slices ----
DIRECT = [
    (1, 16, 8, 5, 5, 1, 1, 0),       # one k-step: three of the four waves have none
    (1, 32, 40, 7, 7, 1, 1, 0),
    (1, 512, 130, 7, 7, 1, 1, 0),
    (2, 80, 33, 9, 8, 1, 1, 0),      # five k-steps
    (1, 16, 65, 13, 11, 3, 1, 1),
    (3, 48, 24, 10, 9, 3, 2, 1),
    (2, 32, 64, 9, 9, 5, 1, 0),
    (1, 512, 512, 14, 14, 1, 1, 0),
]


@pytest.mark.parametrize("shape", ["1", "2", None])
@pytest.mark.parametrize("case", DIRECT)
def test_short_calls(case, shape):
    print("case", case, shape, flush=True)
    cunn_amd.set_switch("THCUNN_CONV_DIRECT", shape)
    try:
        for kind in ("normal", "one-signed", "tiny", "smallest"):
            _check_error(case, kind)
        for sizes in SIZES:
            _check_sizes(case, *sizes, passes=2)
        _check_non_finite(case, passes=2)    # forward and gradInput
    finally:
        cunn_amd.set_switch("THCUNN_CONV_DIRECT", None)


# ---- the tiled kernels also where the kernel for short calls would be taken, and their 96-row tiles (65 ... 96 rows, a
#      strided gradInput by phases, split along K) ----
ROWS96 = [
    (2, 32, 80, 14, 13, 3, 1, 1),
    (2, 80, 40, 13, 12, 3, 1, 1),
    (2, 72, 16, 15, 14, 3, 2, 1),
    (1, 32, 96, 9, 9, 1, 1, 0),
    (2, 512, 96, 8, 8, 3, 1, 1),
]


@pytest.mark.parametrize("case", CASES + ROWS96)
def test_tiled(case):
    print("case", case, flush=True)
    cunn_amd.set_switch("THCUNN_CONV_DIRECT", "0")
    try:
        _check_error(case, "normal")
        _check_non_finite(case, passes=2)
    finally:
        cunn_amd.set_switch("THCUNN_CONV_DIRECT", None)
