"""Backward pass of BatchNormalization in training with a team of workgroups per channel (bn_teams.h): one piece and many,
pieces that end inside a plane, the last piece short, planes off the 16-byte boundaries, more planes than lanes, and every
workgroup computing the pieces that it does not wait for itself (the bounded wait forced to zero polls; the numbers have to be
the same bit for bit). Shapes alternate on one stream, so that launches find what others left in the shared scratch block.

Against 64-bit formulas. Bounds: the sums are of at most 32 floats per lane and a tree, merged in double, so a
few units in the last place (2^-24 each) of quantities of the outputs' size; 2e-6 of the norm is four times the measured worst."""
import ctypes

import numpy as np
import pytest

import cunn_amd

pytestmark = pytest.mark.gpu

SHAPES = [
    (8, 16, 28, 28),       # one piece
    (32, 20, 56, 56),      # pieces end inside a plane
    (9, 33, 30, 44),
    (40, 5, 27, 27),       # not a multiple of 4
    (3, 100, 61, 35),
    (300, 3, 4, 8),        # more planes than a walk step holds units
    (700, 2, 3, 5),
    (2, 7, 150, 180),
    (2, 300, 3),           # 3-D, tiny
]


def _passes(shape, relu, seed, inplace=False):
    THNN, CT = cunn_amd.THNN, cunn_amd.CudaTensor
    rng = np.random.default_rng(seed)
    C = shape[1]
    x = (rng.standard_normal(shape) * 2 + 0.5).astype(np.float32)
    gy = rng.standard_normal(shape).astype(np.float32)
    w, b = (rng.random(C) + 0.5).astype(np.float32), rng.standard_normal(C).astype(np.float32)
    ax = tuple(i for i in range(len(shape)) if i != 1)
    bc = (1, C) + (1,) * (len(shape) - 2)
    xd, n = x.astype(np.float64), x.size // C
    mean, var = xd.mean(ax), xd.var(ax)
    inv = 1 / np.sqrt(var + 1e-5)
    xh = (xd - mean.reshape(bc)) * inv.reshape(bc)
    z = xh * w.reshape(bc) + b.reshape(bc)
    if relu:               # signs within rounding of zero are anyone's: no gradient there
        gy[np.abs(z) < 1e-4] = 0
    gd = gy * (z > 0) if relu else gy.astype(np.float64)
    g0, g1 = gd.sum(ax), (gd * xh).sum(ax)
    gx = (gd - (g0.reshape(bc) + xh * g1.reshape(bc)) / n) * (w.astype(np.float64) * inv).reshape(bc)
    ref = [np.maximum(z, 0) if relu else z, gx, g1, g0, mean, inv, 0.9 * 1 + 0.1 * var * n / (n - 1)]
    t = [CT.from_numpy(v) for v in (x, gy, w, b, np.zeros(C, np.float32), np.ones(C, np.float32))]
    tx, tgy, tw, tb, rm, rv = t
    sm, ss, gg, gb = (CT.from_numpy(np.zeros(C, np.float32)) for _ in range(4))
    y, tgx = CT.from_numpy(np.zeros(shape, np.float32)), CT.from_numpy(np.zeros(shape, np.float32))
    if relu:
        THNN.BatchNormalizationReLU_updateOutput(tx, y, tw, tb, rm, rv, sm, ss, True, 0.1, 1e-5)
        THNN.BatchNormalizationReLU_backward(tx, tgy, tgx, gg, gb, tw, tb, rm, rv, sm, ss, True, 1.0, 1e-5)
    else:
        THNN.BatchNormalization_updateOutput(tx, y, tw, tb, rm, rv, sm, ss, True, 0.1, 1e-5)
        if inplace:
            tgx = tgy
        THNN.BatchNormalization_backward(tx, tgy, tgx, gg, gb, tw, rm, rv, sm, ss, True, 1.0, 1e-5)
        if inplace:
            rm2, rv2 = CT.from_numpy(np.zeros(C, np.float32)), CT.from_numpy(np.ones(C, np.float32))
            THNN.BatchNormalization_updateOutput(tx, tx, tw, tb, rm2, rv2, sm, ss, True, 0.1, 1e-5)
            y = tx
    return [v.numpy() for v in (y, tgx, gg, gb, sm, ss, rv)], ref


def _check(got, ref):
    for name, a, r in zip(("output", "gradInput", "gradWeight", "gradBias", "mean", "1/std", "runningVar"), got, ref):
        scale = max(np.linalg.norm(r), 1e-3 * np.sqrt(r.size))
        assert np.linalg.norm(a.astype(np.float64) - r) <= 2e-6 * scale, name


@pytest.mark.parametrize("relu", [False, True])
def test_teams(relu):
    for rounds in range(2):
        for i, shape in enumerate(SHAPES):
            print("case", shape, relu, rounds, flush=True)
            results = []
            for mode in ("1", "2"):
                cunn_amd.set_switch("THCUNN_BN_TEAMS", mode)
                try:
                    got, ref = _passes(shape, relu, 20 + i)
                finally:
                    cunn_amd.set_switch("THCUNN_BN_TEAMS", None)
                _check(got, ref)
                results.append(got)
            for a, b in zip(*results):
                assert np.array_equal(a, b)


@pytest.mark.parametrize("shape", [(16, 24, 56, 56), (64, 128, 28, 28), (8, 40, 27, 27)])
def test_by_shape_and_over_the_input(shape):
    """The kernels that the rule takes; results written over the input or gradOutput come from kernels that allow it."""
    print("case", shape, flush=True)
    for inplace in (False, True):
        _check(*_passes(shape, False, 41, inplace))


@pytest.mark.parametrize("shape, warm", [((64, 128, 28, 28), False), ((64, 128, 28, 28), True), ((16, 40, 56, 56), True)])
def test_capture(shape, warm):
    """A call that has a kernel without scratch takes that one, captured also as the first call on its stream; one that always
    needed scratch is captured on the teams once they ran. Either gives the bits of an eager call."""
    THNN, CT = cunn_amd.THNN, cunn_amd.CudaTensor
    lib, st = cunn_amd._lib.load(), cunn_amd.tensor.state()
    hip = ctypes.CDLL("libamdhip64.so")
    print("case", shape, warm, flush=True)
    rng = np.random.default_rng(3)
    C = shape[1]
    tx, tgy, tw, tb = (CT.from_numpy(rng.standard_normal(s).astype(np.float32)) for s in (shape, shape, C, C))
    rm, rv = CT.from_numpy(np.zeros(C, np.float32)), CT.from_numpy(np.ones(C, np.float32))
    sm, ss, gg, gb = (CT.from_numpy(np.zeros(C, np.float32)) for _ in range(4))
    y, gx = CT.from_numpy(np.zeros(shape, np.float32)), CT.from_numpy(np.zeros(shape, np.float32))
    THNN.BatchNormalization_updateOutput(tx, y, tw, tb, rm, rv, sm, ss, True, 0.1, 1e-5)

    def backward():
        for t in (gg, gb):
            lib.THCudaTensor_fill(st, t.handle, 0.0)
        THNN.BatchNormalization_backward(tx, tgy, gx, gg, gb, tw, rm, rv, sm, ss, True, 1.0, 1e-5)

    def results():
        lib.THCState_synchronize(st)
        return [t.numpy().copy() for t in (gx, gg, gb)]

    backward()
    expected = results()
    s, graph, run = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(s)) == 0
    lib.THCState_setCurrentStream(st, s)
    try:
        if warm:
            backward()
            results()
        assert hip.hipStreamBeginCapture(s, 0) == 0
        backward()
        assert hip.hipStreamEndCapture(s, ctypes.byref(graph)) == 0
        assert hip.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)) == 0
        for _ in range(3):
            lib.THCudaTensor_fill(st, gx.handle, -7.0)
            lib.THCState_synchronize(st)
            assert hip.hipGraphLaunch(run, s) == 0
            for a, b in zip(results(), expected):
                assert np.array_equal(a, b)
            backward()
        lib.THCState_synchronize(st)
        assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0
    finally:
        lib.THCState_synchronize(st)
        lib.THCState_setCurrentStream(st, None)
        hip.hipStreamDestroy(s)


def test_replays_beside_eager_calls():
    """A captured graph replayed on another stream while calls of other shapes run on the one it was captured on, and after a larger
    call has made the scratch grow: neither side finds what the other leaves, then or later."""
    THNN, CT = cunn_amd.THNN, cunn_amd.CudaTensor
    lib, st = cunn_amd._lib.load(), cunn_amd.tensor.state()
    hip = ctypes.CDLL("libamdhip64.so")
    rng = np.random.default_rng(6)

    def layer(shape):
        C = shape[1]
        f = lambda *s: CT.from_numpy(rng.standard_normal(s).astype(np.float32))
        z = lambda: CT.from_numpy(np.zeros(C, np.float32))
        x, gy, w, rm, rv, sm, ss, gg, gb = f(*shape), f(*shape), f(C), z(), CT.from_numpy(np.ones(C, np.float32)), z(), z(), z(), z()
        y, gx = CT.from_numpy(np.zeros(shape, np.float32)), CT.from_numpy(np.zeros(shape, np.float32))
        THNN.BatchNormalization_updateOutput(x, y, w, z(), rm, rv, sm, ss, True, 0.1, 1e-5)

        def backward():
            for t in (gg, gb):
                lib.THCudaTensor_fill(st, t.handle, 0.0)
            THNN.BatchNormalization_backward(x, gy, gx, gg, gb, w, rm, rv, sm, ss, True, 1.0, 1e-5)
        return backward, lambda: [t.numpy().copy() for t in (gx, gg, gb)], gx

    (graphed, graphed_out, graphed_gx), (eager, eager_out, _), (larger, larger_out, _) = (
        layer(s) for s in ((16, 40, 56, 56), (16, 24, 72, 72), (64, 48, 112, 112)))
    s, t, graph, run = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(s)) == 0 and hip.hipStreamCreate(ctypes.byref(t)) == 0
    lib.THCState_setCurrentStream(st, s)
    try:
        graphed(), eager()
        lib.THCState_synchronize(st)
        want_graphed, want_eager = graphed_out(), eager_out()
        assert hip.hipStreamBeginCapture(s, 0) == 0
        graphed()
        assert hip.hipStreamEndCapture(s, ctypes.byref(graph)) == 0
        assert hip.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)) == 0
        for turn in range(3):
            print("turn", turn, flush=True)
            lib.THCudaTensor_fill(st, graphed_gx.handle, -7.0)
            lib.THCState_synchronize(st)
            for _ in range(20):
                assert hip.hipGraphLaunch(run, t) == 0
                eager()
            if turn == 1:
                larger()
            lib.THCState_synchronize(st)
            assert hip.hipStreamSynchronize(t) == 0
            for got, want in ((graphed_out(), want_graphed), (eager_out(), want_eager)):
                assert all(np.array_equal(a, b) for a, b in zip(got, want))
        want = larger_out()
        larger()
        lib.THCState_synchronize(st)
        assert all(np.array_equal(a, b) for a, b in zip(larger_out(), want))
        assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0
    finally:
        lib.THCState_synchronize(st)
        lib.THCState_setCurrentStream(st, None)
        hip.hipStreamDestroy(s)
        hip.hipStreamDestroy(t)
