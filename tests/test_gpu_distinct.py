"""Coincident nodes of a quadrature, found when its first operator is made:
a node repeated within a tile of 256, in the next tile or in the last,
partial one, a pair closer than the coincidence tolerance apart, and none.
The symmetric sum drops its coincidence mask only for distinct nodes; with a
coincident pair left unmasked the sums are infinite or NaN, so the apply is
compared with the oracle (FP64 <= 1e-12)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("shuffled", [False, True])
@pytest.mark.parametrize("pair", [None, (10, 200), (255, 256), (3, 2299), (700, 1900)])
@pytest.mark.parametrize("gap", [0.0, 4e-15])
def test_coincident_nodes(inti, oracle, dim, shuffled, pair, gap):
    n = 2300
    i = np.arange(n) + 0.5
    if dim == 3:
        pol, az = np.arccos(1 - 2 * i / n), np.pi * (1 + 5 ** 0.5) * i
        X = np.stack([np.cos(az) * np.sin(pol), np.sin(az) * np.sin(pol), np.cos(pol)])
    else:
        X = np.stack([np.cos(2 * np.pi * i / n), np.sin(2 * np.pi * i / n)])
    rng = np.random.default_rng(0)
    if shuffled:
        X = X[:, rng.permutation(n)]
    if pair:
        X[:, pair[1]] = X[:, pair[0]]
        X[0, pair[1]] += gap
    Q = inti.Quadrature(X, X / np.linalg.norm(X, axis=0), np.full(n, 1.0 / n), np.zeros((1, 0), dtype=np.int64))
    A = inti.IntegralOperator(inti.SingleLayerKernel(inti.Laplace(dim=dim)), Q, Q)
    A.set_symmetric(2)
    x = rng.normal(size=n)
    y, ref = A @ x, oracle.matvec(0, dim, 0, 0.0, Q, Q, x).real
    print(f"[gpu] dim {dim} shuffled {shuffled} pair {pair} gap {gap}: "
          f"{np.linalg.norm(y - ref) / np.linalg.norm(ref):.2e}", flush=True)
    assert np.linalg.norm(y - ref) <= 1e-12 * np.linalg.norm(ref)


def test_many_nodes(inti):
    """More pairs of tiles than one launch holds blocks for (5,793 tiles: 2^24
    blocks of 256 threads would be 2^32 threads): the operator is made, and
    sums at three of its nodes on the unit circle, where the double layer's
    kernel is -1/(4 pi), are -(n - 1) / (2 n): neighbours 4e-6 apart leave
    errors of 2^-53 / r^2, in all 1e-11."""
    n = 5793 * 256 - 5
    t = 2 * np.pi * np.arange(n) / n
    X = np.stack([np.cos(t), np.sin(t)])
    Q = inti.Quadrature(X, X, np.full(n, 2 * np.pi / n), np.zeros((1, 0), dtype=np.int64))
    A = inti.IntegralOperator(inti.DoubleLayerKernel(inti.Laplace(dim=2)), Q, Q)
    A.handle
    T = inti.points(X[:, [0, n // 3, n - 1]])
    y = inti.IntegralOperator(inti.DoubleLayerKernel(inti.Laplace(dim=2)), T, Q) @ np.ones(n)
    print(f"[gpu] {n} nodes: {y}", flush=True)
    assert np.all(np.abs(y + 0.5 - 0.5 / n) <= 1e-9)


@pytest.mark.parametrize("captured", ["own stream", "another stream"])
@pytest.mark.parametrize("pair", [None, (3, 900)])
def test_operator_made_during_a_capture(inti, oracle, captured, pair):
    """An operator made while a stream is captured in the global mode (its
    context's own, where the test is put off, or another): the capture ends
    whole, its graph replays, and the operator masks a coincident pair."""
    hip = ctypes.CDLL("libamdhip64.so")
    n = 1300
    i = np.arange(n) + 0.5
    X = np.stack([np.cos(2 * np.pi * i / n), np.sin(2 * np.pi * i / n)])
    if pair:
        X[:, pair[1]] = X[:, pair[0]]
    Q = inti.Quadrature(X, X, np.full(n, 1.0 / n), np.zeros((1, 0), dtype=np.int64))
    ctx = inti.default_context()
    Q.device(ctx)
    own, stream, dev = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    ctx.check(ctx.lib.inti_ctx_stream(ctx.handle, ctypes.byref(own)))
    assert hip.hipStreamCreateWithFlags(ctypes.byref(stream), 1) == 0
    s = own if captured == "own stream" else stream
    src, dst = (ctypes.c_double * 4)(1.0, 2.0, 3.0, 4.0), (ctypes.c_double * 4)()
    assert hip.hipMalloc(ctypes.byref(dev), ctypes.c_size_t(64)) == 0
    up = ctypes.c_void_p(dev.value + 32)
    assert hip.hipMemcpy(dev, src, ctypes.c_size_t(32), 1) == 0
    graph, run = ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamBeginCapture(s, 0) == 0
    try:
        rc = hip.hipMemcpyAsync(up, dev, ctypes.c_size_t(32), 3, s)
        A = inti.IntegralOperator(inti.SingleLayerKernel(inti.Laplace(dim=2)), Q, Q)
        A.handle
    finally:
        ended = hip.hipStreamEndCapture(s, ctypes.byref(graph))
    assert rc == 0 and ended == 0
    assert hip.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)) == 0
    x = np.random.default_rng(1).normal(size=n)
    ref = oracle.matvec(0, 2, 0, 0.0, Q, Q, x).real
    B = inti.IntegralOperator(inti.SingleLayerKernel(inti.Laplace(dim=2)), Q, Q)
    for r in range(3):
        src[0] = float(r)
        assert hip.hipMemcpy(dev, src, ctypes.c_size_t(32), 1) == 0
        assert hip.hipGraphLaunch(run, s) == 0 and hip.hipStreamSynchronize(s) == 0
        assert hip.hipMemcpy(dst, up, ctypes.c_size_t(32), 2) == 0
        assert list(dst) == list(src)
        for op in (A, B):
            op.set_symmetric(2)
            y = op @ x
            print(f"[gpu] {captured}, pair {pair}: {np.linalg.norm(y - ref) / np.linalg.norm(ref):.2e}", flush=True)
            assert np.linalg.norm(y - ref) <= 1e-12 * np.linalg.norm(ref)
    assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0
    assert hip.hipFree(dev) == 0 and hip.hipStreamDestroy(stream) == 0
