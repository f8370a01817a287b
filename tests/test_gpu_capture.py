"""Applies captured after one eager call of the same operator on a fresh
context: nothing may be allocated while the stream records, whatever the eager
call's route was. One column in place after one column out of place (small
sums in one launch need no scratch of their own), one column after 16 (at
70,003 nodes the symmetric sum's slots are larger than the 16 columns' partial
sums), and the one-direction sum after the symmetric one. Three replays with
eager work between them, each against the eager result (1e-13: other sums of
the same terms)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
CONTEXTS = []  # outlive the operators on them


@pytest.mark.parametrize("pde,dim,n,eager_cols,in_place,sym", [(1, 3, 1500, 1, True, 1), (1, 2, 700, 4, True, 1),
                                                               (0, 2, 70003, 16, False, 1), (0, 3, 9000, 1, False, 0)])
def test_captured_after_one_eager_call(inti, pde, dim, n, eager_cols, in_place, sym):
    hip, ctx = ctypes.CDLL("libamdhip64.so"), inti.Context(0)
    CONTEXTS.append(ctx)
    i = np.arange(n) + 0.5
    if dim == 3:
        pol, az = np.arccos(1 - 2 * i / n), np.pi * (1 + 5 ** 0.5) * i
        X = np.stack([np.cos(az) * np.sin(pol), np.sin(az) * np.sin(pol), np.cos(pol)])
    else:
        X = np.stack([np.cos(2 * np.pi * i / n), 0.6 * np.sin(2 * np.pi * i / n)])
    Q = inti.Quadrature(X, X / np.linalg.norm(X, axis=0), np.full(n, 1.0 / n), np.zeros((1, 0), dtype=np.int64))
    K = inti.DoubleLayerKernel(inti.Helmholtz(k=3.0, dim=dim) if pde else inti.Laplace(dim=dim))
    A = inti.IntegralOperator(K, Q, Q, ctx=ctx)
    rng = np.random.default_rng(7)
    x = rng.normal(size=(eager_cols, n)) + (1j * rng.normal(size=(eager_cols, n)) if pde else 0.0)
    one, zero = (ctypes.c_double * 2)(1.0, 0.0), (ctypes.c_double * 2)(0.0, 0.0)
    dx, dy = ctypes.c_void_p(), ctypes.c_void_p()
    for d in (dx, dy):
        assert hip.hipMalloc(ctypes.byref(d), ctypes.c_size_t(x.nbytes)) == 0

    def copy(dst, src, kind, nbytes):
        assert hip.hipMemcpy(dst, src, ctypes.c_size_t(nbytes), kind) == 0

    def apply(cols, out):
        return ctx.lib.inti_op_apply_device(A.handle, cols, dx, n, out, n, one, zero)

    copy(dx, x.ctypes.data_as(ctypes.c_void_p), 1, x.nbytes)
    ctx.check(apply(eager_cols, dy))
    ctx.synchronize()
    A.set_symmetric(sym)
    s, graph, run = ctypes.c_void_p(ctx.stream()), ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamBeginCapture(s, 1) == 0
    rc = apply(1, dx if in_place else dy)
    assert hip.hipStreamEndCapture(s, ctypes.byref(graph)) == 0
    ctx.check(rc)
    assert hip.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)) == 0
    for r in range(3):
        v = np.ascontiguousarray((r + 1.0) * x[0][::-1])
        y = np.empty_like(v)
        copy(dx, v.ctypes.data_as(ctypes.c_void_p), 1, v.nbytes)
        assert hip.hipGraphLaunch(run, s) == 0
        ctx.synchronize()
        copy(y.ctypes.data_as(ctypes.c_void_p), dx if in_place else dy, 2, y.nbytes)
        copy(dx, v.ctypes.data_as(ctypes.c_void_p), 1, v.nbytes)
        ctx.check(apply(1, dy))
        ctx.synchronize()
        ref = np.empty_like(v)
        copy(ref.ctypes.data_as(ctypes.c_void_p), dy, 2, ref.nbytes)
        err = np.linalg.norm(y - ref) / np.linalg.norm(ref)
        print(f"[gpu] n {n}, {eager_cols} eager columns, in place {in_place}: replay {r} {err:.2e}", flush=True)
        assert err <= 1e-13
    assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0
    assert hip.hipFree(dx) == 0 and hip.hipFree(dy) == 0


def test_dense_product_outlives_builds(inti):
    hip, ctx = ctypes.CDLL("libamdhip64.so"), inti.Context(0)
    CONTEXTS.append(ctx)
    Q = inti.sphere_quadrature(3, qorder=4)
    n, nrhs, op = len(Q), 3, inti.Helmholtz(k=2.0, dim=3)
    S = inti.IntegralOperator(inti.SingleLayerKernel(op), Q, Q, ctx=ctx)
    D = inti.IntegralOperator(inti.DoubleLayerKernel(op), Q, Q, ctx=ctx)
    M = inti.DenseOperator(D)
    rng = np.random.default_rng(3)
    x = rng.normal(size=(nrhs, n)) + 1j * rng.normal(size=(nrhs, n))
    ref, y = np.ascontiguousarray(M.apply(x.T).T), np.empty_like(x)
    one, zero = (ctypes.c_double * 2)(1.0, 0.0), (ctypes.c_double * 2)(0.0, 0.0)
    dx, dy, graph, run = (ctypes.c_void_p() for _ in range(4))
    for d in (dx, dy):
        assert hip.hipMalloc(ctypes.byref(d), ctypes.c_size_t(x.nbytes)) == 0
    assert hip.hipMemcpy(dx, x.ctypes.data_as(ctypes.c_void_p), ctypes.c_size_t(x.nbytes), 1) == 0
    s = ctypes.c_void_p(ctx.stream())
    assert hip.hipStreamBeginCapture(s, 1) == 0
    rc = ctx.lib.inti_dense_gemm(ctx.handle, 1, n, n, nrhs, M.device_pointer, n, dx, n, dy, n, one, zero)
    assert hip.hipStreamEndCapture(s, ctypes.byref(graph)) == 0
    ctx.check(rc)
    assert hip.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)) == 0
    for r in range(3):
        dS, dD = inti.bdim_correction(op, Q, Q, S, D, green_multiplier=np.full(n, -0.5))
        E = inti.IntegralOperator(inti.DoubleLayerKernel(op), Q, Q, ctx=ctx)
        E.attach(dD)
        E.attach(dS, 0.3)
        E.pullback(x[0], x[1])
        assert hip.hipMemcpy(dy, x.ctypes.data_as(ctypes.c_void_p), ctypes.c_size_t(x.nbytes), 1) == 0
        assert hip.hipGraphLaunch(run, s) == 0
        ctx.synchronize()
        assert hip.hipMemcpy(y.ctypes.data_as(ctypes.c_void_p), dy, ctypes.c_size_t(x.nbytes), 2) == 0
        print(f"[gpu] dense product, replay {r}: {np.linalg.norm(y - ref) / np.linalg.norm(ref):.2e}", flush=True)
        assert np.array_equal(y, ref)
    assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0
    assert hip.hipFree(dx) == 0 and hip.hipFree(dy) == 0
