"""The one-launch sum of few targets and the symmetric sum with 64- and
128-node tiles, at the edges of their ranges and of their tiles: against the
oracle (FP64 <= 1e-12, the bar of every direct sum; mixed <= 1e-6) on all rows
of the small sizes and on the first and last rows of the large ones. The
densities are random, the nodes a spiral on the sphere or an ellipse."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)


def _nodes(inti, dim, n, seed=0):
    i = np.arange(n) + 0.5
    if dim == 3:
        pol, az = np.arccos(1 - 2 * i / n), np.pi * (1 + 5 ** 0.5) * i
        X = np.stack([np.cos(az) * np.sin(pol), np.sin(az) * np.sin(pol), np.cos(pol)])
    else:
        X = np.stack([np.cos(2 * np.pi * i / n), 0.6 * np.sin(2 * np.pi * i / n)])
    N = X / np.linalg.norm(X, axis=0)
    w = np.random.default_rng(seed).uniform(0.5, 1.5, n) / n
    return inti.Quadrature(X, N, w, np.zeros((1, 0), dtype=np.int64))


def _kernel(inti, pde, dim, kind):
    op = inti.Laplace(dim=dim) if pde == 0 else inti.Helmholtz(k=7.3, dim=dim)
    if kind == 4:
        c = (-7.3j, 1.0) if pde else (0.4, 1.0)
        return inti.CombinedFieldKernel(op, *c, "SD"), c
    names = {0: inti.SingleLayerKernel, 1: inti.DoubleLayerKernel, 2: inti.AdjointDoubleLayerKernel,
             3: inti.HyperSingularKernel}
    return names[kind](op), None


def _check(inti, oracle, pde, dim, kind, Q, T, precision, alpha=1.0, beta=0.0, identity=0.0):
    k = 7.3 if pde else 0.0
    K, coefs = _kernel(inti, pde, dim, kind)
    A = inti.IntegralOperator(K, T, Q, precision=precision)
    rng = np.random.default_rng(3)
    n, m = len(Q), len(T)
    x = rng.normal(size=n) + (1j * rng.normal(size=n) if pde else 0.0)
    y0 = rng.normal(size=m) + (1j * rng.normal(size=m) if pde else 0.0)
    if identity:
        A.set_identity(identity)
    y = A.apply(x, y0.copy(), alpha=alpha, beta=beta)  # writes into its y
    ref = np.zeros(m, dtype=np.complex128)
    blocks = [(0, m)] if m * n <= 1.7e7 else [(0, 130), (m - 130, m)]
    rows = np.concatenate([np.arange(*b) for b in blocks])
    for b in blocks:
        r = oracle.matvec(pde, dim, kind, k, T, Q, x, coefs=coefs, rows=b)
        ref[b[0]:b[1]] = r[b[0]:b[1]]
    ref = alpha * (ref + (identity * x if identity else 0.0)) + beta * y0
    err, size = np.linalg.norm((y - ref)[rows]), np.linalg.norm(ref[rows])
    say(f"[gpu] pde {pde} dim {dim} kind {kind} {precision} m={m} n={n}: {err:.2e} of {size:.2e}")
    assert err <= (1e-12 if precision == "fp64" else 1e-6) * size  # (one node alone: both are zero)


@pytest.mark.parametrize("pde,dim,kind", [(0, 2, 1), (0, 3, 0), (0, 3, 3), (1, 2, 4), (1, 3, 4), (1, 3, 2)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [1, 3, 65, 257, 1799, 1801, 3401])
def test_square(inti, oracle, pde, dim, kind, precision, n):
    Q = _nodes(inti, dim, n)
    _check(inti, oracle, pde, dim, kind, Q, Q, precision)


# the 64 / 128 and 128 / 256 tile edges (two partial tiles among them)
@pytest.mark.parametrize("pde,dim,kind,n", [(0, 3, 1, 9855), (0, 3, 1, 9985), (1, 3, 4, 9857), (1, 3, 4, 10050),
                                            (0, 2, 0, 48705), (0, 3, 0, 49025), (1, 3, 4, 48897), (1, 2, 4, 46000)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_tile_edges(inti, oracle, pde, dim, kind, n, precision):
    Q = _nodes(inti, dim, n)
    _check(inti, oracle, pde, dim, kind, Q, Q, precision)


# targets that are not the sources: few and many, with alpha, beta
@pytest.mark.parametrize("pde,dim,kind", [(0, 3, 1), (1, 2, 0), (1, 3, 4)])
@pytest.mark.parametrize("m,n", [(1, 5000), (5, 8192), (7, 8193), (1023, 700), (1025, 9000), (2501, 640)])
def test_rectangular(inti, oracle, pde, dim, kind, m, n):
    Q = _nodes(inti, dim, n)
    T = _nodes(inti, dim, m, seed=1)
    T = inti.Quadrature(1.7 * T.coords, T.normals, T.weights, T.qtags)
    _check(inti, oracle, pde, dim, kind, Q, T, "fp64", alpha=1.3, beta=-0.4)


@pytest.mark.parametrize("n", [500, 5000])
def test_identity(inti, oracle, n):
    Q = _nodes(inti, 3, n)
    _check(inti, oracle, 1, 3, 4, Q, Q, "fp64", alpha=0.5 - 0.2j, beta=0.3j, identity=0.5 + 0.1j)


@pytest.mark.parametrize("n", [700, 1500, 9000, 20000])
def test_repeat_is_bit_identical(inti, n):
    Q = _nodes(inti, 3, n)
    A = inti.IntegralOperator(_kernel(inti, 1, 3, 4)[0], Q, Q)
    x = np.random.default_rng(5).normal(size=n) + 0j
    assert np.array_equal(A @ x, A @ x)


# four right-hand sides at once: around the largest one-launch sums, the plans
# of one LDS tile per chunk, and a remainder of single columns
@pytest.mark.parametrize("pde,dim,kind", [(0, 2, 1), (0, 3, 3), (1, 2, 4), (1, 3, 1)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n,nrhs", [(1, 4), (67, 5), (1801, 4), (2201, 4), (3701, 6), (2900, 16)])
def test_columns(inti, oracle, pde, dim, kind, precision, n, nrhs):
    Q = _nodes(inti, dim, n)
    K, coefs = _kernel(inti, pde, dim, kind)
    A = inti.IntegralOperator(K, Q, Q, precision=precision)
    rng = np.random.default_rng(11)
    x = rng.normal(size=(n, nrhs)) + (1j * rng.normal(size=(n, nrhs)) if pde else 0.0)
    y = A @ x
    for r in range(nrhs):
        ref = oracle.matvec(pde, dim, kind, 7.3 if pde else 0.0, Q, Q, np.ascontiguousarray(x[:, r]), coefs=coefs)
        err, size = np.linalg.norm(y[:, r] - ref), np.linalg.norm(ref)
        say(f"[gpu] pde {pde} dim {dim} kind {kind} {precision} n={n} column {r}: {err:.2e} of {size:.2e}")
        assert err <= (1e-12 if precision == "fp64" else 1e-6) * size


# an apply in place: no row may be written while others still read it
@pytest.mark.parametrize("nrhs", [1, 4])
def test_in_place(inti, nrhs):
    n = 1500
    Q = _nodes(inti, 3, n)
    A = inti.IntegralOperator(_kernel(inti, 1, 3, 4)[0], Q, Q)
    rng = np.random.default_rng(13)
    x = rng.normal(size=(nrhs, n)) + 1j * rng.normal(size=(nrhs, n))
    ctx, lib, hip = A.ctx, A.ctx.lib, ctypes.CDLL("libamdhip64.so")
    one, zero = (ctypes.c_double * 2)(1.0, 0.0), (ctypes.c_double * 2)(0.0, 0.0)
    dx = ctypes.c_void_p()
    assert hip.hipMalloc(ctypes.byref(dx), ctypes.c_size_t(x.nbytes)) == 0
    assert hip.hipMemcpy(dx, x.ctypes.data_as(ctypes.c_void_p), ctypes.c_size_t(x.nbytes), 1) == 0
    ctx.check(lib.inti_op_apply_device(A.handle, nrhs, dx, n, dx, n, one, zero))
    ctx.synchronize()
    y = np.empty_like(x)
    assert hip.hipMemcpy(y.ctypes.data_as(ctypes.c_void_p), dx, ctypes.c_size_t(x.nbytes), 2) == 0
    assert hip.hipFree(dx) == 0
    ref = np.stack([A @ x[r] for r in range(nrhs)])
    err = np.linalg.norm(y - ref) / np.linalg.norm(ref)
    say(f"[gpu] in place, {nrhs} columns: {err:.2e}")
    assert err <= 1e-12


# an explicit source split below the sizes whose 256-node tiles fill the GPU:
# the same one-direction sum as without the symmetric one, bit for bit
@pytest.mark.parametrize("pde,dim,kind,n", [(0, 3, 0, 300), (1, 3, 4, 4320), (1, 2, 1, 5000)])
def test_explicit_split(inti, pde, dim, kind, n):
    Q = _nodes(inti, dim, n)
    x = np.random.default_rng(5).normal(size=n) + (1j if pde else 0.0)
    out = {}
    for sym in (0, 1):
        A = inti.IntegralOperator(_kernel(inti, pde, dim, kind)[0], Q, Q)
        A.set_symmetric(sym)
        for split in (1, 2, 7):
            A.ctx.check(A.ctx.lib.inti_op_set_launch(A.handle, 256, 1, split))
            out[sym, split] = A @ x
    for split in (1, 2, 7):
        assert np.array_equal(out[0, split], out[1, split])
    err = np.linalg.norm(out[1, 1] - out[1, 2]) / np.linalg.norm(out[1, 1])
    say(f"[gpu] explicit split pde {pde} dim {dim} n={n}: 1 / 2 chunks differ by {err:.1e}")
    assert 0 < err <= 1e-13


# an explicit group in automatic mode: below two blocks of 256-node tile pairs
# per CU the sum without the symmetric one, above it the group's own, bit for bit
@pytest.mark.parametrize("pde,dim,kind,precision", [(0, 3, 0, "mixed"), (1, 3, 4, "fp64"), (1, 2, 1, "fp64")])
@pytest.mark.parametrize("n", [300, 4320, 7900, 9000])
@pytest.mark.parametrize("group", [1, 2, 4])
def test_explicit_group(inti, pde, dim, kind, precision, n, group):
    Q = _nodes(inti, dim, n)
    x = np.random.default_rng(5).normal(size=n) + (1j if pde else 0.0)
    A, B = (inti.IntegralOperator(_kernel(inti, pde, dim, kind)[0], Q, Q, precision=precision) for _ in range(2))
    A.set_symmetric(1, group)
    B.set_symmetric(2 if n == 9000 else 0, group)
    assert np.array_equal(A @ x, B @ x)


# both sides of the lines between the one-launch sum and the one-direction one
# (long chains, many targets of few sources, far fields), against the
# one-direction sum in chunks of its own: the same terms in another order
@pytest.mark.parametrize("pde,dim,kind", [(0, 2, "SL"), (0, 3, "DL"), (1, 2, "CF"), (1, 3, "SL"), (1, 2, "FFSL"),
                                          (1, 2, "FFCF"), (1, 3, "FFDL")])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("m,n", [(3, 3657), (3, 6145), (300, 8193), (1023, 16400), (1024, 8200), (2050, 3100), (20480, 64),
                                 (20481, 65), (180001, 5), (1000003, 3)])
@pytest.mark.parametrize("nrhs", [1, 4])
def test_row_lines(inti, pde, dim, kind, precision, m, n, nrhs):
    Q, T = _nodes(inti, dim, n), _nodes(inti, dim, m, seed=1)
    T = inti.points(T.coords / np.linalg.norm(T.coords, axis=0) if "FF" in kind else 1.7 * T.coords)
    op = inti.Helmholtz(k=7.3, dim=dim) if pde else inti.Laplace(dim=dim)
    K = (inti.CombinedFieldKernel(op, -7.3j, 1.0, "FF" if "FF" in kind else "SD") if "CF" in kind else
         {"SL": inti.SingleLayerKernel, "DL": inti.DoubleLayerKernel, "FFSL": inti.FarFieldSingleLayerKernel,
          "FFDL": inti.FarFieldDoubleLayerKernel}[kind](op))
    rng = np.random.default_rng(17)
    x = rng.normal(size=(n, nrhs)) + (1j * rng.normal(size=(n, nrhs)) if pde else 0.0)
    A = inti.IntegralOperator(K, T, Q, precision=precision)
    y = A @ x
    A.ctx.check(A.ctx.lib.inti_op_set_launch(A.handle, 256, 1, 3))
    ref = A @ x
    err, size = np.linalg.norm(y - ref), np.linalg.norm(ref)
    say(f"[gpu] {pde} {dim} {kind} {precision} {m} x {n}, {nrhs} columns: {err:.2e} of {size:.2e}")
    assert err <= (1e-13 if precision == "fp64" else 1e-6) * size


def test_more_targets_than_a_launch_of_64_threads_each(inti):
    """2^26 targets of three 2D Helmholtz sources (64 threads per target would
    be 2^32): accepted, and its first, middle and last rows those of a small sum
    (1e-13, the same pairs by the other kernel)."""
    m, Q = 1 << 26, _nodes(inti, 2, 3)
    X = np.empty((2, m))
    X[0], X[1] = np.linspace(2.0, 9.0, m), 0.5
    K = inti.SingleLayerKernel(inti.Helmholtz(k=1.3, dim=2))
    x = np.array([1.0, -0.5j, 0.25 + 1j])
    rows = np.r_[0:5, m // 2:m // 2 + 5, m - 5:m]
    y = inti.IntegralOperator(K, inti.points(X), Q).apply(x)[rows]
    ref = inti.IntegralOperator(K, inti.points(np.ascontiguousarray(X[:, rows])), Q) @ x
    say(f"[gpu] {m} targets: {np.linalg.norm(y - ref) / np.linalg.norm(ref):.2e}")
    assert np.linalg.norm(y - ref) <= 1e-13 * np.linalg.norm(ref)


# both sides of the rounds of 256-node tile pairs that some kinds keep
@pytest.mark.parametrize("pde,dim,kind", [(0, 2, 1), (0, 3, 3), (1, 3, 0), (0, 2, 0)])
@pytest.mark.parametrize("n", [16128, 16129, 25599])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_full_rounds(inti, oracle, pde, dim, kind, n, precision):
    Q = _nodes(inti, dim, n)
    _check(inti, oracle, pde, dim, kind, Q, Q, precision)
