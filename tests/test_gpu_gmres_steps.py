"""The Gram-Schmidt kernels of GMRES. test_gmres_edges: systems of one row, of
one row past a 64-row group and of more rows than 256 blocks of 64 hold, real
and complex, with and without the captured step; well conditioned (I/2 + K with
a small K), they converge in about ten steps: the residual of the returned x,
recomputed with the operator, equals the reported one, and x solves the dense
system to 1e-10 where the dense matrix is small. test_gmres_long_bases: systems
that don't converge, so that every step of the stated restarts runs (past the 64
columns of a sum, the 256 and 512 Hessenberg entries held in LDS, and over
restarts of one captured step), against GMRES in numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pde", [0, 1])
@pytest.mark.parametrize("use_graph", [False, True])
@pytest.mark.parametrize("n,restart,maxiter", [(1, 4, 4), (2, 3, 3), (65, 70, 70), (300, 64, 200), (1000, 65, 65),
                                               (700, 300, 290), (16500, 20, 20)])
def test_gmres_edges(inti, pde, use_graph, n, restart, maxiter):
    i = np.arange(n) + 0.5
    pol, az = np.arccos(1 - 2 * i / n), np.pi * (1 + 5 ** 0.5) * i
    X = np.stack([np.cos(az) * np.sin(pol), np.sin(az) * np.sin(pol), np.cos(pol)])
    rng = np.random.default_rng(0)
    X *= rng.uniform(0.7, 1.3, n)
    Q = inti.Quadrature(X, X / np.linalg.norm(X, axis=0), np.full(n, 1.0 / n), np.zeros((1, 0), dtype=np.int64))
    op = inti.Helmholtz(k=4.0, dim=3) if pde else inti.Laplace(dim=3)
    A = inti.IntegralOperator(inti.DoubleLayerKernel(op), Q, Q)
    A.set_identity(0.5)
    b = rng.normal(size=n) + (1j * rng.normal(size=n) if pde else 0.0)
    x, info = inti.gmres(A, b, restart=restart, maxiter=maxiter, rtol=1e-13, use_graph=use_graph)
    rel = np.linalg.norm(b - A @ x) / np.linalg.norm(b)
    print(f"[gpu] pde {pde} n {n} restart {restart}: {info['iterations']} steps, {info['relres']:.2e} / {rel:.2e}",
          flush=True)
    assert abs(rel - info["relres"]) <= 1e-14 + 1e-6 * rel
    if n <= 1000:
        M = inti.assemble_matrix(A) + 0.5 * np.eye(n)
        assert np.linalg.norm(x - np.linalg.solve(M, b)) <= 1e-10 * np.linalg.norm(x)
    else:
        assert rel < 1e-6


def _numpy_gmres(A, b, restart, maxiter):
    x, it = np.zeros_like(b), 0
    while it < maxiter:
        m, r = min(restart, maxiter - it), b - A @ x
        V, H = np.zeros((len(b), m + 1), dtype=A.dtype), np.zeros((m + 1, m), dtype=A.dtype)
        V[:, 0] = r / np.linalg.norm(r)
        for k in range(m):
            w = A @ V[:, k]
            for _ in range(2):
                h = V[:, :k + 1].conj().T @ w
                H[:k + 1, k] += h
                w = w - V[:, :k + 1] @ h
            H[k + 1, k] = np.linalg.norm(w)
            V[:, k + 1] = w / H[k + 1, k]
        e = np.zeros(m + 1, dtype=A.dtype)
        e[0] = np.linalg.norm(r)
        x, it = x + V[:, :m] @ np.linalg.lstsq(H, e, rcond=None)[0], it + m
    return x


# first-kind single layers on scattered nodes, the node itself left out: spectra
# on both sides of zero, condition numbers of 5e2 to 3e5. Where restarts stagnate
# rounding travels from cycle to cycle, so the bar is the reference's own spread
# when the matrix entries move in their last bits (2^-52), times 30.
@pytest.mark.parametrize("pde", [0, 1])
@pytest.mark.parametrize("use_graph", [False, True])
@pytest.mark.parametrize("n,restart,maxiter", [(300, 70, 200), (700, 300, 300), (1200, 520, 520)])
def test_gmres_long_bases(inti, pde, use_graph, n, restart, maxiter):
    i = np.arange(n) + 0.5
    pol, az = np.arccos(1 - 2 * i / n), np.pi * (1 + 5 ** 0.5) * i
    X = np.stack([np.cos(az) * np.sin(pol), np.sin(az) * np.sin(pol), np.cos(pol)])
    rng = np.random.default_rng(0)
    X *= rng.uniform(0.7, 1.3, n)
    Q = inti.Quadrature(X, X / np.linalg.norm(X, axis=0), np.full(n, 1.0 / n), np.zeros((1, 0), dtype=np.int64))
    A = inti.IntegralOperator(inti.SingleLayerKernel(inti.Helmholtz(k=0.5, dim=3) if pde else inti.Laplace(dim=3)), Q, Q)
    b = rng.normal(size=n) + (1j * rng.normal(size=n) if pde else 0.0)
    x, info = inti.gmres(A, b, restart=restart, maxiter=maxiter, rtol=1e-13, use_graph=use_graph)
    M = np.ascontiguousarray(inti.assemble_matrix(A))
    ref, moved = (_numpy_gmres(M * (1 + s * 2.0 ** -52 * rng.uniform(-1, 1, M.shape)), b, restart, maxiter) for s in (0, 1))
    rel, want, off = (np.linalg.norm(b - M @ v) / np.linalg.norm(b) for v in (x, ref, moved))
    err, spread = (np.linalg.norm(v - ref) / np.linalg.norm(ref) for v in (x, moved))
    print(f"[gpu] pde {pde} n {n} restart {restart}: {info['iterations']} steps, {rel:.3e} ({want:.3e}, {off - want:.0e}), "
          f"x {err:.1e} ({spread:.0e})", flush=True)
    assert info["iterations"] == maxiter
    assert abs(rel - info["relres"]) <= 1e-14 + 1e-6 * rel
    assert abs(rel - want) <= 30 * abs(off - want) + 1e-12 and err <= 30 * spread + 1e-12
