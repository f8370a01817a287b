"""The Gram-Schmidt kernels of GMRES at the edges of their blocks: systems of
one row, of one row past a 64-row group and of more rows than 256 blocks of 64
hold, restarts below, at and past the 64 columns of a sum and the 256
Hessenberg entries in LDS, real and complex, with and without the captured
step. Both solves run all `maxiter` steps of a well-conditioned system
(I/2 + K with a small K); the residual of the returned x, recomputed with the
operator, equals the reported one, and x solves the dense system to 1e-10
where the dense matrix is small."""
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
