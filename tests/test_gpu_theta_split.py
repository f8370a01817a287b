"""The source split of Theta at its edges: sizes below 8 chunks of 256 sources
(fewest rounds), from 8 chunks on, and from 16, with node counts that leave
ragged chunks, in 2D and 3D. The corrected double layer on a smooth density
against the oracle's, <= 1e-12 (rules of 3 and 6 nodes, whose least squares
are well conditioned there)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pde,dim,size", [(0, 2, 681), (0, 2, 683), (1, 2, 1365), (1, 2, 1367), (0, 3, 4), (1, 3, 4),
                                          (0, 3, 5), (1, 3, 6)])
def test_split(inti, oracle, pde, dim, size):
    Q = inti.ellipse_quadrature(1.0, 0.7, size, qorder=5) if dim == 2 else inti.sphere_quadrature(size, qorder=4)
    k = 3.0 if pde else 0.0
    op = inti.Helmholtz(k=k, dim=dim) if pde else inti.Laplace(dim=dim)
    S = inti.IntegralOperator(inti.SingleLayerKernel(op), Q, Q)
    D = inti.IntegralOperator(inti.DoubleLayerKernel(op), Q, Q)
    mu = np.full(len(Q), -0.5)
    dS, dD = inti.bdim_correction(op, Q, Q, S, D, green_multiplier=mu)
    x = np.cos(Q.coords[0] + 2 * Q.coords[1]) + (0.3j * Q.coords[0] if pde else 0.0)
    D.attach(dD)
    ref = oracle.corrected_matvec(pde, dim, 1, k, Q, x, mu, which="D")
    y = D @ x
    err = np.linalg.norm(y - ref) / np.linalg.norm(ref)
    print(f"[gpu] pde {pde} dim {dim} n {len(Q)}: {err:.2e}", flush=True)
    assert err <= 1e-12
