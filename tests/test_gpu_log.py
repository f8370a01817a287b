"""The FP64 logarithm of the 2D Laplace single layer (-log(d) / (2 pi)), one
source against targets on an axis, so that d is exact: every binade, both
sides of the reduction's edges (1, sqrt(1/2), sqrt 2, powers of two), tiny and
huge distances, and an infinite one, against the extended-precision logarithm.
d^2 is rounded once (2^-53 of the logarithm, absolute), the logarithm and the
two products each to within an ulp: 4 * 2^-53 (1 + |log d^2|) / (4 pi)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_log(inti):
    e = np.arange(-40, 40)
    near = np.concatenate([[c * (1 + s * t) for t in (0.0, 2.0 ** -52, 1e-12, 1e-3)] for c in (1.0, 2 ** 0.5, 2 ** -0.25,
                                                                                          2 ** 0.25, 0.5, 4.0)
                           for s in (1, -1)])
    d = np.concatenate([2.0 ** e, 1.37 * 2.0 ** e, near, np.exp(np.linspace(-27, 27, 4001))])
    T = inti.points(np.stack([d, np.zeros_like(d)]))
    src = inti.Quadrature(np.zeros((2, 1)), np.array([[1.0], [0.0]]), np.ones(1), np.zeros((1, 0), dtype=np.int64))
    y = inti.IntegralOperator(inti.SingleLayerKernel(inti.Laplace(dim=2)), T, src) @ np.ones(1)
    ref = -np.log(d.astype(np.longdouble)) / (2 * np.pi)
    tol = 4 * 2.0 ** -53 * (1 + 2 * np.abs(ref) * 2 * np.pi) / (4 * np.pi)
    err = np.abs(y - ref)
    print(f"[gpu] log: largest error {np.max(err / tol):.2f} of its bound", flush=True)
    assert np.all(err <= tol)
    T = inti.points(np.array([[np.inf, 1.0], [0.0, 0.0]]))
    y = inti.IntegralOperator(inti.SingleLayerKernel(inti.Laplace(dim=2)), T, src) @ np.ones(1)
    assert y[0] == -np.inf and y[1] == 0.0
