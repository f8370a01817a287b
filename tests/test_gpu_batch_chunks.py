"""The automatic chunk length of a batch: batches that take 256- and 512-source
chunks, and an explicit 2048, each against the problems' own operators (1e-13
FP64, the bar of the batched apply), for 1, 4 and 16 densities."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(51, 300), (257, 1290, 700), (900,) * 40])
@pytest.mark.parametrize("nrhs", [1, 4, 16])
def test_chunks(inti, sizes, nrhs):
    quads = [inti.ellipse_quadrature(1.0 + 0.01 * p, 0.5, s, qorder=5) for p, s in enumerate(sizes)]
    kern = [inti.DoubleLayerKernel(inti.Helmholtz(k=2.0 + 0.3 * p, dim=2)) for p in range(len(sizes))]
    B = inti.BatchOperator(kern, quads)
    rng = np.random.default_rng(0)
    X = rng.normal(size=(B.ntot, nrhs)) + 1j * rng.normal(size=(B.ntot, nrhs))
    Y = B.apply(X)
    B.set_launch(2048, 0)
    Z = B.apply(X)
    assert np.linalg.norm(Y - Z) <= 1e-13 * np.linalg.norm(Z)
    for p in (0, len(sizes) - 1):
        o = slice(B.offsets[p], B.offsets[p + 1])
        ref = inti.IntegralOperator(kern[p], quads[p], quads[p]).apply(X[o])
        err = np.linalg.norm(Y[o] - ref) / np.linalg.norm(ref)
        print(f"[gpu] batch of {len(sizes)}, {nrhs} densities, problem {p}: {err:.2e}", flush=True)
        assert err <= 1e-13
