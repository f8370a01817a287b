"""The symmetric pullback with 128- and 256-node tiles against the two passes,
at the edges of its range and of its tiles: every gradient to 1e-11 of its own
size (FP64 sums of up to 20,000 terms in another order, with cancellation)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _nodes(inti, dim, n):
    i = np.arange(n) + 0.5
    if dim == 3:
        pol, az = np.arccos(1 - 2 * i / n), np.pi * (1 + 5 ** 0.5) * i
        X = np.stack([np.cos(az) * np.sin(pol), np.sin(az) * np.sin(pol), np.cos(pol)])
    else:
        X = np.stack([np.cos(2 * np.pi * i / n), 0.6 * np.sin(2 * np.pi * i / n)])
    w = np.random.default_rng(2).uniform(0.5, 1.5, n) / n
    return inti.Quadrature(X, X / np.linalg.norm(X, axis=0), w, np.zeros((1, 0), dtype=np.int64))


@pytest.mark.parametrize("pde,dim,kind", [(0, 2, "DL"), (0, 3, "SL"), (1, 2, "CF"), (1, 3, "CF"), (1, 3, "DL")])
@pytest.mark.parametrize("n", [1, 128, 129, 255, 257, 1025, 19969])
@pytest.mark.parametrize("comb", [True, False])
def test_tiles_match_two_passes(inti, pde, dim, kind, n, comb):
    Q = _nodes(inti, dim, n)
    op = inti.Helmholtz(k=4.1, dim=dim) if pde else inti.Laplace(dim=dim)
    K = {"SL": inti.SingleLayerKernel, "DL": inti.DoubleLayerKernel}[kind](op) if kind != "CF" else \
        inti.CombinedFieldKernel(op, -4.1j, 1.0, "SD")
    rng = np.random.default_rng(4)
    x, u = (rng.normal(size=n) + (1j * rng.normal(size=n) if pde else 0.0) for _ in range(2))
    wrt = ("sigma", "source_normals", "source_weights") + (("nodes",) if comb else ("source_nodes", "target_nodes"))
    wrt += ("k",) if pde else ()
    out = {}
    for mode in (0, 1):
        A = inti.IntegralOperator(K, Q, Q)
        A.set_symmetric(mode)
        out[mode] = A.pullback(u, x, wrt=wrt, **({"dcoefs": (-1j, 0.0)} if kind == "CF" else {}))
    for key in wrt:
        a, b = np.asarray(out[1][key]), np.asarray(out[0][key])
        err, size = np.linalg.norm(a - b), np.linalg.norm(b)
        if key == "k":  # one number, the sum of n terms of any sign
            size = max(size, np.linalg.norm(u) * np.linalg.norm(x) / n)
        print(f"[gpu] pde {pde} dim {dim} {kind} n={n} {key}: {err:.2e} of {size:.2e}", flush=True)
        assert err <= 1e-11 * size


@pytest.mark.parametrize("pde,dim,kind", [(0, 2, "DL"), (0, 3, "SL"), (0, 3, "DL"), (1, 2, "CF"), (1, 3, "SL"), (1, 3, "CF")])
@pytest.mark.parametrize("n,mode,group", [(700, 2, 0), (700, 2, 1), (700, 2, 2), (1300, 2, 4), (1025, 1, 0), (7900, 1, 0),
                                          (10001, 1, 0), (10001, 2, 2), (49409, 1, 0), (66000, 1, 0)])
def test_sigma_only_tiles(inti, pde, dim, kind, n, mode, group):
    """sigma-bar alone, A^H ubar, by the transposed symmetric sum: 64-node tiles
    (small n), 128 (10,001), 256 (explicit groups, and 49,409 nodes up) and both
    forms of its reduction (16 slots, 65,536 nodes), against the one-direction
    sum, to 1e-12 of its size (FP64 sums of n terms of one size in another order:
    sqrt(66,000) 2^-53 = 3e-14)."""
    Q = _nodes(inti, dim, n)
    op = inti.Helmholtz(k=4.1, dim=dim) if pde else inti.Laplace(dim=dim)
    K = {"SL": inti.SingleLayerKernel, "DL": inti.DoubleLayerKernel}[kind](op) if kind != "CF" else \
        inti.CombinedFieldKernel(op, -4.1j, 1.0, "SD")
    rng = np.random.default_rng(6)
    x, u = (rng.normal(size=n) + (1j * rng.normal(size=n) if pde else 0.0) for _ in range(2))
    out = {}
    for m, g in ((0, 0), (mode, group)):
        A = inti.IntegralOperator(K, Q, Q)
        A.set_symmetric(m, g)
        out[m] = A.pullback(u, x, wrt=("sigma",))["sigma"]
    err, size = np.linalg.norm(out[mode] - out[0]), np.linalg.norm(out[0])
    print(f"[gpu] sigma-bar pde {pde} dim {dim} {kind} n={n} mode {mode} group {group}: {err:.2e} of {size:.2e}", flush=True)
    assert err <= 1e-12 * size
