"""The transposed pattern of an attached correction (built on the GPU by the
attach) through sigma-bar = A^H ubar: corrections of each element's own nodes (a
pattern that is its own transpose), of these and twenty more targets for one
element (nearly so: the lookup finds an entry missing and the sort runs), of all targets for every element (columns of every length up to all rows), and
of all targets for a few elements only (long and short columns, some empty).
Against the dense matrix's conjugate transpose (1e-12: sums of a few hundred
terms), twice attached, and bit-identical for two operators. The first pullback
after an attach is an ordinary one: nothing is left for it to build."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _near(n, ne, lists):
    ptr = np.concatenate([[0], np.cumsum([len(l) for l in lists])]).astype(np.int64)
    return ptr, np.concatenate(lists).astype(np.int64)


@pytest.mark.parametrize("pde", [0, 1])
@pytest.mark.parametrize("pattern", ["own", "lopsided", "all", "few", "targets"])
def test_sigma_bar(inti, pde, pattern):
    Q = inti.sphere_quadrature(2, qorder=4)
    n, ne = len(Q), Q.ne
    op = inti.Helmholtz(k=2.0, dim=3) if pde else inti.Laplace(dim=3)
    T = inti.Quadrature(1.02 * Q.coords[:, 5:], Q.normals[:, 5:], Q.weights[5:], np.zeros((1, 0), dtype=np.int64)) \
        if pattern == "targets" else Q
    m = len(T)
    every, own = np.arange(m), [np.sort(Q.qtags[:, e]) for e in range(ne)]
    near = {"own": None, "lopsided": _near(n, ne, [np.union1d(own[e], every[100:120]) if e == 70 else own[e] for e in range(ne)]),
            "all": _near(n, ne, [every] * ne),
            "few": _near(n, ne, [every if e % 7 == 3 else own[e] if e % 7 < 3 else own[0][:0] for e in range(ne)]),
            "targets": _near(n, ne, [every[e % 3::3] if e < 60 else every[:0] for e in range(ne)])}[pattern]
    S, D = (inti.IntegralOperator(K(op), T, Q) for K in (inti.SingleLayerKernel, inti.DoubleLayerKernel))
    dS, dD = inti.bdim_correction(op, T, Q, S, D, green_multiplier=np.full(m, -0.5 if T is Q else 0.0), near=near)
    rng = np.random.default_rng(1)
    u, x = (rng.normal(size=s) + (1j * rng.normal(size=s) if pde else 0.0) for s in (m, n))
    M = inti.assemble_matrix(D) + dD.to_scipy() + 0.3 * dS.to_scipy()
    ref = np.asarray(np.conj(M).T @ u).ravel()
    out = []
    for _ in range(2):
        A = inti.IntegralOperator(inti.DoubleLayerKernel(op), T, Q)
        A.attach(dD)
        A.attach(dS, 0.3)
        out.append(A.pullback(u, x, wrt=("sigma",))["sigma"])
    lengths = np.diff(dD.to_scipy().tocsc().indptr)
    err = np.linalg.norm(out[0] - ref) / np.linalg.norm(ref)
    print(f"[gpu] pde {pde} {pattern}: columns of {lengths.min()} to {lengths.max()} entries, {err:.2e}", flush=True)
    assert err <= 1e-12
    assert np.array_equal(out[0], out[1])
    A.detach()
    B = inti.IntegralOperator(inti.DoubleLayerKernel(op), T, Q)
    assert np.array_equal(A.pullback(u, x)["sigma"], B.pullback(u, x)["sigma"])


def test_first_pullback_is_an_ordinary_one(inti):
    """Nothing of the pattern is left for the first gradient (it had cost four
    pullbacks' time at this size): the median first one of nine operators takes
    no more than twice the median second one."""
    Q = inti.sphere_quadrature(6, qorder=4)
    n, op = len(Q), inti.Laplace(dim=3)
    S, D = (inti.IntegralOperator(K(op), Q, Q) for K in (inti.SingleLayerKernel, inti.DoubleLayerKernel))
    _, dD = inti.bdim_correction(op, Q, Q, S, D, green_multiplier=np.full(n, -0.5))
    u = np.random.default_rng(0).normal(size=n)
    times = [[], []]
    for _ in range(9):
        A = inti.IntegralOperator(inti.DoubleLayerKernel(op), Q, Q)
        A.attach(dD)
        for t in times:
            t0 = time.perf_counter()
            A.pullback(u, u)
            t.append(time.perf_counter() - t0)
    first, second = (np.median(t) * 1e6 for t in times)
    print(f"[gpu] pullback of {n} nodes: first {first:.0f} us, second {second:.0f} us", flush=True)
    assert first <= 2 * second
