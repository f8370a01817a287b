"""What is timed: the calls that a program on corrected Nystrom operators makes.

A program builds quadratures and DIM corrections, applies operators to one or
many densities (by hand or inside GMRES), evaluates potentials off the
surface, and differentiates an objective through the operator. Each family
below is one of those calls, through the package's Python interface or the
C-ABI of include/inti_amd.h, over the sizes of this repository's workloads,
examples and tests:

  matvec     y = (A + dA) x, operands resident on the device
  solve      GMRES on a corrected combined-field operator, host operands
  build      DIM correction of a combined-field operator and its first apply
  potential  single- and double-layer potentials at points off the surface
  pullback   every gradient of y = A sigma (density, nodes, normals, weights, k)
  batch      one block-diagonal operator over many 2D boundaries, 16 densities
  dense      an assembled corrected matrix times a block of densities

listed(): the cases; draw(rng): one more of the same ranges; prepare(case,
seed): what the program holds before the call; run(state): one call;
exact(case, seed): what the call returns, in 64 bits, in plain torch and numpy
(the meshes and seeded densities are the inputs, shared with prepare);
work(case): the operations and bytes that the call cannot do without.
"""
import ctypes as C
import math

import numpy as np
import torch

from __graft_entry__ import load_package

inti = load_package()
DEV = "cuda" if torch.cuda.is_available() else "cpu"

# canonical operations of one ordered pair (combined field c0 SL + c1 DL,
# factors of one node hoisted); a Hankel evaluation counts as 40
PAIR_FLOPS = {("laplace", 2, "SL"): 6, ("laplace", 2, "DL"): 10, ("laplace", 3, "SL"): 10,
              ("laplace", 3, "DL"): 17, ("laplace", 3, "HS"): 26, ("helmholtz", 2, "SL"): 50,
              ("helmholtz", 2, "DL"): 60, ("helmholtz", 2, "CF"): 70, ("helmholtz", 3, "SL"): 20,
              ("helmholtz", 3, "DL"): 28, ("helmholtz", 3, "HS"): 44, ("helmholtz", 3, "CF"): 36}


def listed():
    return [
        # smallest call: one application of a corrected 2D Laplace double
        # layer on 128 elements (launches and latency)
        {"name": "matvec_laplace2d_dl_640", "do": "matvec", "pde": "laplace", "dim": 2, "kind": "DL", "nel": 128,
         "q": 9, "prec": "fp64", "nrhs": 1},
        # 2D scattering by an ellipse, resolved at k = 40: the operator that
        # an iterative solver applies
        {"name": "matvec_helm2d_cf_6006", "do": "matvec", "pde": "helmholtz", "dim": 2, "kind": "CF", "nel": 1001,
         "q": 11, "prec": "fp64", "nrhs": 1, "k": 40.0},
        # 3D scattering, an everyday size, in double precision
        {"name": "matvec_helm3d_cf_12000", "do": "matvec", "pde": "helmholtz", "dim": 3, "kind": "CF", "nel": 10,
         "q": 4, "prec": "fp64", "nrhs": 1, "k": 2 * math.pi},
        # 3D scattering at the size of the headline benchmark, mixed precision
        {"name": "matvec_helm3d_cf_63480_mixed", "do": "matvec", "pde": "helmholtz", "dim": 3, "kind": "CF",
         "nel": 23, "q": 4, "prec": "mixed", "nrhs": 1, "k": 2 * math.pi},
        # a large first-kind electrostatics operator
        {"name": "matvec_laplace3d_sl_122880", "do": "matvec", "pde": "laplace", "dim": 3, "kind": "SL", "nel": 32,
         "q": 4, "prec": "fp64", "nrhs": 1},
        # many incident waves at once, matrix-free
        {"name": "matvec_helm3d_dl_17280_16rhs", "do": "matvec", "pde": "helmholtz", "dim": 3, "kind": "DL",
         "nel": 12, "q": 4, "prec": "fp64", "nrhs": 16, "k": 2 * math.pi},
        # a whole scattering solve at a small size
        {"name": "solve_helm3d_cf_4320", "do": "solve", "pde": "helmholtz", "dim": 3, "nel": 6, "q": 4,
         "k": 2 * math.pi},
        # set-up of a new geometry: the correction and the first apply
        {"name": "build_helm3d_cf_30720", "do": "build", "pde": "helmholtz", "dim": 3, "nel": 16, "q": 4,
         "k": 2 * math.pi},
        # the scattered field on a plotting grid
        {"name": "potential_helm2d_40401", "do": "potential", "pde": "helmholtz", "dim": 2, "nel": 500, "q": 9,
         "m": 40401, "k": 20.0},
        # shape derivatives of a scattering objective
        {"name": "pullback_helm3d_cf_12000", "do": "pullback", "dim": 3, "nel": 10, "q": 4, "k": 10.0},
        # a sweep over shapes and wavenumbers
        {"name": "batch_helm2d_dl_16rhs", "do": "batch", "nprob": 48, "lo": 50, "hi": 1400, "q": 7,
         "prec": "mixed"},
        # small problems kept as dense matrices
        {"name": "dense_helm3d_dl_12000_16rhs", "do": "dense", "nel": 10, "q": 4, "nrhs": 16, "k": 2 * math.pi},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    do = rng.choice(["matvec", "matvec", "matvec", "solve", "build", "potential", "pullback", "batch", "dense"])
    k = round(rng.uniform(1.0, 12.0), 3)
    if do == "matvec":
        pde, dim = rng.choice(["laplace", "helmholtz"]), rng.choice([2, 3])
        kinds = [t[2] for t in PAIR_FLOPS if t[:2] == (pde, dim)]
        c = {"do": do, "pde": pde, "dim": dim, "kind": rng.choice(kinds),
             "prec": rng.choice(["fp64", "fp64", "mixed"]), "nrhs": rng.choice([1, 1, 1, 1, 4, 16, 5])}
        if dim == 2:
            c.update(nel=_log_int(rng, 60, 4000), q=rng.choice([5, 7, 9, 11]))
        else:
            c.update(nel=_log_int(rng, 3, 18 if c["nrhs"] > 1 else 26), q=rng.choice([2, 4, 5]))
        if pde == "helmholtz":
            c["k"] = k * (4 if dim == 2 else 1)
        return c
    if do in ("solve", "build"):
        dim = rng.choice([2, 3])
        if dim == 2:
            nel, q = _log_int(rng, 60, 1200 if do == "solve" else 3000), rng.choice([5, 9, 11])
        else:
            nel, q = _log_int(rng, 3, 7 if do == "solve" else 16), rng.choice([2, 4])
        return {"do": do, "pde": "helmholtz", "dim": dim, "nel": nel, "q": q, "k": k}
    if do == "potential":
        dim = rng.choice([2, 3])
        return {"do": do, "pde": rng.choice(["laplace", "helmholtz"]), "dim": dim,
                "nel": _log_int(rng, 60, 500) if dim == 2 else _log_int(rng, 3, 12), "q": 9 if dim == 2 else 4,
                "m": _log_int(rng, 500, 40000), "k": k}
    if do == "pullback":
        dim = rng.choice([2, 3])
        return {"do": do, "dim": dim, "nel": _log_int(rng, 60, 1200) if dim == 2 else _log_int(rng, 3, 10),
                "q": rng.choice([5, 9]) if dim == 2 else rng.choice([2, 4]), "k": k}
    if do == "batch":
        return {"do": do, "nprob": _log_int(rng, 3, 48), "lo": 50, "hi": _log_int(rng, 100, 1100),
                "q": rng.choice([7, 9]), "prec": rng.choice(["fp64", "mixed"])}
    return {"do": do, "nel": _log_int(rng, 3, 10), "q": rng.choice([2, 4]), "nrhs": rng.choice([1, 3, 8, 16, 32]),
            "k": k}


# ------------------------------------------------------------------- inputs
def _quad(dim, nel, q):
    """The ellipse or the sphere that the case is posed on."""
    return inti.ellipse_quadrature(1.0, 0.6, nel, qorder=q) if dim == 2 else inti.sphere_quadrature(nel, qorder=q)


def _nodes(case):
    if case["dim"] == 2:
        return case["nel"] * ((case["q"] + 2) // 2)
    return 20 * case["nel"] ** 2 * {2: 3, 4: 6, 5: 10}[case["q"]]


def _waves(rng, X, nrhs, cplx, k):
    """Smooth seeded densities (nrhs, n): two plane waves each."""
    out = np.empty((nrhs, X.shape[1]), dtype=np.complex128)
    for r in range(nrhs):
        s = 0
        for _ in range(2):
            d = rng.normal(size=X.shape[0])
            d /= np.linalg.norm(d)
            s = s + complex(rng.normal(), rng.normal()) * np.exp(1j * k * (d @ X))
        out[r] = s
    return out if cplx else np.ascontiguousarray(out.real)


def _batch_inputs(case, seed):
    rng = np.random.default_rng(seed)
    P = case["nprob"]
    ne = np.exp(np.linspace(math.log(case["lo"]), math.log(case["hi"]), P)).astype(int) | 1
    quads = [inti.ellipse_quadrature(rng.uniform(1, 3), rng.uniform(0.3, 1), int(e), qorder=case["q"]) for e in ne]
    ks = rng.uniform(1, 40, P)
    X = np.concatenate([_waves(rng, Q.coords, 16, True, 3.0) for Q in quads], axis=1)
    return quads, ks, X


def _targets(case, seed, rng):
    """Points outside the obstacle: a shell (2D, 3D) between 1.5 and 4 radii."""
    d = rng.normal(size=(case["dim"], case["m"]))
    d /= np.linalg.norm(d, axis=0)
    return np.ascontiguousarray(d * rng.uniform(1.5, 4.0, size=case["m"]))


def _op(case):
    if case.get("pde", "helmholtz") == "laplace":
        return inti.Laplace(dim=case["dim"])
    return inti.Helmholtz(k=case["k"], dim=case["dim"])


KERNELS = {"SL": inti.SingleLayerKernel, "DL": inti.DoubleLayerKernel, "HS": inti.HyperSingularKernel}


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def prepare(case, seed):
    do = case["do"]
    one, zero = (C.c_double * 2)(1.0, 0.0), (C.c_double * 2)(0.0, 0.0)
    if do == "batch":
        quads, ks, X = _batch_inputs(case, seed)
        B = inti.BatchOperator([inti.DoubleLayerKernel(inti.Helmholtz(k=float(k), dim=2)) for k in ks], quads,
                               precision=case["prec"])
        for p, (dS, dD) in enumerate(B.bdim_correction()):
            B.attach(p, dD)
        B.set_identity(0.5)
        x = torch.from_numpy(X).to(DEV)
        return {"do": do, "B": B, "x": x, "y": torch.empty_like(x), "one": one, "zero": zero}
    rng = np.random.default_rng(seed)
    case = dict(case, dim=case.get("dim", 3))
    Q = _quad(case["dim"], case["nel"], case["q"])
    n, k = len(Q), case.get("k", 0.0)
    op = _op(case)
    cplx = isinstance(op, inti.Helmholtz)
    if do == "matvec":
        x = torch.from_numpy(_waves(rng, Q.coords, case["nrhs"], cplx, 3.0)).to(DEV)
        if case["kind"] == "CF":
            A = inti.combined_field(op=op, quad=Q, c_single=-1j * k, c_double=1.0, precision=case["prec"])[0].iop
        else:
            S, D = inti.single_double_layer(op=op, target=Q, source=Q, compression={"method": "gpu"},
                                            correction={"method": "dim"}, derivative=case["kind"] == "HS",
                                            precision=case["prec"])
            A = (S if case["kind"] == "SL" else D).iop
        return {"do": do, "A": A, "x": x, "y": torch.empty_like(x), "n": n, "nrhs": case["nrhs"], "one": one,
                "zero": zero}
    if do == "dense":
        D = inti.IntegralOperator(inti.DoubleLayerKernel(op), Q, Q)
        S = inti.IntegralOperator(inti.SingleLayerKernel(op), Q, Q)
        _, dD = inti.bdim_correction(op, Q, Q, S, D, green_multiplier=np.full(n, -0.5))
        x = torch.from_numpy(_waves(rng, Q.coords, case["nrhs"], True, 3.0)).to(DEV)
        return {"do": do, "M": inti.DenseOperator(D, corrections=[(dD, 1.0)]), "x": x, "y": torch.empty_like(x),
                "n": n, "nrhs": case["nrhs"], "one": one, "zero": zero}
    sigma = _waves(rng, Q.coords, 1, cplx, 3.0)[0]
    if do == "solve":
        L = inti.combined_field(op=op, quad=Q, c_single=-1j * k, c_double=1.0, c_identity=0.5)[0]
        return {"do": do, "L": L, "b": sigma}
    if do == "build":
        Q.device(inti.default_context())
        return {"do": do, "op": op, "Q": Q, "k": k, "x": sigma}
    if do == "potential":
        Q.device(inti.default_context())
        S, D = inti.single_double_layer_potential(op=op, source=Q)
        return {"do": do, "S": S, "D": D, "x": sigma, "X": _targets(case, seed, rng)}
    if do == "pullback":
        A = inti.IntegralOperator(inti.CombinedFieldKernel(op, -1j * k, 1.0, "SD"), Q, Q)
        ubar = _waves(rng, Q.coords, 1, True, 2.0)[0]
        A.handle
        return {"do": do, "A": A, "x": sigma, "u": ubar}
    raise ValueError(do)


def run(state):
    do = state["do"]
    if do == "matvec":
        A, n = state["A"], state["n"]
        A.ctx.check(A.ctx.lib.inti_op_apply_device(A.handle, state["nrhs"], _ptr(state["x"]), n, _ptr(state["y"]), n,
                                                   state["one"], state["zero"]))
        return state["y"]
    if do == "solve":
        x, info = inti.gmres(state["L"], state["b"], restart=60, maxiter=120, rtol=1e-11)
        return x
    if do == "build":
        L, _ = inti.combined_field(op=state["op"], quad=state["Q"], c_single=-1j * state["k"], c_double=1.0)
        return L @ state["x"]
    if do == "potential":
        return [state["S"][state["x"]](state["X"]), state["D"][state["x"]](state["X"])]
    if do == "pullback":
        return state["A"].pullback(state["u"], state["x"], dcoefs=(-1j, 0.0),
                                   wrt=("sigma", "nodes", "source_normals", "source_weights", "k"))
    if do == "batch":
        B = state["B"]
        B.ctx.check(B.ctx.lib.inti_batch_apply_device(B.handle, 16, _ptr(state["x"]), B.ntot, _ptr(state["y"]),
                                                      B.ntot, state["one"], state["zero"]))
        return state["y"]
    M, n = state["M"], state["n"]
    M.ctx.check(M.ctx.lib.inti_dense_gemm(M.ctx.handle, 1, n, n, state["nrhs"], M.device_pointer, n, _ptr(state["x"]),
                                          n, _ptr(state["y"]), n, state["one"], state["zero"]))
    return state["y"]


def work(case):
    do = case["do"]
    if do == "batch":
        ne = np.exp(np.linspace(math.log(case["lo"]), math.log(case["hi"]), case["nprob"])).astype(int) | 1
        n = ne * ((case["q"] + 2) // 2)
        return {"bytes": float(n.sum()) * (40 + 2 * 16 * 16 + 6 * 20),
                "flops": float((n.astype(float) ** 2).sum()) * (60 + 16 * 8)}
    case = dict(case, dim=case.get("dim", 3))
    pde, dim, n = case.get("pde", "helmholtz"), case["dim"], float(_nodes(case))
    cw = 16 if pde == "helmholtz" else 8
    geo = (2 * dim + 1) * 8
    if do == "matvec":
        r, nq = case["nrhs"], (case["q"] + 2) // 2 if dim == 2 else {2: 3, 4: 6, 5: 10}[case["q"]]
        per = PAIR_FLOPS[(pde, dim, case["kind"])] + (r - 1) * (8 if cw == 16 else 2)
        return {"bytes": n * (geo + 2 * cw * r + nq * (cw + 4)), "flops": n * n * per}
    if do == "solve":  # about twenty products of the iteration
        return {"bytes": n * geo + 20 * 21 * 2 * cw * n, "flops": 20 * n * n * PAIR_FLOPS[(pde, dim, "CF")]}
    if do == "build":  # two kernels against the monopole columns
        nq = (case["q"] + 2) // 2 if dim == 2 else {2: 3, 4: 6, 5: 10}[case["q"]]
        return {"bytes": n * (geo + 2 * cw + nq * 2 * (cw + 4)),
                "flops": n * n * (PAIR_FLOPS[(pde, dim, "DL")] + 16 * 3 * nq + 36)}
    if do == "potential":
        m = float(case["m"])
        return {"bytes": n * (geo + 2 * cw) + m * (dim * 8 + 2 * cw),
                "flops": m * n * (PAIR_FLOPS[(pde, dim, "SL")] + PAIR_FLOPS[(pde, dim, "DL")])}
    if do == "pullback":
        return {"bytes": n * (geo + 2 * 16 + (2 * dim + 1) * 8 + 16), "flops": 3 * n * n * PAIR_FLOPS[(pde, dim, "CF")]}
    return {"bytes": 16 * n * n + 32 * n * case["nrhs"], "flops": 8 * n * n * case["nrhs"]}


# -------------------------------------------------- the same in plain torch
def _hankel(z):
    """H0(z), H1(z) of the first kind, z > 0: ascending series below 2.5,
    above it Poisson's integral sqrt(2/(pi z)) e^{i(z - nu pi/2 - pi/4)} /
    Gamma(nu + 1/2) int_0^inf e^{-t} t^(nu - 1/2) (1 + it/(2z))^(nu - 1/2) dt
    with t = v^2 by the trapezoidal rule (step 1/4, exponentially convergent)."""
    zs, zl = z.clamp(max=2.5), z.clamp(min=2.5)
    u = -0.25 * zs * zs
    t, harm = torch.ones_like(u), 0.0
    j0, j1, y0, y1 = torch.zeros_like(u), torch.zeros_like(u), torch.zeros_like(u), torch.zeros_like(u)
    for m in range(18):  # t = u^m / m!^2, harm = 1 + 1/2 + ... + 1/m
        j0 += t
        j1 += t / (m + 1)
        y0 -= harm * t
        y1 += (2 * harm + 1 / (m + 1)) * t / (m + 1)
        harm += 1 / (m + 1)
        t = t * u / ((m + 1) ** 2)
    lg = torch.log(zs / 2) + 0.57721566490153286061
    j1 = 0.5 * zs * j1
    y0 = (2 / math.pi) * (lg * j0 + y0)
    y1 = (2 / math.pi) * (lg * j1 - 1 / zs) - zs / (2 * math.pi) * y1
    i0 = torch.full_like(zl, 0.125).to(torch.complex128)
    i1 = torch.zeros_like(i0)
    for q in range(1, 27):
        v2 = (0.25 * q) ** 2
        root = torch.sqrt(1 + (0.5j * v2) / zl)
        i0 += 0.25 * math.exp(-v2) / root
        i1 += 0.25 * math.exp(-v2) * v2 * root
    e = torch.sqrt(2 / (math.pi * zl)) * torch.exp(1j * (zl - math.pi / 4)) * (2 / math.sqrt(math.pi))
    low = z < 2.5
    return torch.where(low, torch.complex(j0, y0), e * i0), torch.where(low, torch.complex(j1, y1), -2j * e * i1)


def _pairs(pde, dim, k, X, NX, Y, NY, want, grad=False):
    """Kernel values K(X_i, Y_j) (rows, columns), zero where the points are
    the same; want among G, DL (d/dn_y), ADL (d/dn_x), HS (d2/dn_x dn_y)."""
    r = [X[d][:, None] - Y[d][None, :] for d in range(dim)]
    d2 = sum(t * t for t in r)
    same = d2 <= 1e-28
    d = torch.sqrt(torch.where(same, torch.ones_like(d2), d2))
    out = {}
    dot = lambda N, rows: sum(r[c] * (N[c][:, None] if rows else N[c][None, :]) for c in range(dim))  # noqa: E731
    if pde == "laplace":
        if dim == 2:
            g, g1, g2 = -torch.log(d) / (2 * math.pi), -1 / (2 * math.pi * d), 1 / (2 * math.pi * d * d)
        else:
            g, g1, g2 = 1 / (4 * math.pi * d), -1 / (4 * math.pi * d ** 2), 2 / (4 * math.pi * d ** 3)
    elif dim == 3:
        g = torch.exp(1j * k * d) / (4 * math.pi * d)
        a = 1j * k - 1 / d
        g1, g2 = g * a, g * (a * a + 1 / d ** 2)
    else:
        z = k * d
        h0, h1 = _hankel(z)
        g, g1, g2 = 0.25j * h0, -0.25j * k * h1, -0.25j * k * k * (h0 - h1 / z)
    keep = (~same).to(torch.float64)
    if "G" in want:
        out["G"] = g * keep
    if "DL" in want:
        out["DL"] = -g1 * dot(NY, False) / d * keep
    if "ADL" in want:
        out["ADL"] = g1 * dot(NX, True) / d * keep
    if "HS" in want:
        nn = sum(NX[c][:, None] * NY[c][None, :] for c in range(dim))
        ab = dot(NX, True) * dot(NY, False) / d ** 2
        out["HS"] = (-(g2 - g1 / d) * ab - g1 / d * nn) * keep
    return out


def _geo(Q):
    return (torch.from_numpy(Q.coords).to(DEV), torch.from_numpy(Q.normals).to(DEV), torch.from_numpy(Q.weights).to(DEV))


def _monopoles(Q, ns):
    lo, hi = Q.coords.min(axis=1), Q.coords.max(axis=1)
    c, R = (lo + hi) / 2, 1.5 * np.linalg.norm(hi - lo) / 2
    if Q.dim == 2:
        t = 2 * np.pi * np.arange(ns) / ns
        z = np.stack([np.cos(t), np.sin(t)])
    else:
        i = np.arange(1, ns + 1)
        y = 1 - 2 * (i - 1) / (ns - 1)
        t = math.pi * (3 - math.sqrt(5.0)) * i
        z = np.stack([np.cos(t) * np.sqrt(1 - y * y), y, np.sin(t) * np.sqrt(1 - y * y)])
    return torch.from_numpy(c[:, None] + R * z).to(DEV)


def _corrected(pde, Q, k, c0, c1, X, deriv=False, dense=False):
    """(c0 S + c1 D) X with the density-interpolation correction of every
    element's own nodes ((ADL, HS) with deriv), X (n, nrhs) on the device; the
    matrix itself with dense."""
    dim, (xy, nrm, w) = Q.dim, _geo(Q)
    n, nq, ns = len(Q), Q.nq, 3 * Q.nq
    z = _monopoles(Q, ns)
    b = _pairs(pde, dim, k, xy, nrm, z, z, ("G", "ADL"))
    B0, B1 = b["G"], b["ADL"]
    theta = -0.5 * (B1 if deriv else B0)
    sname, dname = ("ADL", "HS") if deriv else ("G", "DL")
    y = [] if not dense else torch.empty(n, n, dtype=B0.dtype, device=DEV)
    step = max(1, (1 << 24) // n)
    for i in range(0, n, step):
        K = _pairs(pde, dim, k, xy[:, i:i + step], nrm[:, i:i + step], xy, nrm, (sname, dname))
        S, D = K[sname] * w, K[dname] * w
        theta[i:i + step] += S @ B1 - D @ B0
        A = c0 * S + c1 * D
        if dense:
            y[i:i + step] = A
        else:
            y.append(A.to(X.dtype) @ X)
    tags = Q.qtags.T  # (ne, nq)
    M = torch.cat([B0[tags], B1[tags]], dim=1).cpu().numpy()            # (ne, 2 nq, ns)
    q, r = np.linalg.qr(np.swapaxes(M, 1, 2))                           # ns x 2 nq
    rhs = np.swapaxes(theta[tags].cpu().numpy(), 1, 2)                  # (ne, ns, targets)
    W = np.linalg.solve(r, np.swapaxes(q.conj(), 1, 2) @ rhs)           # (ne, 2 nq, targets)
    W = torch.from_numpy(c1 * W[:, :nq] - c0 * W[:, nq:]).to(DEV).to(B0.dtype if dense else X.dtype)
    t = torch.from_numpy(tags).to(DEV)
    if dense:
        y[t[:, None, :], t[:, :, None]] += W
        return y
    y = torch.cat(y)
    y[t.reshape(-1)] += (W.transpose(1, 2) @ X[t]).reshape(-1, X.shape[1])
    return y


def exact(case, seed):
    do = case["do"]
    if do == "batch":
        quads, ks, X = _batch_inputs(case, seed)
        out, o = [], 0
        for Q, k in zip(quads, ks):
            x = torch.from_numpy(X[:, o:o + len(Q)]).to(DEV).T.contiguous()
            out.append((_corrected("helmholtz", Q, float(k), 0.0, 1.0, x) + 0.5 * x).T)
            o += len(Q)
        return torch.cat(out, dim=1)
    rng = np.random.default_rng(seed)
    case = dict(case, dim=case.get("dim", 3))
    Q = _quad(case["dim"], case["nel"], case["q"])
    k, pde = case.get("k", 0.0), case.get("pde", "helmholtz")
    cplx = pde == "helmholtz"
    if do in ("matvec", "dense"):
        x = torch.from_numpy(_waves(rng, Q.coords, case["nrhs"], cplx, 3.0)).to(DEV).T.contiguous()
        kind = case.get("kind", "DL")
        c0, c1 = {"SL": (1.0, 0.0), "DL": (0.0, 1.0), "HS": (0.0, 1.0), "CF": (-1j * k, 1.0)}[kind]
        return _corrected(pde, Q, k, c0, c1, x, deriv=kind == "HS").T.contiguous()
    sigma = _waves(rng, Q.coords, 1, cplx, 3.0)[0]
    x = torch.from_numpy(sigma).to(DEV)[:, None]
    if do == "solve":
        A = _corrected(pde, Q, k, -1j * k, 1.0, x, dense=True)
        A.diagonal().add_(0.5)
        return torch.linalg.solve(A, x)[:, 0].cpu().numpy()
    if do == "build":
        return _corrected(pde, Q, k, -1j * k, 1.0, x)[:, 0].cpu().numpy()
    xy, nrm, w = _geo(Q)
    if do == "potential":
        X = torch.from_numpy(_targets(case, seed, rng)).to(DEV)
        S, D = [], []
        step = max(1, (1 << 24) // len(Q))
        for i in range(0, case["m"], step):
            K = _pairs(pde, case["dim"], k, X[:, i:i + step], None, xy, nrm, ("G", "DL"))
            S.append((K["G"] * w) @ x)
            D.append((K["DL"] * w) @ x)
        return [torch.cat(S)[:, 0].cpu().numpy(), torch.cat(D)[:, 0].cpu().numpy()]
    # pullback: reverse mode of Re <ubar, y>, row blocks at a time (in 2D
    # torch does not differentiate the Bessel functions)
    if case["dim"] == 2:
        return None
    u = torch.from_numpy(_waves(rng, Q.coords, 1, True, 2.0)[0]).to(DEV)
    v = {"sigma": x[:, 0], "nodes": xy, "source_normals": nrm, "source_weights": w,
         "k": torch.tensor(float(k), dtype=torch.float64, device=DEV)}
    v = {a: t.clone().requires_grad_(True) for a, t in v.items()}
    n = len(Q)
    step = max(1, (1 << 21) // n)
    for i in range(0, n, step):
        K = _pairs(pde, 3, v["k"], v["nodes"][:, i:i + step], None, v["nodes"], v["source_normals"], ("G", "DL"))
        y = (-1j * v["k"] * K["G"] + K["DL"]) @ (v["source_weights"] * v["sigma"])
        (u[i:i + step].conj() * y).real.sum().backward()
    return {a: np.float64(t.grad.item()) if a == "k" else t.grad.cpu().numpy() for a, t in v.items()}
