"""The FP64 sin/cos of a phase in revolutions used by the device kernels
(devmath.hpp: sincos_rev64): its coefficient tables, read from the header,
and its reduction q = rint(4u), f = u - q/4, evaluated here in numpy with
the same Horner order, against 50-digit mpmath sin(2 pi u), cos(2 pi u) of
the same double u. A wrong coefficient digit, degree or quadrant rule
breaks the 4-ulp bound."""
import os
import re

import mpmath as mp
import numpy as np

HDR = os.path.join(os.path.dirname(__file__), "..", "inti.jl_amd", "csrc", "devmath.hpp")


def _table(name):
    text = open(HDR).read()
    body = re.search(name + r"\[\d+\]\s*=\s*\{([^}]*)\}", text).group(1)
    return [float.fromhex(t.strip()) for t in body.split(",") if t.strip()]


def _sincos_rev(u):
    sinc, cosc = _table("kSinRev"), _table("kCosRev")
    q = np.rint(4.0 * u)
    f = u - 0.25 * q
    z = f * f
    ps = np.full_like(u, sinc[-1])
    for c in sinc[-2::-1]:
        ps = ps * z + c
    pc = np.full_like(u, cosc[-1])
    for c in cosc[-2::-1]:
        pc = pc * z + c
    S, C = f * ps, pc
    qi = q.astype(np.int64) & 3
    s0 = np.where(qi & 1, C, S)
    c0 = np.where(qi & 1, S, C)
    s = np.where(qi & 2, -s0, s0)
    c = np.where((qi ^ (qi >> 1)) & 1, -c0, c0)
    return s, c


def test_tables_are_the_taylor_coefficients():
    mp.mp.dps = 50
    tp = 2 * mp.pi
    sinc, cosc = _table("kSinRev"), _table("kCosRev")
    assert len(sinc) == 8 and len(cosc) == 9
    for k, v in enumerate(sinc):
        assert v == float((-1) ** k * tp ** (2 * k + 1) / mp.factorial(2 * k + 1))
    for k, v in enumerate(cosc):
        assert v == float((-1) ** k * tp ** (2 * k) / mp.factorial(2 * k))


def test_sincos_rev_against_mpmath():
    mp.mp.dps = 40
    rng = np.random.default_rng(5)
    u = np.concatenate([rng.uniform(-1, 1, 3000), rng.uniform(-300, 300, 3000),
                        np.arange(-8, 9) / 8.0, np.arange(-8, 9) / 8.0 + 1e-12,
                        np.arange(-8, 9) / 8.0 - 1e-12, [0.0, 1e-300, -1e-300, 1e6 + 0.3]])
    s, c = _sincos_rev(u)
    es = max(abs(float(mp.sin(2 * mp.pi * mp.mpf(x))) - y) for x, y in zip(u, s))
    ec = max(abs(float(mp.cos(2 * mp.pi * mp.mpf(x))) - y) for x, y in zip(u, c))
    assert es <= 4.5e-16 and ec <= 4.5e-16, (es, ec)


def _log64(x, off):
    """devmath.hpp's log64 with every FMA rounded once (exact rationals), the
    hardware reciprocal estimate off by the relative error `off`."""
    from fractions import Fraction as F

    def fma(a, b, c):
        return float(F(a) * F(b) + F(c))

    def rcp64(d):
        r = float(F(1) / F(d) * (1 + F(off)))
        e = fma(-d, r, 1.0)
        return fma(r, fma(e, e, e), r)

    hi, lo = (float.fromhex(re.search(n + r" = (\S+?)[,;]", open(HDR).read()).group(1)) for n in ("kLn2Hi", "kLn2Lo"))
    m, e = np.frexp(x)
    m, k = float(m), float(e)
    if m < float.fromhex("0x1.6a09e667f3bcdp-1"):
        m, k = m + m, k - 1.0
    f = m - 1.0
    d = 2.0 + f
    dl = f - (d - 2.0)
    r = rcp64(d)
    s = f * r
    sl = fma(-s, dl, fma(-s, d, f)) * r
    z = s * s
    p = 0.0
    for c in _table("kLogR")[::-1]:
        p = fma(p, z, c)
    a = k * hi
    h = fma(2.0, s, a)
    t = fma(2.0, sl, fma(k, lo, fma(2.0, s, a - h)))
    return h + fma(s * z, p, t)


def test_log64_against_mpmath():
    """Within 0.54 ulp (the bound its comment states) for estimates of the
    reciprocal up to 2^-24 off either way: random mantissas in every binade of
    distances squared, and both sides of the reduction's edges."""
    mp.mp.dps = 40
    rng = np.random.default_rng(9)
    x = np.concatenate([2.0 ** rng.uniform(-1, 1, 1200), 2.0 ** rng.uniform(-90, 60, 600),
                        [c * (1 + t) for c in (0.5, 0.5 ** 0.5, 1.0, 2 ** 0.5, 2.0) for t in (-1e-3, -1e-9, -2 ** -52, 0, 2 ** -52, 1e-9, 1e-3)]])
    worst = 0.0
    for i, v in enumerate(map(float, x)):
        y, ref = _log64(v, (-1) ** i * 2.0 ** -24), mp.log(mp.mpf(v))
        if ref == 0:
            assert y == 0.0
            continue
        worst = max(worst, abs(float((mp.mpf(y) - ref) / mp.mpf(float(np.spacing(abs(float(ref))))))))
    assert worst <= 0.54, worst
