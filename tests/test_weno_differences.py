"""The device's WENO combination (enl_device.h weno_pair5, weno_pair3): the
reference's pf1 + mf1 - pf2 - mf2 (rhs_hybrid_high_llf.m4:286-354,
rhs_hybrid_low_llf.m4:349-399) from the differences of the split fluxes.

A numpy model of its arithmetic (without fused multiply-adds) and the
reference's expressions, both in float64, against the reference's expressions
in extended precision: the model's RMS and largest errors must not exceed the
reference's own.  Stratified, smooth, shocked, constant and random stencils.
"""
import numpy as np
import pytest

L = np.longdouble
pytestmark = pytest.mark.skipif(np.finfo(L).eps >= np.finfo(np.float64).eps, reason="needs extended long double")
C13_12, EPS, C1_6 = (L(np.float32(v)) for v in (13.0 / 12.0, 10.0e-6, 1.0 / 6.0))
W01, W06, W03 = (L(np.float32(v)) for v in (0.1, 0.6, 0.3))
C1_3, C2_3 = (L(np.float32(a) / np.float32(3)) for a in (1.0, 2.0))


def parts(a, b, c, d, e, T, plus):
    b0 = T(C13_12) * (c - 2 * d + e) ** 2 + T(0.25) * (3 * c - 4 * d + e) ** 2
    b1 = T(C13_12) * (b - 2 * c + d) ** 2 + T(0.25) * (b - d) ** 2
    b2 = T(C13_12) * (a - 2 * b + c) ** 2 + T(0.25) * (a - 4 * b + 3 * c) ** 2
    if plus:  # wenop
        cs = (T(W03), T(W06), T(W01))
        f = (T(C1_6) * (2 * c + 5 * d - e), T(C1_6) * (-b + 5 * c + 2 * d), T(C1_6) * (2 * a - 7 * b + 11 * c))
    else:  # wenom
        cs = (T(W01), T(W06), T(W03))
        f = (T(C1_6) * (11 * c - 7 * d + 2 * e), T(C1_6) * (2 * b + 5 * c - d), T(C1_6) * (-a + 5 * b + 2 * c))
    D = [(T(EPS) + x) ** 2 for x in (b0, b1, b2)]
    return cs, D, f


def reference(cs, D, f):
    z = [c / d for c, d in zip(cs, D)]
    s = z[0] + z[1] + z[2]
    return (z[0] / s) * f[0] + (z[1] / s) * f[1] + (z[2] / s) * f[2]


def divergence(form, T, fp, fm):
    """p1 + m1 - p2 - m2 at every cell (rhs_hybrid_high_llf.m4:286-354)."""
    out = []
    for i in range(3, len(fp) - 3):
        p1 = form(*parts(*fp[i - 3:i + 2], T, True))
        m1 = form(*parts(*fm[i - 2:i + 3], T, False))
        p2 = form(*parts(*fp[i - 2:i + 3], T, True))
        m2 = form(*parts(*fm[i - 1:i + 4], T, False))
        out.append(p1 + m1 - p2 - m2)
    return np.array(out)


def pair5(e, T):
    e0, e1, e2, e3, e4 = e
    kC, kE, r2 = T(4) * T(C13_12), T(16) * T(EPS), T(W01) / T(W06)
    c1, c2, c3, c4 = e1 - e0, e2 - e1, e3 - e2, e4 - e3
    t1, t2, t3 = c2 - c1, c3 - c2, c4 - c3
    s1, s2, s3, s4 = (kC * c * c + kE for c in (c1, c2, c3, c4))
    quad = lambda l, s: (l * l + s) ** 2

    def frac(q0, q1, q2, ta, tb):
        return q1 * (4 * r2 * q0 * ta + tb * q2), q1 * (2 * r2 * q0 + q2) + 2 * (q0 * q2)

    n1, d1 = frac(quad(e3 - 3 * e2, s3), quad(e1 + e2, s2), quad(3 * e1 - e0, s1), t1, t2)
    n2, d2 = frac(quad(e4 - 3 * e3, s4), quad(e2 + e3, s3), quad(3 * e2 - e1, s2), t2, t3)
    return (n2 * d1 - n1 * d2) / (d1 * d2) + ((e1 - 5 * e2) - 2 * e3)


def pair3(e1, e2, e3, T):
    kE = T(4) * T(EPS)
    q1, q2, q3 = ((e * e + kE) ** 2 for e in (e1, e2, e3))
    n1, d1, n2, d2 = 2 * q1 * e2 + q2 * e1, 2 * q1 + q2, 2 * q2 * e3 + q3 * e2, 2 * q2 + q3
    return (n1 * d2 - n2 * d1) / (d1 * d2) - 2 * e2


def device(order, F, aW, T):
    """At every cell, from the flux F and alpha * w (the split fluxes are half
    their sum and difference)."""
    dF, dW = F[1:] - F[:-1], aW[1:] - aW[:-1]
    out = []
    for i in range(3, len(F) - 3):
        p, m = dF[i - 3:i + 3] + dW[i - 3:i + 3], dF[i - 3:i + 3] - dW[i - 3:i + 3]
        if order == 5:
            out.append((pair5(p[:5], T) + pair5(m[:0:-1], T)) * (T(0.5) * T(C1_6)))
        else:
            out.append((pair3(*p[1:4], T) + pair3(*m[4:1:-1], T)) * T(0.25))
    return np.array(out)


def reference3(F, aW, T):
    def rec(a, b, c):  # wenop3; wenom3 is its mirror image
        z0, z1 = T(C2_3) / (T(EPS) + (c - b) ** 2) ** 2, T(C1_3) / (T(EPS) + (b - a) ** 2) ** 2
        s = z0 + z1
        return (z0 / s) * (T(0.5) * (b + c)) + (z1 / s) * (T(0.5) * (-a + 3 * b))

    fp, fm = T(0.5) * (F + aW), T(0.5) * (F - aW)
    return np.array([rec(*fp[i - 2:i + 1]) + rec(*fm[i + 1:i - 2:-1]) - rec(*fp[i - 1:i + 2]) - rec(*fm[i + 2:i - 1:-1])
                     for i in range(3, len(F) - 3)])


def fields():
    x = np.arange(400) / 400
    rng = np.random.default_rng(3)
    rho = 1.2 * np.exp(-x * 2000 / 8000)
    yield "stratified", 1e-3 * rho * np.sin(9 * x), 344.0 * rho * 294.0
    yield "smooth", 1e5 + 3e3 * np.sin(12 * x), 4e2 * np.cos(7 * x)
    yield "shock", np.where(x < 0.5, 1e5, 6e5) + 10 * x, np.where(x < 0.52, 4e2, 2e3)
    yield "random", rng.normal(size=400) * 1e2, rng.normal(size=400)
    yield "constant", np.full(400, 101325.0), np.full(400, 412.5)


@pytest.mark.parametrize("order", [5, 3])
@pytest.mark.parametrize("name,F,aW", list(fields()), ids=lambda v: v if isinstance(v, str) else "")
def test_no_less_exact_than_the_reference(order, name, F, aW):
    if order == 5:
        ref = lambda F, aW, T: divergence(reference, T, T(0.5) * (F + aW), T(0.5) * (F - aW))
    else:
        ref = reference3
    true = ref(F.astype(L), aW.astype(L), L)
    e_ref = np.abs(ref(F, aW, np.float64) - true)
    e_dev = np.abs(device(order, F, aW, np.float64) - true)
    rms = lambda e: float(np.sqrt(np.mean(e ** 2)))
    # the same expressions agree where both are exact
    assert np.abs(device(order, F.astype(L), aW.astype(L), L) - true).max() <= 1e-17 * max(np.abs(F).max(), np.abs(aW).max())
    assert rms(e_dev) <= rms(e_ref) and e_dev.max() <= e_ref.max(), (name, rms(e_dev), rms(e_ref))
