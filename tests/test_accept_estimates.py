"""The FP64 samplers' FP32 accept estimates and the inversion's division by a count
(csrc/tm_device.h): ptrs_estimate, gamma_estimate, div_k, restated in numpy FP32.

An estimate may only call a trial (+1 accept, -1 reject) where the FP64 test has the
same outcome; div_k must round t / k correctly.  No GPU needed."""
from fractions import Fraction

import numpy as np
import pytest
from scipy.special import gammaln

F = np.float32


def ptrs_estimate(z, kd, us, V):
    slam = np.sqrt(z)
    b = 0.931 + 2.53 * slam
    a = -0.059 + 0.02483 * b
    k, zf, dk = F(kd), F(z), (kd - z).astype(F)
    s = k + zf
    w = dk / s
    w2 = w * w
    near = np.abs(dk) < F(0.1) * s
    bd0 = np.where(near, dk * w + F(2) * k * w * w2 * (F(1 / 3) + w2 * (F(0.2) + w2 * (F(1 / 7) + w2 * F(1 / 9)))),
                   k * np.log(k / zf) - dk)
    r = F(1) / k
    rhs = -r * (F(1 / 12) - r * r * F(1 / 360)) - bd0 - F(0.5) * np.log(F(2 * np.pi) * k)
    usf, bf = F(us), F(b)
    inva = F(1.1239) + F(1.1328) / (bf - F(3.4))
    lhs = np.log(F(V) * inva / (F(a) / (usf * usf) + bf))
    m = F(1e-3) + F(1e-5) * (np.abs(lhs) + np.abs(rhs))
    ok = (kd >= 5) & (z < 1e9) & (near | (kd < 1000))
    return np.where(ok, np.where(lhs < rhs - m, 1, np.where(lhs > rhs + m, -1, 0)), 0)


@pytest.mark.parametrize("z", [12.0, 13.7, 40.0, 300.0, 1.6e3, 1.4e5, 2e7, 9.9e8])
def test_ptrs_estimate_agrees_with_the_logarithmic_test(z):
    rng = np.random.default_rng(int(z))
    n = 400_000
    U = (rng.integers(0, 2 ** 32, n) + 0.5) * 2.0 ** -32 - 0.5
    V = (rng.integers(0, 2 ** 32, n) + 0.5) * 2.0 ** -32
    us = 0.5 - np.abs(U)
    b = 0.931 + 2.53 * np.sqrt(z)
    a = -0.059 + 0.02483 * b
    kd = np.floor((2 * a / us + b) * U + z + 0.43)
    keep = (kd >= 0) & ~((us < 0.013) & (V > us))
    U, V, us, kd = U[keep], V[keep], us[keep], kd[keep]
    est = ptrs_estimate(np.full(kd.size, z), kd, us, V)
    lhs = np.log(V) + np.log(1.1239 + 1.1328 / (b - 3.4)) - np.log(a / us ** 2 + b)
    # the right side without cancellation: scipy's poisson log-pmf loses digits at large z
    lp = -z + kd * np.log(z) - gammaln(kd + 1) if z < 1e6 else None
    if lp is None:
        d = kd - z
        w = d / (kd + z)
        bd0 = d * w + 2 * kd * w * w * w * (1 / 3 + w * w / 5 + w ** 4 / 7)
        lp = -1 / (12 * kd) - bd0 - 0.5 * np.log(2 * np.pi * kd)
    exact = np.where(lhs <= lp, 1, -1)
    called = est != 0
    domain = (kd >= 5) & ((np.abs(kd - z) < 0.1 * (kd + z)) | (kd < 1000))   # where the estimate is offered at all
    assert called.mean() > domain.mean() - 0.02              # margin 1e-3 of a log-uniform scale: a few 1e-3
    assert np.array_equal(est[called], exact[called])
    # not vacuous: without its margin the estimate of a shifted test would disagree
    assert not np.array_equal(est[called], np.where(lhs[called] <= lp[called] - 0.1, 1, -1))


@pytest.mark.parametrize("d", [2 / 3, 0.8, 1.5, 4.0, 30.0, 455.0, 7e4, 1e9])
def test_gamma_estimate_agrees_with_the_logarithmic_test(d):
    rng = np.random.default_rng(3)
    n = 400_000
    x = rng.standard_normal(n) * rng.choice([1.0, 2.0], n)
    u = (rng.integers(0, 2 ** 32, n) + 0.5) * 2.0 ** -32
    c = 1 / np.sqrt(9 * d)
    y = c * x
    ok = y > -1
    x, u, y = x[ok], u[ok], y[ok]
    v = (1 + y) ** 3
    yf, df, vf = F(y), F(d), F(v)
    y2 = yf * yf
    ser = df * y2 * y2 * (F(-0.75) + yf * (F(0.6) + yf * (F(-0.5) + yf * (F(3 / 7) - F(0.375) * yf))))
    dirr = F(0.5) * F(x * x) + df * (F(1) - vf + np.log(vf))
    rhs = np.where(np.abs(yf) < F(0.1), ser, dirr)
    lhs = np.log(F(u))
    est = np.where(lhs < rhs - F(1e-3), 1, np.where(lhs > rhs + F(1e-3), -1, 0))
    q = 3 * d * (np.log1p(y) - y + y * y / 2 - y ** 3 / 3)
    small = np.abs(y) < 0.02
    q[small] = 3 * d * (-y[small] ** 4 / 4 + y[small] ** 5 / 5 - y[small] ** 6 / 6 + y[small] ** 7 / 7)
    exact = np.where(np.log(u) < q, 1, -1)
    called = est != 0
    assert called.mean() > 0.99
    assert np.array_equal(est[called], exact[called])


def _fma(a, b, c):
    return float(Fraction(a) * Fraction(b) + Fraction(c))   # rounded once


@pytest.mark.parametrize("lo", [1, 50, 150])
def test_division_by_a_count_rounds_correctly(lo):
    rng = np.random.default_rng(lo)
    for k in range(lo, lo + 50):
        inv = 1.0 / k
        for t in np.concatenate([rng.random(6), 10.0 ** rng.uniform(-60, 1, 6), [k * 0.1, np.nextafter(k, 0)]]):
            t = float(t)
            q = t * inv
            q = _fma(_fma(-q, float(k), t), inv, q)
            q = _fma(_fma(-q, float(k), t), inv, q)
            assert q == t / k
