"""The polynomial of the Ewald pair (csrc/ewald_pair.hpp): its coefficients
derived again, and its error.

(1 + 2 x) exp(x^2) erfc(x), x >= 0, is smooth in t = (x - K) / (x + K) (the
variable and factor of Shepherd and Laframboise, Math. Comp. 36, 249 (1981)).
Its Chebyshev series in t, K = 3.75, cut after the 22nd term and written in
powers of t, gives the coefficients."""
import os
import re

import numpy as np
import pytest

mp = pytest.importorskip("mpmath").mp

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
K, DEG = 3.75, 22


def header():
    with open(os.path.join(ROOT, "atomistica_amd", "csrc", "ewald_pair.hpp")) as f:
        body = re.search(r"ewp_c\[EWP_DEG \+ 1\] = \{(.*?)\}", f.read(), re.S).group(1)
    return [float(v) for v in body.split(",")]


def function(x):
    if x < 60:
        return (1 + 2 * x) * mp.exp(x * x) * mp.erfc(x)
    # asymptotic series; 12 terms are below 1e-30 here
    s, term = mp.mpf(1), mp.mpf(1)
    for k in range(1, 13):
        term *= -(2 * k - 1) / (2 * x * x)
        s += term
    return (1 + 2 * x) * s / (x * mp.sqrt(mp.pi))


def test_coefficients_are_those_of_the_series():
    mp.dps = 50
    n = 96
    theta = [mp.pi * (i + mp.mpf(1) / 2) / n for i in range(n)]
    y = [function(K * (1 + mp.cos(a)) / (1 - mp.cos(a))) for a in theta]
    cheb = [2 * sum(v * mp.cos(k * a) for v, a in zip(y, theta)) / n for k in range(DEG + 1)]
    cheb[0] /= 2
    power = [mp.mpf(0)] * (DEG + 1)
    t0, t1 = [mp.mpf(1)], [mp.mpf(0), mp.mpf(1)]
    for k in range(DEG + 1):
        if k >= 2:
            t0, t1 = t1, [a - b for a, b in zip([mp.mpf(0)] + [2 * v for v in t1], t0 + [mp.mpf(0)] * 2)]
        for i, v in enumerate(t1 if k else t0):
            power[i] += cheb[k] * v
    got = header()
    assert len(got) == DEG + 1
    # Powers of t amplify the last digits of the series' coefficients by up to
    # 2^21: 1e-24 (six terms of the asymptotic series at x = 60) becomes 2e-17.
    # |t| <= 1 and the function is at least 1, so that is a fifth of its rounding.
    for a, b in zip(got, power):
        assert abs(a - b) <= 2.0 ** -53 * abs(float(b)) + 4e-17


def test_error_is_below_the_stated_bound():
    """The polynomial in exact arithmetic (the rounding of its evaluation comes
    on top): below 5.2e-16 of the value, 1.2e-16 rms."""
    mp.dps = 50
    c = [mp.mpf(v) for v in header()]
    rng = np.random.default_rng(0)
    x = np.concatenate([[0.0], rng.uniform(0, 7, 1500), 10 ** rng.uniform(-4, 1.7, 700)])
    err = []
    for v in x:
        v = mp.mpf(float(v))
        t = (v - K) / (v + K)
        p = mp.mpf(0)
        for a in reversed(c):
            p = p * t + a
        f = function(v)
        err.append(float((p - f) / f))
    print("largest %.2e rms %.2e" % (np.abs(err).max(), np.sqrt(np.mean(np.square(err)))))
    assert np.abs(err).max() < 5.2e-16
    assert np.sqrt(np.mean(np.square(err))) < 1.2e-16
