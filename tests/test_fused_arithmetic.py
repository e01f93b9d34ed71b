"""Arithmetic that the kernels form with fused operations, restated with the C
library's fma (exact by IEEE 754) and checked on the CPU: the squared weight chain
behind the flags of Generate + Unweight (generate_unweight.hip, chain_q2 and
chain3_q2) against extended precision and its bound's rounding terms, and the
range's uniforms (hpsp_device.h, to_unit of minstd_rand) against the division."""
import ctypes
import ctypes.util

import numpy as np
import pytest

from test_chain_bound import EPS, THREE_BODY

libm = ctypes.CDLL(ctypes.util.find_library("m"))
libm.fma.restype = ctypes.c_double
libm.fma.argtypes = [ctypes.c_double] * 3
fma = np.vectorize(libm.fma, otypes=[np.float64])
L = np.longdouble


def exact_chain(mw, inv_mas, m):
    """The weight chain for given invariant masses, in extended precision."""
    w = L(mw)
    for s in range(len(m) - 1):
        a, b, c = inv_mas[s + 1].astype(L), L(m[s + 1]), inv_mas[s].astype(L)
        w = w * np.sqrt((a - b - c) * (a + b + c) * (a - b + c) * (a + b - c)) / (2 * a)
    return w


def rounding_bound(inv_mas, m, floor):
    """B with K = 0: floor + 4 eps (ka + kc) of each step; where it is defined."""
    B = np.full(inv_mas[0].shape, floor)
    ok = np.ones(B.shape, dtype=bool)
    for s in range(len(m) - 1):
        a, b, c = inv_mas[s + 1], m[s + 1], inv_mas[s]
        spc, smc = b + c, b - c
        d1, d2 = (a - spc) * (a + spc), (a - smc) * (a + smc)
        ok &= np.minimum(d1, d2) > 0
        B = B + 4 * EPS * ((a * a + c * np.abs(smc)) / d2 + (a * a + c * spc) / d1 + 1)
    return B, ok


def worst(q, exact, B, sel):
    assert sel.any()
    rel = np.abs((q[sel].astype(L) - exact[sel]) / exact[sel])
    return float((rel / B[sel]).max())


@pytest.mark.parametrize("case", THREE_BODY, ids=[c[0] for c in THREE_BODY])
def test_three_body_chain(oracle, case):
    """chain3_q2: x0 and x1 from a^2 - s^2 with one fused operation each, the
    constants as the host rounds them, no test of q^2's range."""
    name, M, masses = case
    m = np.asarray(masses, dtype=np.float64)
    _, ecm, mw = oracle.params(M, m)
    rng = np.random.default_rng(5)
    # uniforms of the 32-bit words, the ends of [0, 1] among them
    v = np.concatenate([rng.integers(0, 2 ** 32, 1 << 14), [0, 1, 2, 9, 2 ** 31, 2 ** 32 - 2,
                                                            2 ** 32 - 1]]).astype(np.float64)
    s01 = (0.0 + m[0]) + m[1]
    A = 1.0 * ecm + (s01 + m[2])
    a0 = v * (ecm * 2.0 ** -32) + s01
    sp2, sm2, A2 = (m[1] + m[0]) ** 2, (m[1] - m[0]) ** 2, A * A
    x0 = fma(a0, a0, -sp2) * fma(a0, a0, -sm2)
    spc1, smc1 = m[2] + a0, m[2] - a0
    x1 = fma(-spc1, spc1, A2) * fma(-smc1, smc1, A2)
    inv_mas = [np.full_like(a0, m[0]), a0, np.full_like(a0, A)]
    with np.errstate(divide="ignore", invalid="ignore"):
        q2 = mw * mw / 16.0 / A2 * (x0 * x1) * (1.0 / (a0 * a0))
        q = np.sqrt(q2)
        exact = exact_chain(mw, inv_mas, m)
        B, ok = rounding_bound(inv_mas, m, 120 * EPS)
    # trusted where B is below 2^-10: there q^2 is positive and normal without a test
    sel = ok & (B < 2.0 ** -10)
    assert sel.mean() > 0.5, name
    assert np.all(q2[sel] >= 2.0 ** -1000) and np.all(np.isfinite(q2[sel]))
    # the mixed form's margin is 4 B, beside the weight's own rounding; 5 % of it
    assert worst(q, exact, B, sel) <= 0.2, name


@pytest.mark.parametrize("M,masses", [(3.0969, [0.1057, 0.1057]), (12.0, [0.5, 1.2, 0.8, 2.0, 0.3]),
                                      (10.0, [0.999] * 10), (100.0, [0.000511, 90.0, 0.000511, 1.0]),
                                      (20.0, [0.5] * 12)])
def test_chain(oracle, M, masses):
    """chain_q2: d1 and d2 from the rounded square of a and a fused operation."""
    m = np.asarray(masses, dtype=np.float64)
    N = len(m)
    _, ecm, mw = oracle.params(M, m)
    rng = np.random.default_rng(N)
    n = 1 << 12
    rno = np.vstack([np.zeros(n), np.sort(rng.integers(0, 2 ** 32, (N - 2, n)) * 2.0 ** -32, axis=0),
                     np.ones(n)])
    csum = np.cumsum(m)
    inv_mas = [rno[i] * ecm + csum[i] for i in range(N)]
    P, Q = np.ones(n), np.ones(n)
    with np.errstate(divide="ignore", invalid="ignore"):
        for s in range(N - 1):
            a, b, c = inv_mas[s + 1], m[s + 1], inv_mas[s]
            spc, smc, a2 = b + c, b - c, a * a
            P = P * (fma(-spc, spc, a2) * fma(-smc, smc, a2))
            Q = Q * a2
        q = np.sqrt(mw * mw * 4.0 ** (1 - N) * P * (1.0 / Q))
        exact = exact_chain(mw, inv_mas, m)
        B, ok = rounding_bound(inv_mas, m, 40 * N * EPS)
    sel = ok & (B < 2.0 ** -10)
    if sel.any():
        assert worst(q, exact, B, sel) <= 1.0, (M, masses)


def test_minstd_uniform_is_the_rounded_division():
    """x / 2147483646 through RN(1 / 2147483646) and one residual: both ends, the
    neighbourhoods of powers of two and 2^18 states of the engine."""
    div = 2147483646.0
    inv = 1.0 / div
    rng = np.random.default_rng(1)
    near = [2 ** k + d for k in range(31) for d in range(-3, 4)]
    x = np.concatenate([np.arange(5000), 2147483646 - np.arange(5000), near,
                        rng.integers(0, 2147483646, 1 << 18)])
    x = x[(x >= 0) & (x <= 2147483645)].astype(np.float64)
    q = x * inv
    got = fma(fma(np.full_like(x, -div), q, x), np.full_like(x, inv), q)
    assert np.array_equal(got, x / div)
