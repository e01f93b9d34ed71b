"""The weight chain and PhaseSpaceWeight where their straight-line form does
not apply (genbod_f64, event_weight_f64): radicands outside the range of the
branch-free square root, masses outside that of its division, masses lost in
the momenta's rounding, mothers below threshold.  Weights are compared with
the oracle bit for bit, momenta within 1e-12 E."""
import numpy as np
import pytest
from gpu_util import evaluate, event_weight, generate, make_decay, make_functor, momentum_error
from hydra_amd import capi

pytestmark = pytest.mark.gpu
P_TOL = 1e-12


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float64).view(np.uint64)


def same_bits(a, b):
    a, b = np.asarray(a), np.asarray(b)
    nan = np.isnan(a)
    assert np.array_equal(nan, np.isnan(b))
    assert np.array_equal(bits(a[~nan]), bits(b[~nan]))


def masses(N):
    return [0.2 + 0.1 * ((5 * i) % 7) for i in range(N)]


@pytest.mark.parametrize("engine", ["squares3", "philox"])
@pytest.mark.parametrize("N", [2, 3, 6, 12])
@pytest.mark.parametrize("scale", [0, -190, -200, -230, 245, 250])
def test_scaled_masses(oracle, N, scale, engine):
    # radicands scale by 2^(4 scale): across 2^-767 and 2^1000
    m = [x * 2.0 ** scale for x in masses(N)]
    M = 1.5 * sum(m)
    cols, wt, evw = generate(make_decay(M, m, engine=engine), 77, 1500, first=3)
    ocols, owt = oracle.generate(M, m, 77, 1500, first=3, engine=engine)
    same_bits(wt.cpu().numpy(), owt)
    assert momentum_error(cols.cpu().numpy(), ocols, N)[0] <= P_TOL
    same_bits(evw.cpu().numpy(), oracle.event_weight(M, m, cols.cpu().numpy()))


@pytest.mark.parametrize("light", [1e-95, 1e-12, 1e-9])
@pytest.mark.parametrize("N", [2, 3, 5])
def test_light_daughter(oracle, N, light):
    # 1e-95 lies below the division's range; a mass of 1e-9 or less is lost in
    # the rounding of E^2 - p^2, so that squares come out zero or negative
    m = [light] + masses(N)[1:]
    M = 2.0 * sum(m)
    dec = make_decay(M, m)
    cols, wt, evw = generate(dec, 5, 5000)
    ocols, owt = oracle.generate(M, m, 5, 5000)
    same_bits(wt.cpu().numpy(), owt)
    # a soft light particle's own energy is no scale for its error: M is
    assert np.abs(cols.cpu().numpy() - ocols).max() <= P_TOL * M
    same_bits(evw.cpu().numpy(), oracle.event_weight(M, m, cols.cpu().numpy()))
    same_bits(event_weight(dec, cols).cpu().numpy(), evw.cpu().numpy())


@pytest.mark.parametrize("N", [2, 3, 6])
def test_mothers_around_threshold(oracle, N):
    # each mother's own fECM: far above, at, below threshold, and no number
    m = masses(N)
    rng = np.random.default_rng(3)
    mass = sum(m) * rng.choice([1.7, 1.0, 0.6, 2.0 ** 60], 1000)
    mth = np.zeros((4, 1000))
    mth[1:] = rng.normal(0, 0.3, (3, 1000))
    mth[0] = np.sqrt(mass ** 2 + (mth[1:] ** 2).sum(axis=0))
    mth[0, ::50] = np.nan
    f = make_functor(capi.F_MASS2, (1, 2))
    out = evaluate(make_decay(2 * sum(m), m), [f], 9, 1000, mothers=mth)
    ref = oracle.evaluate_mothers(m, 9, mth, [(capi.F_ONE, None)])
    same_bits(out[0].cpu().numpy(), ref[0])
