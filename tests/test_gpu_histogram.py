"""DenseHistogram fills on the GPU against the oracle (bit-equal to the
reference's DenseHistogram::Fill, see test_oracle) and the golden vectors.

Bars: every event lands in the reference's bin (GetGlobalBin's operations),
so unit-weight counts are exact; weighted bins agree to rounding, since the
additions inside a bin run in another order: |d| <= 1e-13 * (sum of |w| in
the bin).  The fused fill from event columns computes its axes and its
PhaseSpaceWeight from the same momenta the oracle is given.
"""
import ctypes

import numpy as np
import pytest
import torch

from gpu_util import DEV, generate, make_decay, make_functor
from hydra_amd import capi
from hydra_amd.capi import check, lib, ptr, stream_handle

pytestmark = pytest.mark.gpu

C1 = (5.279, [3.0969, 0.493677, 0.13957])


def fill_columns(grid, lo, hi, x, w=None):
    h = capi.make_histogram(grid, lo, hi)
    xt = torch.as_tensor(np.ascontiguousarray(np.atleast_2d(x)), dtype=torch.float64, device=DEV)
    wt = None if w is None else torch.as_tensor(np.ascontiguousarray(w), device=DEV)
    out = torch.empty(int(np.prod(grid)) + 2, dtype=torch.float64, device=DEV)
    check(lib().hpsp_histogram_fill(ctypes.byref(h), ptr(xt), xt.shape[1], xt.shape[1], ptr(wt),
                                    ptr(out), stream_handle()), "hpsp_histogram_fill")
    torch.cuda.synchronize()
    return out.cpu().numpy()


def fill_events(grid, lo, hi, dec, axes, cols, mode, w=None, n=None):
    h = capi.make_histogram(grid, lo, hi)
    n = cols.shape[1] if n is None else n
    out = torch.empty(int(np.prod(grid)) + 2, dtype=torch.float64, device=DEV)
    check(lib().hpsp_histogram_fill_events(ctypes.byref(h), ctypes.byref(dec),
                                           capi.functor_array(axes), ptr(cols), cols.shape[1], n,
                                           mode, ptr(w), ptr(out), stream_handle()),
          "hpsp_histogram_fill_events")
    torch.cuda.synchronize()
    return out.cpu().numpy()


def abs_sums(oracle, grid, lo, hi, x, w):
    return oracle.histogram_fill(grid, lo, hi, x, np.abs(w))


def check_weighted(got, exp, scale):
    assert np.all(np.abs(got - exp) <= 1e-13 * scale + 1e-300)


def m2(v):
    return v[0] * v[0] - v[1] * v[1] - v[2] * v[2] - v[3] * v[3]


@pytest.mark.parametrize("grid", [[50], [100, 100], [8, 9, 10], [5, 6, 7, 8], [300, 300]])
def test_fill_columns_vs_oracle(oracle, grid):
    rng = np.random.default_rng(len(grid) * 1000 + grid[0])
    nd = len(grid)
    lo = rng.uniform(-2, 0, nd)
    hi = lo + rng.uniform(0.5, 3, nd)
    n = 200000
    x = rng.uniform(lo - 0.05 * (hi - lo), hi + 0.05 * (hi - lo), (n, nd)).T.copy()
    # edge cases: exactly the limits, all below, all above, undefined keys
    x[:, 0] = hi
    x[:, 1] = lo
    x[:, 2] = lo - 10 * (hi - lo)
    x[:, 3] = hi + 10 * (hi - lo)
    x[0, 4] = np.nan
    w = rng.exponential(1.0, n)
    assert np.array_equal(fill_columns(grid, lo, hi, x), oracle.histogram_fill(grid, lo, hi, x))
    check_weighted(fill_columns(grid, lo, hi, x, w), oracle.histogram_fill(grid, lo, hi, x, w),
                   abs_sums(oracle, grid, lo, hi, x, w))


def test_fill_golden(golden):
    x = golden["hist_dalitz_x"]
    lo, hi = golden["hist_dalitz_limits"]
    assert np.array_equal(fill_columns([20, 20], lo, hi, x), golden["hist_dalitz_n"])
    got = fill_columns([20, 20], lo, hi, x, golden["gen_c1_w"])
    check_weighted(got, golden["hist_dalitz_w"], golden["hist_dalitz_w"])
    got = fill_columns([25], [lo[0]], [hi[0]], golden["hist_1d_x"][None, :])
    assert np.array_equal(got, golden["hist_1d_n"])
    # the fused fill straight from the reference's own events and weights
    M, m = C1
    dec = make_decay(M, m)
    cols = torch.as_tensor(np.ascontiguousarray(golden["gen_c1_p"].reshape(4096, 12).T),
                           device=DEV)
    wcol = torch.as_tensor(golden["gen_c1_w"], device=DEV)
    axes = [make_functor(capi.F_MASS2, (0, 1)), make_functor(capi.F_MASS2, (1, 2))]
    got = fill_events([20, 20], lo, hi, dec, axes, cols, capi.HIST_WEIGHT_ONE)
    assert np.array_equal(got, golden["hist_dalitz_n"])
    got = fill_events([20, 20], lo, hi, dec, axes, cols, capi.HIST_WEIGHT_COLUMN, wcol)
    check_weighted(got, golden["hist_dalitz_w"], golden["hist_dalitz_w"])
    # PhaseSpaceWeight recomputed in the fill equals the reference's weights
    got = fill_events([20, 20], lo, hi, dec, axes, cols, capi.HIST_WEIGHT_PHSP)
    check_weighted(got, golden["hist_dalitz_w"], golden["hist_dalitz_w"])


@pytest.mark.parametrize("N", [3, 5, 12])
def test_fill_events_vs_oracle(oracle, N):
    rng = np.random.default_rng(70 + N)
    m = list(rng.uniform(0.1, 1.0, N))
    M = sum(m) * 2.0
    dec = make_decay(M, m)
    n = 1 << 20
    cols, _, evw = generate(dec, 11, n, want_wt=False)
    axes = [make_functor(capi.F_MASS2, (0, 1)), make_functor(capi.F_MASS2, (1, N - 1))]
    lo = [(m[0] + m[1]) ** 2, (m[1] + m[N - 1]) ** 2]
    hi = [M * M * 0.6, M * M * 0.7]  # part of the plane: under- and overflow occur
    c = cols.cpu().numpy().reshape(N, 4, n)
    x = np.vstack([m2(c[0] + c[1]), m2(c[1] + c[N - 1])])
    w = evw.cpu().numpy()
    grid = [64, 48]
    got = fill_events(grid, lo, hi, dec, axes, cols, capi.HIST_WEIGHT_ONE)
    assert np.array_equal(got, oracle.histogram_fill(grid, lo, hi, x))
    exp = oracle.histogram_fill(grid, lo, hi, x, w)
    for mode, wc in ((capi.HIST_WEIGHT_COLUMN, evw), (capi.HIST_WEIGHT_PHSP, None)):
        got = fill_events(grid, lo, hi, dec, axes, cols, mode, wc)
        check_weighted(got, exp, exp)


@pytest.mark.parametrize("N", [4, 5, 6, 8, 9, 10, 12])
def test_event_axes_equal_their_columns(N):
    # axes that read fewer daughters than there are, as many and more, from
    # registers or from memory: the counts of the axis values as columns
    m = [0.2 + 0.1 * ((5 * i) % 7) for i in range(N)]
    M = 1.8 * sum(m)
    dec = make_decay(M, m)
    n, ld = 30011, 30020
    cols, _, evw = generate(dec, 17, n, ld=ld, want_wt=False)
    bw = [(1.1, 0.2, 0.7, 0.3, 0, N - 1), (1.5, 0.3, 0.4, -0.2, 1, 2), (0.9, 0.1, 1.0, 0.0, 3, 1)]
    pair = make_functor(capi.F_MASS2, (N - 1, 1))
    sets = [([pair, make_functor(capi.F_MASS, (2, 3))], [[0, M * M], [0, M]]),
            ([make_functor(capi.F_BW_SUM, bw)], [[0, 10]]),
            ([make_functor(capi.F_COS_HELICITY, (0, 1)), pair], [[-1, 1], [0, M * M]])]
    p = capi.Particles()
    p.n = N
    for i in range(N):
        p.cols[i], p.ld[i] = cols.data_ptr() + 32 * ld * i, ld
    for axes, lim in sets:
        x = torch.empty((len(axes), n), dtype=torch.float64, device=DEV)
        check(lib().hpsp_particles_evaluate(ctypes.byref(p), capi.functor_array(axes), len(axes), n,
                                            ptr(x), n, stream_handle()), "evaluate")
        grid, lo, hi = [60] * len(axes), [v[0] for v in lim], [v[1] for v in lim]
        h = capi.make_histogram(grid, lo, hi)
        ref = []
        for w in (None, evw):
            out = torch.empty(60 ** len(axes) + 2, dtype=torch.float64, device=DEV)
            check(lib().hpsp_histogram_fill(ctypes.byref(h), ptr(x), n, n, ptr(w), ptr(out),
                                            stream_handle()), "fill")
            ref.append(out.cpu().numpy())
        got = fill_events(grid, lo, hi, dec, axes, cols, capi.HIST_WEIGHT_ONE, n=n)
        assert np.array_equal(got, ref[0]) and got.sum() == n
        for mode, wc in ((capi.HIST_WEIGHT_COLUMN, evw), (capi.HIST_WEIGHT_PHSP, None)):
            check_weighted(fill_events(grid, lo, hi, dec, axes, cols, mode, wc, n=n), ref[1], ref[1])


@pytest.mark.parametrize("N", [3, 4])
@pytest.mark.parametrize("over", [-1, 7])
def test_events_beside_the_size_where_loads_wait(N, over):
    """2^21 events: from there a wave reads one daughter's columns after the other's."""
    m = [0.2 + 0.1 * ((5 * i) % 7) for i in range(N)]
    M = 1.8 * sum(m)
    dec = make_decay(M, m)
    n = (1 << 21) + over
    cols, _, evw = generate(dec, 17, n, want_wt=False)
    axes = [make_functor(capi.F_MASS2, (0, N - 1)), make_functor(capi.F_COS_HELICITY, (0, 1))]
    p = capi.Particles()
    p.n = N
    for i in range(N):
        p.cols[i], p.ld[i] = cols.data_ptr() + 32 * n * i, n
    x = torch.empty((2, n), dtype=torch.float64, device=DEV)
    check(lib().hpsp_particles_evaluate(ctypes.byref(p), capi.functor_array(axes), 2, n, ptr(x), n,
                                        stream_handle()), "evaluate")
    grid, lo, hi = [60, 60], [0.0, -1.0], [M * M, 1.0]
    h = capi.make_histogram(grid, lo, hi)
    ref = []
    for w in (None, evw):
        out = torch.empty(3602, dtype=torch.float64, device=DEV)
        check(lib().hpsp_histogram_fill(ctypes.byref(h), ptr(x), n, n, ptr(w), ptr(out),
                                        stream_handle()), "fill")
        ref.append(out.cpu().numpy())
    got = fill_events(grid, lo, hi, dec, axes, cols, capi.HIST_WEIGHT_ONE, n=n)
    assert np.array_equal(got, ref[0]) and got.sum() == n
    for mode, wc in ((capi.HIST_WEIGHT_COLUMN, evw), (capi.HIST_WEIGHT_PHSP, None)):
        got = fill_events(grid, lo, hi, dec, axes, cols, mode, wc, n=n)
        # two sums of a bin's entries in any order, each off by a rounding per entry
        assert np.all(np.abs(got - ref[1]) <= 2.0 ** -52 * ref[0] * ref[1])


def test_fill_repeats_and_empty():
    """A fill overwrites the contents; n = 0 leaves them zero."""
    x = np.linspace(0, 1, 1001)[None, :]
    a = fill_columns([10], [0.0], [1.0], x)
    b = fill_columns([10], [0.0], [1.0], x)
    assert np.array_equal(a, b) and a.sum() == 1001
    h = capi.make_histogram([10], [0.0], [1.0])
    out = torch.full((12,), 7.0, dtype=torch.float64, device=DEV)
    check(lib().hpsp_histogram_fill(ctypes.byref(h), None, 0, 0, None, ptr(out),
                                    stream_handle()), "fill")
    torch.cuda.synchronize()
    assert np.all(out.cpu().numpy() == 0.0)
