"""Engine words shared between neighbouring events (event_words.h) at the edges
of the sharing: runs of groups, ragged last groups, and the place where the
64-bit event counter wraps, which the Random123 engines carry on from event by
event (EngineR123's discard)."""
import numpy as np
import pytest
import torch
from gpu_util import average_on, evaluate, generate, make_decay, make_functor, momentum_error
from hydra_amd import capi
from test_gpu_generate_unweight import same, same_mixed

pytestmark = pytest.mark.gpu
R123 = ["philox", "philox_long", "threefry", "threefry_long"]


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float64).view(np.uint64)


def decay(N):
    m = [0.2 + 0.1 * ((5 * i) % 7) for i in range(N)]
    return 1.6 * sum(m), m


@pytest.mark.parametrize("before", [1, 63, 64, 130, 255])
@pytest.mark.parametrize("N", [2, 3, 5, 12])
@pytest.mark.parametrize("engine", ["squares3"] + R123)
def test_counter_wrap(oracle, N, engine, before):
    # `before` events of the call lie before the wrap of event + 3N
    M, m = decay(N)
    dec = make_decay(M, m, engine=engine)
    first = (2 ** 64 - 3 * N - before) % 2 ** 64
    n = before + 150
    cols, wt, _ = generate(dec, 41, n, first=first)
    a, wa = oracle.generate(M, m, 41, n, first=first, engine=engine)
    assert np.array_equal(bits(wt.cpu().numpy()), bits(wa))
    assert momentum_error(cols.cpu().numpy(), a, N)[0] <= 1e-12
    mix, wm, _ = generate(dec, 41, n, first=first, prec=capi.MIXED)
    assert np.abs(wm.cpu().numpy() / wa - 1).max() <= 4e-15
    assert momentum_error(mix.cpu().numpy(), a, N)[0] <= 1e-3
    f = [make_functor(capi.F_MASS2, (0, 1))]
    ev = evaluate(dec, f, 41, n, first=first)
    assert np.array_equal(bits(ev[0].cpu().numpy()), bits(wa))
    st = average_on(dec, 41, n, f=f[0], first=first)
    ref = (wa * ev[1].cpu().numpy()).sum() / wa.sum()
    assert abs(st[1] / ref - 1) <= 1e-12


@pytest.mark.parametrize("engine", R123)
def test_unweight_at_counter_wrap(engine):
    # event + 3N wraps among the last events
    for N in (3, 4):
        dec = make_decay(*decay(N), engine=engine)
        n = 2000 + 77 * N
        same(dec, 5, 2 ** 64 - 1 - n, n, 99)
        same_mixed(dec, 5, 2 ** 64 - 1 - n, n, 99)


@pytest.mark.parametrize("engine,N", [("squares3", 3), ("squares4", 6), ("philox", 3),
                                      ("philox_long", 4), ("threefry", 2), ("threefry_long", 2),
                                      ("threefry_long", 7)])
def test_runs_equal_single_groups(engine, N):
    # a call of runs of several groups against calls of one group per wave, the
    # first of them across the counter's wrap
    M, m = decay(N)
    dec = make_decay(M, m, engine=engine)
    n = (1 << 20) + 4 * 8192 * 64 + 77
    for first in (2 ** 64 - 3 * N - 500000, 12345):
        for prec in (capi.FP64, capi.MIXED):
            cols, wt, _ = generate(dec, 7, n, first=first % 2 ** 64, prec=prec)
            for b, k in ((0, 3000), (499900, 3000), (n - 2500, 2500)):
                c, w, _ = generate(dec, 7, k, first=(first + b) % 2 ** 64, prec=prec)
                assert torch.equal(cols[:, b:b + k], c)
                assert torch.equal(wt[b:b + k], w)


@pytest.mark.parametrize("N,momenta", [(2, True), (3, True), (3, False)])
def test_blocks_in_xcd_ranges(N, momenta):
    # at and above 4 GiB of output each XCD takes a contiguous range of blocks:
    # every range's edge and the ragged end, against short calls at the same events
    per = 32 * N + (0 if momenta else 8)
    n = ((4 << 30) // per // 2048 + 1) * 2048 + 256 * 3 + 17  # blocks no multiple of 8
    dec = make_decay(*decay(N))
    cols, wt, _ = generate(dec, 3, n, want_wt=not momenta, want_evw=False)
    per_xcd = (((n + 255) // 256 + 7) // 8) * 256
    for e in [0] + [x * per_xcd for x in range(1, 8)] + [n - 300]:
        lo, hi = max(0, e - 300), min(n, e + 300)
        ref, wref, _ = generate(dec, 3, hi - lo, first=lo)
        assert torch.equal(cols[:, lo:hi].cpu(), ref.cpu())
        if wt is not None:
            assert torch.equal(wt[lo:hi].cpu(), wref.cpu())
