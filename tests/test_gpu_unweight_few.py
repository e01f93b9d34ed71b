"""Unweighting of few events: the flags formed in one kernel, the counts summed
by the scatter (no scan kernel).  Against the chain of kernels that a call
without outputs, or of more events, takes: the edges of groups, 256-event
blocks, 1024-event tiles, and of the rules (3 * 2^17 and 2^20 events), with each
subset of the outputs."""
import ctypes

import numpy as np
import pytest
import torch
from gpu_util import (DEV, generate, make_decay, make_functor, ptr, rng_words, stream_handle,
                      unweight, unweight_sample)
from hydra_amd import capi

pytestmark = pytest.mark.gpu
SEED, UW = 11, 0x180EC6D33CFD0ABA


def decay(N, engine="squares3"):
    m = [0.2 + 0.1 * ((5 * i) % 7) for i in range(N)]
    return make_decay(1.6 * sum(m), m, engine=engine)


def call(dec, n, mixed, cols=True, idx=True, w=True):
    lib = capi.lib()
    ws = torch.empty(lib.hpsp_generate_unweight_workspace_size(n), dtype=torch.uint8, device=DEV)
    ws.fill_(0xA5)  # nothing is taken for cleared
    out = (torch.zeros((4 * dec.n, n), dtype=torch.float32 if mixed else torch.float64, device=DEV)
           if cols else None)
    io = torch.zeros(n, dtype=torch.int64, device=DEV) if idx else None
    wo = torch.zeros(n, dtype=torch.float64, device=DEV) if w else None
    acc = torch.full((1,), -1, dtype=torch.int64, device=DEV)
    fn = lib.hpsp_generate_unweight_mixed if mixed else lib.hpsp_generate_unweight
    capi.check(fn(ctypes.byref(dec), SEED, 5, n, UW, ptr(out), n, ptr(io), ptr(wo), ptr(ws),
                  ws.numel(), ptr(acc), stream_handle()), "generate_unweight")
    torch.cuda.synchronize()
    return int(acc.item()), out, io, wo


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("N,engine", [(2, "squares4"), (3, "squares3"), (6, "threefry"),
                                      (12, "philox_long")])
def test_few_events(N, engine, mixed):
    dec = decay(N, engine)
    for n in (1, 63, 64, 255, 256, 257, 1023, 1024, 1025, 70000, 262144, 3 * 131072,
              3 * 131072 + 1, 1 << 20, (1 << 20) + 1):
        cols, _, evw = generate(dec, SEED, n, first=5, prec=int(mixed), out_f32=mixed)
        count, _, _, _ = call(dec, n, mixed, cols=False, idx=False, w=False)
        k, out, idx, w = call(dec, n, mixed)
        assert k == count, (n, k, count)
        i = idx.long()
        assert torch.equal(i[:k], i[:k].sort().values) and torch.equal(i[k:], i[k:].sort().values)
        assert torch.equal(i.sort().values, torch.arange(n, device=DEV))
        assert torch.equal(out, cols[:, i]) and torch.equal(w, evw[i])
        # the test itself, w / max > u
        u = torch.as_tensor(rng_words("squares3", UW, 0, n).astype(np.float64) * 2.0 ** -32,
                            device=DEV)
        assert int(((evw[:n] / dec.max_weight) > u).sum().item()) == k
        for sub in ((True, False, False), (False, True, False), (False, False, True)):
            got = call(dec, n, mixed, *sub)
            assert got[0] == k
            for a, b in zip(got[1:], (out, idx, w)):
                assert a is None or torch.equal(a, b)


@pytest.mark.parametrize("N", [2, 3, 7])
def test_moving_unweight(oracle, N):
    m = [0.2 + 0.1 * ((5 * i) % 7) for i in range(N)]
    M = 1.6 * sum(m)
    dec = make_decay(M, m)
    for n in (1, 1000, 1024, 1025, 66000):
        cols, _, evw = generate(dec, SEED, n)
        c = cols.cpu().numpy()
        ref = oracle.unweight(M, m, c, UW)
        for w_in in (None, evw):
            k, out, idx, _ = unweight(dec, cols, UW, w_in=w_in)
            assert k == ref[0]
            assert np.array_equal(out.cpu().numpy()[:, :k], c[:, idx.cpu().numpy()[:k]])
            order = np.concatenate([np.sort(idx.cpu().numpy()[:k]), np.sort(idx.cpu().numpy()[k:])])
            assert np.array_equal(order, idx.cpu().numpy())


@pytest.mark.parametrize("n", [1, 1024, 5000, 1 << 18, (1 << 20) + 7])
def test_sample_counts(n):
    rng = np.random.default_rng(n)
    w, x = rng.random(n), rng.random((2, n))
    u = rng_words("squares3", capi.UNWEIGHT_SAMPLE_SEED, 0, n).astype(np.float64) * 2.0 ** -32
    keep = (u * w.max()) <= w
    for order in (0, 1):
        k, out, _, _ = unweight_sample(x, w, order=order)
        assert k == keep.sum()
        assert np.array_equal(out[:, :k], x[:, keep])
        assert np.array_equal(np.sort(out, axis=1), np.sort(x, axis=1))


@pytest.mark.parametrize("N", [2, 3, 5, 9])
def test_functor_maximum_from_values(N):
    # Unweight(F) that finds the maximum (its values kept in the output until
    # the scatter) against the one that is given it (values formed for the flags)
    dec = decay(N)
    f = make_functor(capi.F_BW_SUM, [(0.9, 0.1, 0.5, -0.1, 0, 1), (1.2, 0.2, 0.6, 1.5, 0, N - 1)])
    lib = capi.lib()
    for n in (1, 255, 1025, 300000, (1 << 20) + 5):
        cols, _, _ = generate(dec, SEED, n)
        ws = torch.empty(lib.hpsp_unweight_workspace_size(n), dtype=torch.uint8, device=DEV)
        top = torch.empty(1, dtype=torch.float64, device=DEV)
        capi.check(lib.hpsp_max_weight(ctypes.byref(dec), ctypes.byref(f), ptr(cols), n, n, ptr(ws),
                                       ws.numel(), ptr(top), stream_handle()), "hpsp_max_weight")
        want = unweight(dec, cols, UW, f=f, max_value=float(top.item()))
        for out, idx in ((True, True), (False, True), (True, False), (False, False)):
            got = unweight(dec, cols, UW, f=f, want_out=out, want_idx=idx)
            assert got[0] == want[0]
            for a, b in zip(got[1:3], want[1:3]):
                assert a is None or torch.equal(a, b)
