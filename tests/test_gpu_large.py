"""Paths that only the largest calls take: the three-kernel scan of Unweight
(beyond 2^28 events) and calls that one launch cannot hold (beyond 2^31)."""
import ctypes

import pytest
import torch
from gpu_util import DEV, check, lib, make_decay, make_functor, ptr, stream_handle
from hydra_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def give_memory_back():
    yield
    torch.cuda.empty_cache()


@pytest.mark.parametrize("n", [1 << 28, (1 << 28) + (1 << 20) + 77])
def test_unweight_scan(n):
    """Values of 0 and 1 with maximum 1: 1 passes every test w / max > u with u < 1
    and 0 none, so the kept events and their order are known."""
    torch.manual_seed(3)
    kept = torch.rand(n, device=DEV) < 0.3
    values = kept.double()
    ws_bytes = lib().hpsp_unweight_workspace_size(n)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=DEV)
    idx = torch.empty(n, dtype=torch.int64, device=DEV)
    nacc = torch.zeros(1, dtype=torch.int64, device=DEV)
    check(lib().hpsp_unweight_values(3, ptr(values), 1.0, 99, None, 0, n, None, 0, ptr(idx), None,
                                     ptr(ws), ws_bytes, ptr(nacc), stream_handle()), "unweight")
    k = int(kept.sum())
    assert int(nacc) == k
    assert torch.equal(idx[:k], kept.nonzero().squeeze(1))
    assert torch.equal(idx[k:], (~kept).nonzero().squeeze(1))


SPLIT = 1 << 31


@pytest.mark.parametrize("engine,prec", [("squares3", capi.FP64), ("philox_long", capi.MIXED)])
def test_generate_in_two_launches(engine, prec):
    """Weights of 2^31 + 1000 three-body events around the first launch's end, against
    a short call at the same events."""
    dec = make_decay(5.279, [3.0969, 0.493677, 0.13957], engine=engine)
    n, first = SPLIT + 1000, 12345

    def call(b, k):
        w = torch.empty(k, dtype=torch.float64, device=DEV)
        check(lib().hpsp_generate(ctypes.byref(dec), 7, first + b, k, prec, None, 0, 0, ptr(w), None,
                                  stream_handle()), "generate")
        return w

    w = call(0, n)
    for b, k in ((0, 2000), (SPLIT - 1000, 2000)):
        assert torch.equal(w[b:b + k], call(b, k))


def test_evaluate_in_two_launches():
    dec = make_decay(5.279, [3.0969, 0.493677, 0.13957])
    fs = capi.functor_array([make_functor(capi.F_MASS2, (0, 2))])
    n = SPLIT + 1000

    def call(b, k):
        out = torch.empty((2, k + 5), dtype=torch.float64, device=DEV)
        check(lib().hpsp_evaluate(ctypes.byref(dec), fs, 1, 7, b, k, ptr(out), k + 5,
                                  stream_handle()), "evaluate")
        return out[:, :k]

    out = call(0, n)
    for b, k in ((0, 2000), (SPLIT - 1000, 2000)):
        assert torch.equal(out[:, b:b + k], call(b, k))
