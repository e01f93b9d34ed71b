"""AverageOn's chunks generated by four waves or by 8 or 16 (few chunks): the
result over many chunks equals, bit for bit, the fixed-order merge of the
chunks' own results, on both sides of the rule and with ragged last chunks."""
import numpy as np
import pytest
import torch
from gpu_util import DEV, average_on, make_decay, make_functor
from hydra_amd import capi

pytestmark = pytest.mark.gpu
CHUNK, WIDE = 4096, 256  # kAvgChunk, kAvgWideChunks


@pytest.mark.parametrize("prec", [capi.FP64, capi.MIXED])
@pytest.mark.parametrize("engine,N", [("squares3", 2), ("squares3", 3), ("philox_long", 6),
                                      ("squares4", 7), ("threefry", 12)])
def test_chunks_merge_to_the_whole(engine, N, prec):
    m = [0.2 + 0.1 * ((5 * i) % 7) for i in range(N)]
    dec = make_decay(1.6 * sum(m), m, engine=engine)
    f = make_functor(capi.F_MASS2, (0, N - 1))
    parts = np.stack([average_on(dec, 3, CHUNK, f=f, first=CHUNK * c, prec=prec)
                      for c in range(WIDE + 1)])
    for chunks, extra in ((2, 0), (WIDE, 0), (WIDE, 1), (WIDE - 1, 700), (WIDE + 1, 0)):
        n = chunks * CHUNK + extra
        rows = list(parts[:chunks])
        if extra:
            rows.append(average_on(dec, 3, extra, f=f, first=chunks * CHUNK, prec=prec))
        p = torch.as_tensor(np.stack(rows), device=DEV)
        out = torch.empty(3, dtype=torch.float64, device=DEV)
        capi.check(capi.lib().hpsp_stats_reduce(capi.ptr(p), len(rows), capi.ptr(out),
                                                capi.stream_handle()), "hpsp_stats_reduce")
        torch.cuda.synchronize()
        whole = average_on(dec, 3, n, f=f, prec=prec)
        assert np.array_equal(out.cpu().numpy().view(np.uint64), whole.view(np.uint64)), (n, N)
