"""The W4A8 activation producer with a scale per 256 inputs, at the edges of how it spreads a row over workgroups (one chunk
of 2048 inputs each, or two, three and four): the oracle's bits.  And its time on long batches: near that of the form
with one scale per row, which moves nearly the same bytes."""
import numpy as np
import pytest
import torch

import oracle as O
from _inputs import acts_bf16

pytestmark = pytest.mark.gpu


def _outs(M, K, groups, dev):
    return (torch.full((M, K), 7, dtype=torch.int8, device=dev), torch.full((groups, M), 7.0, device=dev),
            torch.full((K // 256, M, 16), 7, dtype=torch.int8, device=dev))


# chunks per row (K / 2048 rounded up) 1 to 9, whole and part chunks at the end; rows at which each spread is picked
@pytest.mark.parametrize("M,K,live", [(1, 256, 1), (3, 2304, 2), (1024, 8192, 1000), (1025, 2304, 1025), (1030, 4352, 1029),
                                      (1025, 6400, 1025), (1100, 8448, 1025), (600, 17408, 500), (586, 13824, 586)])
def test_rows_g_spread(dev, M, K, live):
    from prism_amd import quant as KQ
    x = acts_bf16(M, K, seed=M + K)
    q, a, xs = _outs(M, K, K // 256, dev)
    n = torch.tensor([live], dtype=torch.int32, device=dev)
    KQ.rows_g(torch.from_numpy(x.view(np.int16)).to(dev).view(torch.bfloat16), q, a, xs, n, M, group=256)
    torch.cuda.synchronize()
    rq, ra, rxs = O.quant_rows_g(O.bf16_to_f32(x[:live]), 256)
    assert np.array_equal(q[:live].cpu().numpy(), rq) and np.array_equal(a[:, :live].cpu().numpy(), ra)
    assert np.array_equal(xs[:, :live].cpu().numpy(), rxs)
    assert (q[live:] == 7).all() and (a[:, live:] == 7).all() and (xs[:, live:] == 7).all()


@pytest.mark.parametrize("K", [2560, 5120])
def test_rows_g_long_batch_time(dev, K):
    from prism_amd import quant as KQ
    M = 8192
    x = torch.randn(M, K, device=dev).to(torch.bfloat16)
    n = torch.tensor([M], dtype=torch.int32, device=dev)
    outs = {g: _outs(M, K, K // g, dev) for g in (256, K)}
    times = {g: [] for g in outs}
    for rep in range(40):
        for g, o in outs.items():
            e0, e1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            e0.record()
            for _ in range(10):
                KQ.rows_g(x, *o, n, M, group=g)
            e1.record()
            torch.cuda.synchronize()
            if rep >= 10:
                times[g].append(e0.elapsed_time(e1) * 100)
    t, row = (sorted(times[g])[len(times[g]) // 2] for g in (256, K))
    print(f"group 256 {t:.1f} us, one scale per row {row:.1f} us")
    assert t < 1.17 * row            # 1.08 here, 1.24-1.30 with a workgroup per chunk whatever the rows
