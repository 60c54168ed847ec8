"""GPU parity of the W4A8 kernel between the decode and the tile kernels (kernel "mid"; "auto" picks it beyond 16 rows on
shapes off the dispatch table): every form the launch picks from, row tiles per workgroup, rounds that end inside the
super-blocks, one and two weight tiles."""
import numpy as np
import pytest
import torch

import oracle as O
from _inputs import acts_bf16, q6k_random_blocks, rng, weights_f32

pytestmark = pytest.mark.gpu


# rows: 2, 3 and 4 row tiles and several row groups, ends inside a tile; N: one tile, odd and even tile counts, wide (two
# tiles per workgroup) and narrow; K / 256: fewer super-blocks than waves, a last round of one, several rounds; the
# eight-wave, two-tile form (Q4_K, narrow, even tile count, up to three row tiles) below, at and over its waves in one
# round, several and a short last one; rows within the decode kernels'
@pytest.mark.parametrize("M,N,K,live", [(17, 16, 256, 17), (37, 48, 1280, 30), (64, 80, 2304, 64), (40, 8224, 1280, 33),
                                        (64, 8224, 512, 50), (100, 96, 2560, 97), (200, 64, 768, 130),
                                        (37, 96, 2304, 30), (17, 32, 5120, 17), (48, 64, 4352, 48), (33, 160, 1536, 33),
                                        (24, 96, 17408, 20), (5, 64, 1024, 4)])
@pytest.mark.parametrize("kind", ["q4k", "q6k"])
@pytest.mark.parametrize("group", [256, 0])
def test_mid_bits(dev, kind, group, M, N, K, live):
    from prism_amd import w4a8 as K4
    from prism_amd.gguf_formats import KQuant
    if kind == "q6k":
        raw = q6k_random_blocks(N, K // 256, seed=N + K)
    else:
        raw = O.q4k_quantize(weights_f32(N, K, N + K))
    raw = raw.reshape(N, K // 256, -1)
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(dev)            # noqa: E731
    w = K4.repack(KQuant(t(raw), kind, K))
    q, a, xs = O.quant_rows_g(O.bf16_to_f32(acts_bf16(M, K, seed=M)), group or K)
    base = rng(7).standard_normal((M, N), dtype=np.float32)
    n = torch.tensor([live], dtype=torch.int32, device=dev)
    for epi in (0, 1):
        out = t(base).clone() if epi else torch.zeros(M, N, dtype=torch.bfloat16, device=dev)
        ref = t(base).clone() if epi else torch.zeros(M, N, dtype=torch.bfloat16, device=dev)
        auto = ref.clone()
        K4.gemm(t(q), t(a), t(xs), w, out, n, epi=epi, kernel="mid")
        K4.gemm(t(q), t(a), t(xs), w, auto, n, epi=epi)
        K4.gemm(t(q), t(a), t(xs), w, ref, n, epi=epi, kernel="tile")
        torch.cuda.synchronize()
        got = out.cpu().numpy() if epi else out.view(torch.int16).cpu().numpy().view(np.uint16)
        assert torch.equal(out, ref) and torch.equal(auto, ref)
        want = _oracle(kind, q, a, xs, raw, epi, live, base)
        assert np.array_equal(got[:live], want[:live])


def _oracle(kind, q, a, xs, raw, epi, live, base):
    a = a if a.shape[0] > 1 else a[0].copy()
    out = base.copy() if epi else None
    if kind == "q6k":
        return O.w4a8_gemm_q6k(q, a, O.q6k_repack(raw), epi=epi, out=out, live=live)
    return O.w4a8_gemm(q, a, xs, O.q4k_repack(raw), epi=epi, out=out, live=live)
