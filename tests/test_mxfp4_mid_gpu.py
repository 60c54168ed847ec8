"""The MXFP4 kernel between the decode and the tile kernels (kernel "mid", also "auto"'s choice): bit-equal to the tile kernel, whose MFMA
chain and segment order it shares, at the edges of its row groups, segments and rounds."""
import numpy as np
import pytest
import torch

from _inputs import acts_bf16, rng, weights_f32

pytestmark = pytest.mark.gpu


# rows: one to four row tiles, several row groups, ends inside a tile; N: odd and even tile counts; K: part of a segment,
# segments that end short, seven and eight waves (160 KB of LDS at four e2m1 row tiles and two weight tiles), more segments
# than waves (two and three rounds)
@pytest.mark.parametrize("M,N,K,live", [(1, 4096, 5248, 1), (16, 1264, 17408, 11), (17, 8208, 1024, 17),
                                        (33, 4112, 2176, 30), (50, 1664, 5120, 50), (100, 928, 9344, 70),
                                        (130, 544, 17408, 130), (64, 66000, 128, 50), (64, 1680, 5120, 64),
                                        (64, 64, 8192, 60), (50, 32, 7168, 50), (100, 48, 8192, 100),
                                        (97, 96, 16384, 90), (7, 80, 15360, 7)])
@pytest.mark.parametrize("fmt", ["e2m1", "e4m3"])
def test_mid_equals_tile(dev, fmt, M, N, K, live):
    from prism_amd import mxfp4 as MX
    w = MX.pack(torch.from_numpy(weights_f32(N, K, N + K)).to(dev), "max")
    x = torch.from_numpy(acts_bf16(M, K, M + K).view(np.int16)).to(dev).view(torch.bfloat16)
    q = torch.zeros(M, K if fmt == "e4m3" else K // 2, dtype=torch.uint8, device=dev)
    s = torch.zeros(M, K // 32, dtype=torch.uint8, device=dev)
    (MX.quantize_act_fp8 if fmt == "e4m3" else MX.quantize_act)(x, q, s)
    n = torch.tensor([live], dtype=torch.int32, device=dev)
    base = torch.from_numpy(rng(3).standard_normal((M, N), dtype=np.float32)).to(dev)
    for epi in (0, 1):
        outs = [base.clone() if epi else torch.zeros(M, N, dtype=torch.bfloat16, device=dev) for _ in range(3)]
        for out, kernel in zip(outs, ("tile", "mid", "auto")):
            MX.gemm(q, s, w, out, n, epi=epi, kernel=kernel)
        torch.cuda.synchronize()
        assert torch.equal(outs[1], outs[0]) and torch.equal(outs[2], outs[0])


def test_mid_wide_decode(dev):
    """e4m3 batches of up to 16 rows on a wide projection of the split decode's size: the split kernel's bits."""
    from prism_amd import mxfp4 as MX
    M, N, K = 9, 32768, 2560
    g = torch.Generator(device=dev)
    g.manual_seed(4)
    w = MX.pack(torch.randn(N, K, generator=g, device=dev) * 0.02)
    x = torch.randn(M, K, generator=g, device=dev).to(torch.bfloat16)
    q = torch.zeros(M, K, dtype=torch.uint8, device=dev)
    s = torch.zeros(M, K // 32, dtype=torch.uint8, device=dev)
    MX.quantize_act_fp8(x, q, s)
    outs = [torch.zeros(M, N, dtype=torch.bfloat16, device=dev) for _ in range(2)]
    for out, kernel in zip(outs, ("auto", "split")):
        MX.gemm(q, s, w, out, M, kernel=kernel)
    torch.cuda.synchronize()
    assert torch.equal(*outs)
