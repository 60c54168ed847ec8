"""GPU parity of the exact Q8_0 prefill tile kernel (packed weights, kernel "tile") at the edges of its tiles, stages and
column widths, and at the activation scales and sums where its scaled fold hands over to the plain one."""
import numpy as np
import pytest
import torch

import oracle as O
from _inputs import int8_acts, q8_weights, rng

pytestmark = pytest.mark.gpu


def _run(dev, a, s, qs, d, epi, live=None, out0=None):
    from prism_amd import w8a8 as KW
    M, N = a.shape[0], qs.shape[0]
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(dev)            # noqa: E731
    w = KW.pack_q8(t(qs), t(d.view(np.int16)).view(torch.float16))
    out = t(out0) if epi else torch.zeros(M, N, dtype=torch.bfloat16, device=dev)
    n = torch.tensor([M if live is None else live], dtype=torch.int32, device=dev)
    KW.gemm(t(a), t(s), w, None, out, n, 32, epi=epi, kernel="tile")
    torch.cuda.synchronize()
    return out.cpu().numpy() if epi else out.view(torch.int16).cpu().numpy().view(np.uint16)


# two, three and four column subtiles per wave (the last two need several hundred tiles); one, two and more stages; rows
# and columns that end inside a tile, a wave and a subtile; panel activations (M >= 1024, N >= 16384) with four and with
# three subtiles
@pytest.mark.parametrize("M,N,K,live", [(1, 16, 128, 1), (33, 80, 384, 32), (130, 208, 256, 129), (300, 13840, 256, 290),
                                        (500, 16384, 128, 500), (1100, 16400, 256, 1030), (1024, 17424, 384, 1001)])
def test_tile_bits(dev, M, N, K, live):
    a, s = int8_acts(M, K, seed=M + N)
    qs, d = q8_weights(N, K, seed=K + N)
    assert np.array_equal(_run(dev, a, s, qs, d, 0, live)[:live], O.w8a8_gemm(a, s, qs, d, 32, epi=0, live=live)[:live])
    base = rng(5).standard_normal((M, N), dtype=np.float32)
    got = _run(dev, a, s, qs, d, 1, live, base)
    assert np.array_equal(got, O.w8a8_gemm(a, s, qs, d, 32, epi=1, out=base.copy(), live=live))


@pytest.mark.parametrize("scales", [(0.0, -0.5, 2.0 ** -47, 2.0 ** 30.9, 1e-10 / 127), (2.0 ** -49, 1.0),
                                    (2.0 ** 31, 3e-39, 1.0), (float("inf"), 1e-30, 0.25), (float("nan"), 1.0)])
def test_tile_scale_range(dev, scales):
    """Rows of extreme activation scales (in the scaled fold's range, at its ends, and beyond them where the workgroup
    takes the plain fold), the largest sums of either sign (all bytes -128) and zero, subnormal and large weight scales."""
    M, N, K = 140, 112, 256
    g = rng(3)
    a = g.integers(-128, 128, (M, K), dtype=np.int8)
    a[1], a[2], a[3] = -128, 127, 0
    s = np.full(M, 0.01, np.float32)
    s[:2 * len(scales)] = np.repeat(np.array(scales, np.float32), 2)
    qs = g.integers(-128, 128, (N, K), dtype=np.int8)
    qs[0], qs[1] = -128, 127
    d = (g.random((N, K // 32)) * 0.01).astype(np.float16)
    d[2], d[3], d[4] = 0, 6e-8, 60000
    d = d.view(np.uint16)
    got, want = _run(dev, a, s, qs, d, 0), O.w8a8_gemm(a, s, qs, d, 32, epi=0)
    nan = (want & 0x7fff) > 0x7f80
    assert np.array_equal((got & 0x7fff) > 0x7f80, nan) and np.array_equal(got[~nan], want[~nan])


def test_stale_scales_past_the_live_rows_cost_nothing(dev):
    """Scales of a bucket's rows past the live count (whatever its last use left there) do not send the live rows' tile to
    the plain fold.  The two folds give the same bits, so only the time tells them apart: with the stale scales read this
    shape took 56.5 us against 48.4; medians of repeated alternating launches."""
    from prism_amd import w8a8 as KW
    M, N, K, live = 128, 16384, 5120, 100
    g = torch.Generator(device=dev)
    g.manual_seed(1)
    a = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int8, device=dev)
    w = KW.pack_q8(torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8, device=dev),
                   (torch.rand(N, K // 32, generator=g, device=dev) * 1e-3).half())
    clean = torch.full((M,), 0.01, device=dev)
    stale = clean.clone()
    stale[live:] = float("nan")
    n = torch.tensor([live], dtype=torch.int32, device=dev)
    outs = [torch.zeros(M, N, dtype=torch.bfloat16, device=dev) for _ in range(2)]
    times = ([], [])
    for rep in range(30):
        for side, s in enumerate((clean, stale)):
            e0, e1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            e0.record()
            for _ in range(5):
                KW.gemm(a, s, w, None, outs[side], n, 32, kernel="tile")
            e1.record()
            torch.cuda.synchronize()
            if rep >= 10:
                times[side].append(e0.elapsed_time(e1) / 5)
    assert torch.equal(*outs)
    c, t = (sorted(x)[len(x) // 2] for x in times)
    print(f"clean {c * 1e3:.1f} us, stale {t * 1e3:.1f} us")
    assert t < 1.08 * c
