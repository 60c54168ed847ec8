"""The activation quantizers' codes over every value they can round: each code's value, each midpoint and the floats beside
it, both signs, zeros, at scales that leave them exact; and the e2m1 scale's exponent about every power of two and 1.5 of one,
where it steps."""
import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift", [0, -20, 30])
def test_e4m3_codes(dev, shift):
    from prism_amd import mxfp4 as MX
    vals = np.array([O.e4m3_value(c) for c in range(0x7f)], np.float32)
    mids = ((vals[1:] + vals[:-1]) / 2).astype(np.float32)
    x = np.concatenate([vals, mids, np.nextafter(mids, np.float32(0)), np.nextafter(mids, np.float32(1e9)), [0.0, 2e-4]])
    x = np.concatenate([x, -x]).astype(np.float32)
    # one block of 32 per 31 values, its amax 448: the block's exponent is 0, so the values meet the conversion unscaled
    x = np.pad(x, (0, -len(x) % 31)).reshape(-1, 31)
    rows = np.concatenate([x, np.full((len(x), 1), 448.0, np.float32)], 1)
    rows = np.pad(rows, ((0, -len(rows) % 4), (0, 0))).reshape(1, -1) * np.float32(2.0 ** shift)
    q = torch.zeros(1, rows.shape[1], dtype=torch.uint8, device=dev)
    s = torch.zeros(1, rows.shape[1] // 32, dtype=torch.uint8, device=dev)
    MX.quantize_act_fp8(torch.from_numpy(rows).to(dev), q, s)
    torch.cuda.synchronize()
    rq, rs = O.mx_quant_act(rows, "e4m3")
    assert np.array_equal(q.cpu().numpy(), rq) and np.array_equal(s.cpu().numpy(), rs)


def test_e2m1_codes_and_exponents(dev):
    from prism_amd import mxfp4 as MX
    grid = np.array([0, .25, .5, .75, 1, 1.25, 1.5, 1.75, 2, 2.5, 3, 3.5, 4, 5, 6], np.float32)
    near = np.concatenate([grid, np.nextafter(grid, np.float32(-1)), np.nextafter(grid, np.float32(9))])
    near = near[np.abs(near) <= 6]
    codes = np.zeros((4, 32), np.float32)
    codes.reshape(-1)[:len(near)], codes.reshape(-1)[64:64 + len(near)] = near, -near
    codes[:, 31] = 6.0                                                 # the block's scale is 1
    amax = np.concatenate([f(np.float32(m) * np.float32(2.0) ** np.arange(-105, 128 - (m > 1), dtype=np.float32))
                           for m in (1.0, 1.5) for f in (lambda a: a, lambda a: np.nextafter(a, np.float32(0)),
                                                         lambda a: np.nextafter(a, np.float32(np.inf)))])
    amax = np.concatenate([amax, [0, 1e-30, 9e-31, 3.4e38]]).astype(np.float32)
    blocks = np.zeros((len(amax), 32), np.float32)
    blocks[:, 5], blocks[:, 9] = -amax, amax / np.float32(2)
    rows = np.concatenate([codes, blocks])
    rows = np.pad(rows, ((0, -len(rows) % 4), (0, 0))).reshape(1, -1)
    q = torch.zeros(1, rows.shape[1] // 2, dtype=torch.uint8, device=dev)
    s = torch.zeros(1, rows.shape[1] // 32, dtype=torch.uint8, device=dev)
    MX.quantize_act(torch.from_numpy(rows).to(dev), q, s)
    torch.cuda.synchronize()
    rq, rs = O.mx_quant_act(rows, "e2m1")
    assert np.array_equal(s.cpu().numpy(), rs) and np.array_equal(q.cpu().numpy(), rq)


def test_e2m1_long_batch_time(dev):
    """The e2m1 quantizer stays near the e4m3 one, which writes more and computes less: 1.17 times its time, 1.37 with a
    division for every eight inputs and seven compares for each.  The same codes whatever the batch (two pieces per thread
    here, one in a short batch), with a row that ends inside the last workgroup's."""
    from prism_amd import mxfp4 as MX
    M, K = 8192, 17408
    x = torch.randn(M, K, device=dev).to(torch.bfloat16)
    s = torch.zeros(M, K // 32, dtype=torch.uint8, device=dev)
    q4, q8 = (torch.zeros(M, w, dtype=torch.uint8, device=dev) for w in (K // 2, K))
    times = ([], [])
    for rep in range(30):
        for side, fn in enumerate((lambda: MX.quantize_act(x, q4, s), lambda: MX.quantize_act_fp8(x, q8, s))):
            e0, e1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            e0.record()
            for _ in range(5):
                fn()
            e1.record()
            torch.cuda.synchronize()
            if rep >= 10:
                times[side].append(e0.elapsed_time(e1) * 200)
    t4, t8 = (sorted(t)[len(t) // 2] for t in times)
    print(f"e2m1 {t4:.1f} us, e4m3 {t8:.1f} us")
    assert t4 < 1.28 * t8
    few, fs = torch.zeros(1000, K // 2, dtype=torch.uint8, device=dev), torch.zeros(1000, K // 32, dtype=torch.uint8, device=dev)
    MX.quantize_act(x, q4, s)
    MX.quantize_act(x[-1000:], few, fs)
    torch.cuda.synchronize()
    assert torch.equal(q4[-1000:], few) and torch.equal(s[-1000:], fs)
