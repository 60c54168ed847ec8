"""The e4m3 activation quantizer's codes over every value it can round: each code's value, each midpoint and the floats
beside it, both signs, zeros, at scales that leave them exact."""
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
