"""SwiGLU producer at the sizes where its workgroup changes (64 rows; 4096 columns): the oracle's bits for every size."""
import numpy as np
import pytest
import torch

import oracle as O
from _inputs import rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,FF", [(64, 4352), (65, 4096), (65, 4352), (70, 8448), (66, 17408)])
@pytest.mark.parametrize("back", ["q8", "g"])
def test_swiglu_workgroup_sizes(dev, T, FF, back):
    from prism_amd import quant as KQ
    live = T - 1
    gu = O.bf16_to_f32(O.bf16_bits(rng(T + FF).standard_normal((T, 2 * FF)).astype(np.float32) * 2))
    g = torch.from_numpy(gu).to(dev).to(torch.bfloat16)
    q = torch.zeros(T, FF, dtype=torch.int8, device=dev)
    n = torch.tensor([live], dtype=torch.int32, device=dev)
    if back == "q8":
        s = torch.zeros(T, device=dev)
        KQ.swiglu_q8(g, None, q, s, n, T)
        want = O.swiglu_quant(gu, back="q8", live=live)
        assert np.array_equal(s.cpu().numpy()[:live], want[1][:live])
    else:
        s = torch.zeros(FF // 256, T, device=dev)
        xs = torch.zeros(FF // 256, T, 16, dtype=torch.int8, device=dev)
        KQ.swiglu_g(g, q, s, xs, n, T)
        want = O.swiglu_quant(gu, back="g256", live=live)
        assert np.array_equal(s.cpu().numpy()[:, :live], want[1][:, :live])
        assert np.array_equal(xs.cpu().numpy()[:, :live], want[2][:, :live])
    assert np.array_equal(q.cpu().numpy()[:live], want[0][:live])
