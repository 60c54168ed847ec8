"""Which scratch buffer a call gets (prism_amd.scratch), with the device's streams and captures stood in for on the CPU:
calls on two streams, or a captured call and an eager one, never share one; a stream keeps its own; the number kept is
bounded; and a device with no eager call has none to hand out under capture."""
import pytest
import torch

from prism_amd import _lib as L
from prism_amd import scratch


class _Stream:
    def synchronize(self):
        pass


@pytest.fixture
def gpu(monkeypatch):
    state = {"stream": 1, "capturing": False}
    monkeypatch.setattr(L, "raw_stream", lambda idx: state["stream"])
    monkeypatch.setattr(scratch, "_capturing", lambda: state["capturing"])
    monkeypatch.setattr(torch.cuda, "current_stream", lambda idx=None: _Stream())
    monkeypatch.setattr(scratch.Scratch, "_empty", staticmethod(lambda idx, n: torch.full((n,), 7, dtype=torch.uint8)))
    return state


DEV = torch.device("cuda", 0)


def test_one_buffer_per_stream(gpu):
    s = scratch.Scratch(64, zeroed=16)
    a = s.get(DEV)
    gpu["stream"] = 2
    b = s.get(DEV)
    assert a.data_ptr() != b.data_ptr() and not a[:16].any() and not b[:16].any() and a.numel() == b.numel() == 64
    assert s.get(torch.device("cuda", 1)).data_ptr() not in (a.data_ptr(), b.data_ptr())
    gpu["stream"] = 1
    assert s.get(DEV).data_ptr() == a.data_ptr()


@pytest.mark.parametrize("zeroed", [0, 16])
def test_captured_calls_share_with_no_eager_one(gpu, zeroed):
    s = scratch.Scratch(64, zeroed=zeroed)
    gpu["capturing"] = True
    assert s.get(DEV) is None and s.get(DEV, zeroed=False) is None
    gpu["capturing"] = False
    eager = s.get(DEV)
    gpu["capturing"] = True
    a, b = s.get(DEV), s.get(DEV, zeroed=False)
    assert len({t.data_ptr() for t in (eager, a, b)}) == 3
    assert b.numel() == 64 and a.numel() == (zeroed or 64) and not (zeroed and a.any())
    assert s.get(DEV, zeroed=False, need=40).numel() == 40 and s.get(DEV, zeroed=False, need=400).numel() == 64
    gpu["capturing"] = False
    assert s.get(DEV, need=40).data_ptr() == eager.data_ptr()


def test_bounded(gpu):
    s = scratch.Scratch(64)
    first = s.get(DEV)
    other = s.get(torch.device("cuda", 1))
    for i in range(2, 3 * scratch.STREAMS):
        gpu["stream"] = i
        s.get(DEV)
    assert sum(k[0] == 0 for k in s._eager) == scratch.STREAMS
    gpu["stream"] = 1
    assert s.get(torch.device("cuda", 1)).data_ptr() == other.data_ptr()
    assert s.get(DEV).data_ptr() != first.data_ptr()
