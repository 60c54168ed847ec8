"""GEMMs whose kernels hand scratch to one another (the prefill's panel copies, the split decodes' partial sums), in
flight on two streams at once and in a replayed graph beside an eager call: every result is that of the call alone."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _int8(g, *shape):
    return torch.randint(-127, 128, shape, generator=g, dtype=torch.int8, device=g.device)


def _calls(kind, dev):
    """Two calls of one kind on different activations: [(run(out), out)]."""
    from prism_amd import mxfp4 as MX
    from prism_amd import w8a8 as KW
    g = torch.Generator(device=dev)
    g.manual_seed(11)
    M, N, K = {"q8": (1024, 16384, 512), "pc_panels": (2048, 16384, 512), "pc_split": (64, 512, 17408),
               "mx_split": (16, 512, 16384)}[kind]
    n = torch.tensor([M], dtype=torch.int32, device=dev)
    if kind == "q8":
        w = KW.pack_q8(_int8(g, N, K), (torch.rand(N, K // 32, generator=g, device=dev) * 1e-3).half())
    elif kind == "mx_split":
        w = MX.pack(torch.randn(N, K, generator=g, device=dev))
    else:
        w = KW.pack_i8(_int8(g, N, K), torch.rand(N, 1, generator=g, device=dev) * 1e-3)
    calls = []
    for _ in range(2):
        if kind == "mx_split":
            a, s = torch.empty(M, K, dtype=torch.uint8, device=dev), torch.empty(M, K // 32, dtype=torch.uint8, device=dev)
            MX.quantize_act_fp8(torch.randn(M, K, generator=g, device=dev), a, s)
            run = lambda out, a=a, s=s: MX.gemm(a, s, w, out, n, kernel="split")               # noqa: E731
        else:
            a, s = _int8(g, M, K), torch.rand(M, generator=g, device=dev)
            kernel = "split" if kind == "pc_split" else "tile"
            run = lambda out, a=a, s=s: KW.gemm(a, s, w, None, out, n, 32 if kind == "q8" else K, kernel=kernel)  # noqa: E731
        calls.append((run, torch.zeros(M, N, dtype=torch.bfloat16, device=dev)))
    return calls


KINDS = ["q8", "pc_panels", "pc_split", "mx_split"]


@pytest.mark.parametrize("kind", KINDS)
def test_two_streams(dev, kind):
    calls = _calls(kind, dev)
    want = []
    for run, out in calls:
        run(out)
        want.append(out.clone())
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in calls]
    for _ in range(20):
        for (run, out), st in zip(calls, streams):
            with torch.cuda.stream(st):
                run(out)
    torch.cuda.synchronize()
    for (_, out), w in zip(calls, want):
        assert torch.equal(out, w)


@pytest.mark.parametrize("kind", KINDS)
def test_graph_beside_eager(dev, kind):
    (run_g, out_g), (run_e, out_e) = _calls(kind, dev)
    run_g(out_g), run_e(out_e)
    want_g, want_e = out_g.clone(), out_e.clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run_g(out_g)
    st = torch.cuda.Stream()
    for _ in range(10):
        out_g.zero_(), out_e.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(st):
            graph.replay()
        run_e(out_e)
        torch.cuda.synchronize()
        assert torch.equal(out_g, want_g) and torch.equal(out_e, want_e)
