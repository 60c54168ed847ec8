"""The workloads this library's speed is judged on: quantized linear layers and blocks, as an engine calls them.

A case is one call sequence of the public Python API on one GPU, at the sizes of the projections the benchmark and the
dispatch tables name (hidden 5120, MLP 17408 or 13824, gate|up fused, 4096 square, 48 value heads of 128):

  op "linear"  activation producer, then one projection.  producer "rows" quantizes bf16 rows; "gated" is the linear
               attention's gated norm in front of its output projection.  epi 1 adds into the fp32 residual.
  op "mlp"     RMSNorm producer, fused gate|up projection, SwiGLU producer, down projection into the residual.

  fmt "q8"     Q8_0 weights (32-input blocks), int8 activations, one scale per token
  fmt "pc"     per-channel int8 weights, int8 activations
  fmt "q4k", "q6k"   k-quant weights, int8 activations, group 256 (the engine's producer) or "token" (one per token)
  fmt "mx8"    MXFP4 weights, e4m3 activations (panels from 64 rows, the prefill layout)
  fmt "mx4"    MXFP4 weights, e2m1 activations (the engine's W4A4)

"rows" is the number of rows the buffers are launched for (an engine's token bucket) and "live" the rows really there.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "startlux-prism_amd"))

from prism_amd import gguf_formats as GF  # noqa: E402
from prism_amd import mxfp4 as MX  # noqa: E402
from prism_amd import quant as KQ  # noqa: E402
from prism_amd import w4a8 as KW4  # noqa: E402
from prism_amd import w8a8 as KW  # noqa: E402

EPS = 1e-6
HEAD = 128


class _Cfg:
    eps, gdn_dim = EPS, HEAD

    def __init__(self, heads):
        self.v_heads = heads


def _linear(name, fmt, rows, n, k, producer="rows", epi=0, live=None, group=256):
    return dict(name=name, op="linear", fmt=fmt, rows=rows, live=rows if live is None else live, n=n, k=k,
                producer=producer, epi=epi, group=group)


def _mlp(name, fmt, rows, hid, ff, group=256):
    return dict(name=name, op="mlp", fmt=fmt, rows=rows, live=rows, n=hid, k=ff, group=group)


def listed():
    return [
        # one token of one user through one square projection: latency, launches and the host path
        _linear("q8_linear_1", "q8", 1, 4096, 4096),
        # a decode step of a few users through a whole Q8_0 MLP: the weight stream
        _mlp("q8_mlp_4", "q8", 4, 5120, 17408),
        # 40 users in a bucket of 48: the linear attention's gated norm and output projection into the residual
        _linear("q8_attn_out_40", "q8", 48, 5120, 6144, producer="gated", epi=1, live=40),
        # an ordinary prompt of an odd length through a wide projection
        _linear("q8_linear_777", "q8", 777, 13824, 5120),
        # the largest: 8192 prompt tokens through the fused gate|up projection
        _linear("q8_prefill_8192", "q8", 8192, 27648, 5120),
        # a decode step of 16 users through a whole Q4_K MLP
        _mlp("q4k_mlp_16", "q4k", 16, 5120, 13824),
        # 37 users, or a short prompt, through a Q4_K gate or up projection
        _linear("q4k_linear_37", "q4k", 37, 13824, 5120),
        # a long prompt through the same projection, one activation scale per token
        _linear("q4k_prefill_2048", "q4k", 2048, 13824, 5120, group="token"),
        # a short prompt through a Q6_K down projection into the residual (Q4_K_M files keep half of these in Q6_K)
        _linear("q6k_down_100", "q6k", 100, 5120, 17408, epi=1),
        # a decode step of 24 users on W4A4: the fused gate|up projection
        _linear("mx4_linear_24", "mx4", 24, 34816, 5120),
        # a long prompt on MXFP4 weights with e4m3 activations
        _linear("mx8_prefill_4096", "mx8", 4096, 5120, 5120),
        # an odd-length prompt through a whole per-channel MLP
        _mlp("pc_mlp_1500", "pc", 1500, 5120, 17408),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Another case of these ranges: 1 to 4096 rows, widths from 1024 to 34816, inputs from 2048 to 17408, ragged."""
    fmt = rng.choice(["q8", "q8", "q4k", "q6k", "mx4", "mx8", "pc"])
    rows = _log(rng, 1, 4096)
    group = rng.choice([256, "token"]) if fmt in ("q4k", "q6k") else 256
    if fmt in ("q8", "q4k", "pc") and rng.random() < 0.3:
        hid, ff = 256 * _log(rng, 8, 20), 256 * _log(rng, 16, 68)
        c = _mlp("", fmt, min(rows, 2048), hid, ff, group)
    else:
        n, k = 16 * _log(rng, 64, 2176), 256 * _log(rng, 8, 68)
        k = max(2048, min(k, (34816 * 5120 // n) // 256 * 256))          # no more weights than the widest projection
        rows = max(1, min(rows, (1 << 39) // (n * k)))
        live = rows if rng.random() < 0.7 else max(1, int(rows * rng.uniform(0.6, 1.0)))
        gated = fmt in ("q8", "q4k", "q6k", "pc") and rng.random() < 0.2
        c = _linear("", fmt, rows, n, k, "gated" if gated else "rows", rng.choice([0, 0, 1]), live, group)
    del c["name"]
    return c


# ------------------------------------------------------------------------------------------------ inputs

def _gen(seed, dev):
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed))
    return g


def _mx_rows(v, mode):
    """MXFP4 / MXFP8 of fp32 rows [m, k] -> (codes as values fp32 [m, k], exponents int [m, k / 32]).  "e2m1": scale
    2^ceil(log2(amax / 6)), magnitudes by the strict midpoints; "e4m3": 2^(floor(log2 amax) - 8), nearest even."""
    b = v.view(v.shape[0], -1, 32)
    amax = b.abs().amax(-1).clamp_min(1e-30)
    if mode == "e2m1":
        m, e = torch.frexp(amax / 6.0)                                   # amax / 6 = m 2^e, 0.5 <= m < 1
        e = torch.where(m == 0.5, e - 1, e).clamp(-127, 127)
        mid = torch.tensor([.25, .75, 1.25, 1.75, 2.5, 3.5, 5.0], device=v.device)
        grid = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6], device=v.device)
        a = torch.ldexp(b.abs(), -e[..., None])
        val = torch.where(b < 0, -1.0, 1.0) * grid[torch.bucketize(a, mid)]
    else:
        e = torch.frexp(amax)[1] - 1 - 8
        val = torch.ldexp(b, -e[..., None]).clamp(-448, 448).to(torch.float8_e4m3fn).float()
    return val.reshape(v.shape), e


def _mx_bytes(val, e):
    """e2m1 values and exponents -> row-major MX4 bytes (codes low nibble first, e8m0 exponents)."""
    mag = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6], device=val.device)
    c = torch.bucketize(val.abs(), mag).to(torch.uint8) | ((val < 0).to(torch.uint8) << 3)
    return (c[:, 0::2] | (c[:, 1::2] << 4)).contiguous(), (e + 127).to(torch.uint8).contiguous()


def _weight_values(g, n, k, dev):
    return torch.randn(n, k, generator=g, device=dev) * 0.02


def _weight(fmt, g, n, k, dev):
    """The device operand, as the load step of an engine makes it from a file's blocks."""
    w = _weight_values(g, n, k, dev)
    if fmt == "q8":
        return KW.weight_from_q8(GF.quantize_q8_0(w), 32)[0]
    if fmt == "pc":
        return KW.weight_from_q8(GF.quantize_q8_0(w), k)[0]
    if fmt in ("q4k", "q6k"):
        return KW4.repack(GF.quantize_q4k(w) if fmt == "q4k" else GF.quantize_q6k(w))
    return MX.from_rows(*_mx_bytes(*_mx_rows(w, "e2m1")))


def _weight_exact(fmt, g, n, k, dev):
    """The same weights as float64 [n, k] values of the quantized format, decoded here."""
    w = _weight_values(g, n, k, dev)
    if fmt in ("q8", "pc"):
        b = w.view(n, k // 32, 32)
        d = (b.abs().amax(-1) / 127).half()
        inv = torch.where(d > 0, 1.0 / d.float(), torch.zeros_like(d, dtype=torch.float32))
        v = torch.round(b * inv[..., None]).clamp(-127, 127).double() * d.double()[..., None]
        v = v.view(n, k)
        if fmt == "pc":
            s = v.abs().amax(-1, keepdim=True).clamp_min(1e-10) / 127.0
            v = torch.round(v / s).clamp(-127, 127) * s
        return v
    if fmt == "q4k":
        b = GF.quantize_q4k(w).raw.view(n * k // 256, 144).int()
        d, dm = (b[:, i].add(b[:, i + 1] << 8).to(torch.int16).view(torch.float16).double() for i in (0, 2))
        s = b[:, 4:16]
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        q = b[:, 16:].view(-1, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).view(-1, 8, 32).double()
        return ((d[:, None] * sc)[..., None] * q - (dm[:, None] * mn)[..., None]).view(n, k)
    if fmt == "q6k":
        b = GF.quantize_q6k(w).raw.view(n * k // 256, 210).int()
        d = b[:, 208].add(b[:, 209] << 8).to(torch.int16).view(torch.float16).double()
        sc = torch.where(b[:, 192:208] > 127, b[:, 192:208] - 256, b[:, 192:208]).double()
        lo, hi = b[:, :128].view(-1, 2, 2, 32), b[:, 128:192].view(-1, 2, 1, 32)
        sh = torch.tensor([0, 2, 4, 6], device=dev).view(1, 1, 4, 1)
        q = (torch.cat([lo & 15, lo >> 4], 2) | (((hi >> sh) & 3) << 4)).view(-1, 16, 16).double() - 32
        return ((d[:, None] * sc)[..., None] * q).view(n, k)
    val, e = _mx_rows(w, "e2m1")
    return (val.double().view(n, -1, 32) * torch.exp2(e.double())[..., None]).view(n, k)


def _inputs(case, seed, dev):
    """(weights' generator, the activations): fixed by the seed, the same for prepare() and exact()."""
    g = _gen(2 * seed + 1, dev)
    m, n, k = case["rows"], case["n"], case["k"]
    if case["op"] == "mlp":
        x = dict(h=torch.randn(m, n, generator=g, device=dev) * 2.0, w=torch.rand(n, generator=g, device=dev) + 0.5)
    elif case["producer"] == "gated":
        x = dict(o=torch.randn(m, k, generator=g, device=dev),
                 z=torch.randn(m, 2 * k, generator=g, device=dev).to(torch.bfloat16),
                 w=torch.rand(HEAD, generator=g, device=dev) + 0.5)
    else:
        x = dict(x=torch.randn(m, k, generator=g, device=dev).to(torch.bfloat16))
    if case["op"] == "linear" and case["epi"]:
        x["res"] = torch.randn(m, n, generator=g, device=dev)
    return _gen(2 * seed + 2, dev), x


def _buffers(case, k, dev):
    """The quantized activation buffers of a projection of k inputs, kept by the engine between steps."""
    m, fmt = case["rows"], case["fmt"]
    if fmt in ("q8", "pc"):
        return dict(q=torch.zeros(m, k, dtype=torch.int8, device=dev), s=torch.zeros(m, device=dev))
    if fmt in ("q4k", "q6k"):
        ng = 1 if case["group"] == "token" else k // 256
        return dict(q=torch.zeros(m, k, dtype=torch.int8, device=dev), s=torch.zeros(ng, m, device=dev),
                    xs=torch.zeros(k // 256, m, 16, dtype=torch.int8, device=dev))
    if fmt == "mx4":
        q = torch.zeros(m, k // 2, dtype=torch.uint8, device=dev)
    else:
        q = MX.act_panels(m, k, dev).zero_() if m >= 64 else torch.zeros(m, k, dtype=torch.uint8, device=dev)
    return dict(q=q, s=torch.zeros(m, k // 32, dtype=torch.uint8, device=dev))


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    gw, st = _inputs(case, seed, dev)
    m, n, k, fmt = case["rows"], case["n"], case["k"], case["fmt"]
    st.update(case=case, live=torch.tensor([case["live"]], dtype=torch.int32, device=dev))
    if case["op"] == "mlp":
        st.update(gu=_weight(fmt, gw, 2 * k, n, dev), down=_weight(fmt, gw, n, k, dev), a=_buffers(case, n, dev),
                  b=_buffers(case, k, dev), mid=torch.zeros(m, 2 * k, dtype=torch.bfloat16, device=dev),
                  res=st["h"].clone())
        return st
    st.update(wt=_weight(fmt, gw, n, k, dev), a=_buffers(case, k, dev))
    st["out"] = st["res"] if case["epi"] else torch.zeros(m, n, dtype=torch.bfloat16, device=dev)
    if case["producer"] == "gated":
        st["o"], st["cfg"] = st["o"].view(m, k // HEAD, HEAD), _Cfg(k // HEAD)
    return st


# ------------------------------------------------------------------------------------------------ one pass

def _group(case, k):
    return k if case["group"] == "token" else 256


def _gemm(case, a, w, out, live, k, epi):
    fmt = case["fmt"]
    if fmt == "q8":
        KW.gemm(a["q"], a["s"], w, None, out, live, 32, epi=epi)
    elif fmt == "pc":
        KW.gemm(a["q"], a["s"], w, None, out, live, k, epi=epi)
    elif fmt in ("q4k", "q6k"):
        KW4.gemm(a["q"], a["s"], a["xs"], w, out, live, epi=epi)
    else:
        MX.gemm(a["q"], a["s"], w, out, live, epi=epi)


def run(st):
    case, live = st["case"], st["live"]
    m, n, k = case["rows"], case["n"], case["k"]
    a = st["a"]
    w8 = case["fmt"] in ("q8", "pc")
    if case["op"] == "mlp":
        b = st["b"]
        if w8:
            KQ.norm_q8(st["h"], st["w"], a["q"], a["s"], live, m, EPS)
        else:
            KQ.norm_g(st["h"], st["w"], a["q"], a["s"], a["xs"], live, m, EPS, group=_group(case, n))
        _gemm(case, a, st["gu"], st["mid"], live, n, 0)
        if w8:
            KQ.swiglu_q8(st["mid"], None, b["q"], b["s"], live, m)
        else:
            KQ.swiglu_g(st["mid"], b["q"], b["s"], b["xs"], live, m, group=_group(case, k))
        _gemm(case, b, st["down"], st["res"], live, k, 1)
        return st["mid"], st["res"]
    if case["producer"] == "gated":
        if w8:
            KQ.gated_norm_q8(st["o"], st["z"], k, st["w"], None, a["q"], a["s"], live, m, st["cfg"])
        else:
            KQ.gated_norm_g(st["o"], st["z"], k, st["w"], a["q"], a["s"], a["xs"], live, m, st["cfg"],
                            group=_group(case, k))
    elif w8:
        KQ.rows_q8(st["x"], None, a["q"], a["s"], live, m)
    elif case["fmt"] in ("q4k", "q6k"):
        KQ.rows_g(st["x"], a["q"], a["s"], a["xs"], live, m, group=_group(case, k))
    elif case["fmt"] == "mx4":
        MX.quantize_act(st["x"], a["q"], a["s"])
    else:
        MX.quantize_act_fp8(st["x"], a["q"], a["s"], live)
    _gemm(case, a, st["wt"], st["out"], live, k, case["epi"])
    return st["out"]


# ------------------------------------------------------------------------------------------------ what it cannot do without

_WEIGHT_BYTES = {"q8": 34 / 32, "pc": 1.0, "q4k": 144 / 256, "q6k": 210 / 256, "mx4": 17 / 32, "mx8": 17 / 32}


def work(case):
    m, n, k, wb = case["live"], case["n"], case["k"], _WEIGHT_BYTES[case["fmt"]]
    if case["op"] == "mlp":          # residual read, normed, added into; gate|up out, read by SwiGLU
        return dict(bytes=3 * n * k * wb + m * n * 4 * 3 + m * 2 * k * 2, flops=6.0 * m * n * k)
    x = m * k * (6 if case["producer"] == "gated" else 2)
    return dict(bytes=n * k * wb + x + m * n * (8 if case["epi"] else 2), flops=2.0 * m * n * k)


def tolerance(case):
    # bf16 outputs: the store's rounding is 1.7e-3 of the value in the 2-norm.  Through an MLP a changed rounding of
    # gate|up moves some of the next int8 rows by one step; into an fp32 residual only the activations' rounding at
    # half steps shows, measured up to 4e-4.
    if case["op"] == "linear" and case["epi"]:
        return {"rel": 1.5e-3, "max": 0.05}
    return {"rel": 5e-3, "max": 0.05}


def _quantized(case, y):
    """The float64 values of y [m, k] after the case's activation quantizer."""
    fmt = case["fmt"]
    if fmt in ("mx4", "mx8"):
        val, e = _mx_rows(y.float(), "e2m1" if fmt == "mx4" else "e4m3")
        return (val.double().view(y.shape[0], -1, 32) * torch.exp2(e.double())[..., None]).view(y.shape)
    g = 256 if fmt in ("q4k", "q6k") and case["group"] == 256 else y.shape[1]
    b = y.view(y.shape[0], -1, g)
    s = b.abs().amax(-1, keepdim=True).clamp_min(1e-10) / 127
    return (torch.round(b / s) * s).view(y.shape)


def exact(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    gw, x = _inputs(case, seed, dev)
    m, n, k, live, fmt = case["rows"], case["n"], case["k"], case["live"], case["fmt"]
    if case["op"] == "mlp":
        h = x["h"].double()
        y = h * torch.rsqrt(h.square().mean(-1, keepdim=True) + EPS) * x["w"].double()
        mid = _quantized(case, y) @ _weight_exact(fmt, gw, 2 * k, n, dev).T
        gu = mid.to(torch.bfloat16).double()                             # the projection's output is bf16
        act = torch.nn.functional.silu(gu[:, :k]) * gu[:, k:]
        return mid, h + _quantized(case, act) @ _weight_exact(fmt, gw, n, k, dev).T
    if case["producer"] == "gated":
        o, z = x["o"].double().view(m, -1, HEAD), x["z"][:, k:].double()
        y = (o * torch.rsqrt(o.square().mean(-1, keepdim=True) + EPS) * x["w"].double()).view(m, k)
        y = y * torch.nn.functional.silu(z)
    else:
        y = x["x"].double()
    out = _quantized(case, y) @ _weight_exact(fmt, gw, n, k, dev).T
    out[live:] = 0                                                       # rows past the live count stay as they were
    return x["res"].double() + out if case["epi"] else out
