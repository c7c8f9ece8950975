"""The MoE operator's working range as measurable cases.

A case is one call that a host of this library makes: a decoder layer's MoE
block at decode (one token, a small batch, a batch of 32), the block over a
prompt of some length, the routed experts alone on given routes, or one
projection on its own. The three layer shapes are the ones the benchmark and
the tests use:

  qwen   H 2048, 60 experts of 1408, top-4, shared expert of 5632
  olmoe  H 2048, 64 experts of 1024, top-8, no shared expert
  fine   H 2048, 128 experts of 768, top-8, Zipf-distributed expert popularity

Weights are N(0, 0.02) in the packed Q4 / Q8 formats (symmetric, one FP32 scale
per 128 elements) or BF16; hidden states are BF16 N(0, 1).
"""

from __future__ import annotations

import math
import sys
from pathlib import Path
from types import SimpleNamespace

import torch

_PACKAGE = str(Path.cwd() / "uma-qmoe_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from uma_qmoe_amd.native_backend import DenseBlock, DeviceExperts, load_native_extension  # noqa: E402

DEVICE = "cuda:0"
GROUP = 128
STD = 0.02
EPS = 1e-6

# hidden, experts, top-k, expert width, shared width, Zipf exponent of the expert popularity
SHAPES = {
    "qwen": SimpleNamespace(hidden=2048, experts=60, top_k=4, inter=1408, shared=5632, zipf=0.0),
    "olmoe": SimpleNamespace(hidden=2048, experts=64, top_k=8, inter=1024, shared=0, zipf=0.0),
    "fine": SimpleNamespace(hidden=2048, experts=128, top_k=8, inter=768, shared=0, zipf=1.1),
}
ENCODINGS = {"q4": "q4_group128", "q8": "q8_group128", "bf16": "bf16_le"}
WEIGHT_BYTES = {"q4": 0.5 + 4.0 / GROUP, "q8": 1.0 + 4.0 / GROUP, "bf16": 2.0}


def listed():
    return [
        # Decode of one sequence with the fixed Qwen model: a decoder layer's
        # RMSNorm and MoE block for one token, replayed from a HIP graph as
        # the host's decode loop does.
        {"name": "decode_qwen_q4", "call": "norm_layer", "shape": "qwen", "enc": "q4", "tokens": 1, "graph": True},
        # Decode of one sequence with the OLMoE shapes, called eagerly (a host
        # without graph capture): launch latency counts.
        {"name": "decode_olmoe_q4", "call": "layer", "shape": "olmoe", "enc": "q4", "tokens": 1, "graph": False},
        # A few sequences decoded together; the later Qwen layers are Q8.
        {"name": "decode_qwen_q8_b6", "call": "norm_layer", "shape": "qwen", "enc": "q8", "tokens": 6, "graph": True},
        # The benchmark's batch-32 decode.
        {"name": "decode_qwen_q4_b32", "call": "layer", "shape": "qwen", "enc": "q4", "tokens": 32, "graph": True},
        # A short chat prompt through one of the early (BF16) Qwen layers.
        {"name": "prefill_qwen_bf16_t77", "call": "norm_layer", "shape": "qwen", "enc": "bf16", "tokens": 77,
         "graph": False},
        # Fine-grained experts with hot and cold ones, routes from the host.
        {"name": "prefill_fine_q4_t256", "call": "routed", "shape": "fine", "enc": "q4", "tokens": 256,
         "graph": False},
        # The benchmark's 512-token prefill.
        {"name": "prefill_qwen_q4_t512", "call": "layer", "shape": "qwen", "enc": "q4", "tokens": 512, "graph": False},
        # A prompt of odd length through a Q8 layer.
        {"name": "prefill_qwen_q8_t999", "call": "norm_layer", "shape": "qwen", "enc": "q8", "tokens": 999,
         "graph": False},
        # A longer prompt through a BF16 layer.
        {"name": "prefill_qwen_bf16_t1535", "call": "norm_layer", "shape": "qwen", "enc": "bf16", "tokens": 1535,
         "graph": False},
        # A full prefill chunk.
        {"name": "prefill_qwen_q4_t2048", "call": "layer", "shape": "qwen", "enc": "q4", "tokens": 2048,
         "graph": False},
        # A long context (OLMoE's 4096 less one): 32760 routes.
        {"name": "prefill_olmoe_q4_t4095", "call": "layer", "shape": "olmoe", "enc": "q4", "tokens": 4095,
         "graph": False},
        # One expert's gate projection on the tokens that a 2048-token prompt
        # sends it, as a host with its own per-expert loop calls it.
        {"name": "linear_q4_r137", "call": "linear", "shape": "qwen", "enc": "q4", "tokens": 137, "graph": False},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    most = max(work(c)["flops"] for c in listed())
    while True:
        call = rng.choice(["layer", "norm_layer", "layer", "norm_layer", "routed", "linear"])
        shape = rng.choice(["qwen", "qwen", "olmoe"]) if call in ("layer", "norm_layer") else \
            rng.choice(["qwen", "olmoe", "fine"])
        tokens = _log_int(rng, 1, 1024 if call == "linear" else 4096)
        # a graph holds a decode step: one token per sequence of a batch
        graph = call in ("layer", "norm_layer") and tokens <= 64 and rng.random() < 0.5
        case = {"call": call, "shape": shape, "enc": rng.choice(["q4", "q4", "q8", "bf16"]), "tokens": tokens,
                "graph": graph}
        if work(case)["flops"] <= most:
            return case


# ------------------------------------------------------------------ inputs --
def _pack(w, enc):
    """(codes, scales) of fp32 matrices [E, rows, cols]: absmax per 128 elements over 7 or 127."""
    if enc == "bf16":
        return w.to(torch.bfloat16), None
    e, rows, cols = w.shape
    top = 7.0 if enc == "q4" else 127.0
    g = w.view(e, rows * cols // GROUP, GROUP)
    scales = g.abs().amax(-1) / top
    q = torch.round(g / scales.unsqueeze(-1)).clamp_(-top, top).to(torch.int8).view(e, rows, cols)
    if enc == "q4":
        n = q.view(torch.uint8) & 0xF
        q = n[..., 0::2] | (n[..., 1::2] << 4)
    return q.contiguous(), scales


def _unpack(codes, scales, enc):
    """float64 values of packed matrices [E, rows, cols]."""
    if enc == "bf16":
        return codes.double()
    if enc == "q4":
        lo, hi = codes & 0xF, codes >> 4
        q = torch.stack([lo, hi], -1).flatten(-2).to(torch.int16)
        q = q - 16 * (q >= 8).to(torch.int16)
    else:
        q = codes
    e, rows, cols = q.shape
    return (q.double().view(e, -1, GROUP) * scales.double().unsqueeze(-1)).view(e, rows, cols)


def _inputs(case, seed):
    """Everything the call needs, from the seed alone (device tensors)."""
    s = SHAPES[case["shape"]]
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)

    def normal(*size, std=1.0):
        return torch.randn(size, generator=gen, device=DEVICE, dtype=torch.float32) * std

    i = SimpleNamespace(shape=s, enc=case["enc"])
    i.x = normal(case["tokens"], s.hidden).to(torch.bfloat16)
    if case["call"] == "linear":
        i.w, i.ws = _pack(normal(1, s.inter, s.hidden, std=STD), case["enc"])
        return i
    i.gate, i.gate_s = _pack(normal(s.experts, s.inter, s.hidden, std=STD), case["enc"])
    i.up, i.up_s = _pack(normal(s.experts, s.inter, s.hidden, std=STD), case["enc"])
    i.down, i.down_s = _pack(normal(s.experts, s.hidden, s.inter, std=STD), case["enc"])
    i.router = normal(s.experts, s.hidden, std=STD).to(torch.bfloat16)
    i.sg = i.su = i.sd = i.seg = None
    if s.shared and case["call"] != "routed":
        i.sg, i.su = (normal(s.shared, s.hidden, std=STD).to(torch.bfloat16) for _ in range(2))
        i.sd = normal(s.hidden, s.shared, std=STD).to(torch.bfloat16)
        i.seg = normal(1, s.hidden, std=STD).to(torch.bfloat16)
    if case["call"] == "norm_layer":
        i.norm = (1.0 + normal(s.hidden, std=0.1)).to(torch.bfloat16)
    if case["call"] == "routed":
        logits = torch.nn.functional.linear(i.x, i.router).float()
        if s.zipf:
            ranks = torch.randperm(s.experts, generator=gen, device=DEVICE) + 1
            logits = logits - s.zipf * torch.log(ranks.float())
        logits = logits.to(torch.bfloat16).float()
        i.indices = torch.topk(logits, s.top_k, dim=-1).indices.contiguous()
        i.weights = torch.softmax(logits, -1).gather(-1, i.indices).to(torch.bfloat16)
    return i


def prepare(case, seed):
    _platform, ext = load_native_extension()
    i = _inputs(case, seed)
    st = SimpleNamespace(ext=ext, case=case, inputs=i, graph=None, outputs=None)
    s = i.shape
    if case["call"] == "linear":
        return st
    st.experts = DeviceExperts(ENCODINGS[case["enc"]], GROUP, s.experts, s.hidden, s.inter, i.gate, i.gate_s, i.up,
                               i.up_s, i.down, i.down_s)
    st.dense = DenseBlock(i.router, i.sg, i.su, i.sd, i.seg)
    st.workspace = None
    if case["graph"]:
        # a decode loop's graph: its own workspace, one eager step, then the capture
        shared = s.shared if i.sg is not None else 0
        st.workspace = ext.new_workspace(DEVICE, case["tokens"], s.hidden, s.inter, shared, s.experts, s.top_k)
        _call(st)
        torch.cuda.synchronize()
        st.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st.graph):
            st.outputs = _call(st)
    return st


def _call(st):
    i, ext, call = st.inputs, st.ext, st.case["call"]
    if call == "linear":
        n, k = i.shape.inter, i.shape.hidden
        if i.enc == "q4":
            return ext.q4_linear(i.x, i.w, i.ws, n, k, GROUP)
        if i.enc == "q8":
            return ext.q8_linear(i.x, i.w, i.ws, n, k, GROUP)
        return ext.bf16_linear(i.x, i.w[0])
    if call == "routed":
        return ext.moe_forward(st.experts, i.x, i.indices, i.weights)
    if call == "norm_layer":
        return ext.norm_moe_layer(st.experts, st.dense, i.x, i.shape.top_k, EPS, i.norm, workspace=st.workspace)
    return ext.moe_layer(st.experts, st.dense, i.x, i.shape.top_k, workspace=st.workspace)


def run(state):
    if state.graph is not None:
        state.graph.replay()
        return state.outputs
    return _call(state)


# -------------------------------------------------------------------- work --
def work(case):
    s = SHAPES[case["shape"]]
    t, per_weight = case["tokens"], WEIGHT_BYTES[case["enc"]]
    if case["call"] == "linear":
        n = s.inter * s.hidden
        return {"bytes": n * per_weight + 2.0 * t * (s.hidden + s.inter), "flops": 2.0 * t * n}
    # experts that at least one token chooses (on average, routes spread evenly)
    distinct = s.experts * (1.0 - (1.0 - s.top_k / s.experts) ** t)
    expert = 3 * s.inter * s.hidden
    data = distinct * expert * per_weight + 4.0 * t * s.hidden + 10.0 * t * s.top_k
    flops = 2.0 * t * s.top_k * expert
    if case["call"] != "routed":
        data += 2.0 * s.experts * (s.hidden + t)
        flops += 2.0 * t * s.experts * s.hidden
        if s.shared:
            data += 2.0 * s.hidden * (3 * s.shared + 1)
            flops += 2.0 * t * s.hidden * (3 * s.shared + 1)
    return {"bytes": data, "flops": flops}


def tolerance(case):
    # BF16 outputs over FP32 sums, with the SiLU product rounded to BF16 in
    # between: 3e-3 against 64 bits. Router logits are rounded to BF16 before
    # the top-k, so a sum in another order can swap two experts whose logits
    # round to neighbours: rare, and then that token's output moves.
    if case["call"] == "linear":
        return {"rel": 8e-3}
    if case["call"] == "routed":
        return {"rel": 1e-2}
    return {"rel": 1.5e-2, "differ": 4e-3}


# ------------------------------------------------------------------- exact --
def _bf16(v):
    return v.to(torch.bfloat16).double()


def _ffn(x, g, u, d):
    a = x @ g.T
    return (a * torch.sigmoid(a) * (x @ u.T)) @ d.T


def exact(case, seed):
    i = _inputs(case, seed)
    s, x = i.shape, i.x.double()
    if case["call"] == "linear":
        return x @ _unpack(i.w, i.ws, case["enc"])[0].T
    if case["call"] == "norm_layer":
        # the block's input is a BF16 tensor: RMSNorm rounds the normalised
        # value and the product with its weight
        x = _bf16(_bf16(x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)) * i.norm.double())
    logits = None
    if case["call"] == "routed":
        indices, p = i.indices, i.weights.double()
    else:
        logits = x @ i.router.double().T
        rounded = _bf16(logits)  # the router's output is BF16; ties go to the lower id
        indices = torch.sort(rounded, dim=-1, descending=True, stable=True).indices[:, :s.top_k]
        p = torch.softmax(rounded, -1).gather(-1, indices)
    out = torch.zeros_like(x)
    for e in range(s.experts):
        tok, slot = (indices == e).nonzero(as_tuple=True)
        if tok.numel() == 0:
            continue
        g, u, d = (_unpack(c[e:e + 1], None if sc is None else sc[e:e + 1], case["enc"])[0]
                   for c, sc in ((i.gate, i.gate_s), (i.up, i.up_s), (i.down, i.down_s)))
        out.index_add_(0, tok, _bf16(p[tok, slot]).unsqueeze(1) * _ffn(x[tok], g, u, d))
    if case["call"] == "routed":
        return out
    if s.shared:
        scale = _bf16(torch.sigmoid(_bf16(x @ i.seg.double().T)))
        out += scale * _ffn(x, i.sg.double(), i.su.double(), i.sd.double())
    return out, logits, p, indices
