"""GPU parity of the large-tile grouped GEMM (many routes per expert) against
the CPU oracle.

Its outputs are BF16 roundings of FP32 sums over BF16-rounded SiLU products, as
the oracle's, so both differ from the exact value by about 2^-9 per rounding:
rel-L2 <= 1e-2 and max-abs <= 2e-2, the bounds of every routed path."""

from __future__ import annotations

from dataclasses import replace

import pytest
import torch

from oracle import codec as oc
from oracle import moe as om
from test_gpu_kernels import assert_bf16_rounded
from test_gpu_mfma import (DEV, LARGE, RAGGED, close, dense_cpu, dense_plan, layout_of, mfma_on, note,  # noqa: F401
                           plan_of, to_dev)
from uma_qmoe_amd import _native
from uma_qmoe_amd import synthetic as syn

pytestmark = pytest.mark.gpu

# Routes per expert: one route, both sides of a 16-route step (every tile size
# of the kernel), the largest single tile, the first split, several tiles, none.
COUNTS = [1, 15, 16, 17, 32, 33, 49, 64, 65, 81, 97, 112, 113, 128, 129, 144, 145, 289, 0, 433]
# (H, I): K groups even and odd in either projection, from the smallest K on
SHAPES = [(640, 384), (256, 640), (512, 256), (1152, 896)]


def skewed_routes(counts, seed):
    """idx [T, 1] with counts[e] routes of expert e, in random order."""
    g = torch.Generator().manual_seed(seed)
    ids = torch.repeat_interleave(torch.arange(len(counts)), torch.tensor(counts))
    ids = ids[torch.randperm(ids.numel(), generator=g)]
    return ids.view(-1, 1), torch.rand(ids.numel(), 1, generator=g).to(torch.bfloat16)


@pytest.mark.parametrize("encoding", ["q4_group128", "q8_group128", "bf16_le"])
@pytest.mark.parametrize("hidden,inter", SHAPES)
def test_tile_sizes_against_oracle(mfma_on, encoding, hidden, inter):  # noqa: F811
    shape = syn.MoEShape("prefill", hidden, len(COUNTS), 1, inter, encoding=encoding)
    note(f"prefill {encoding} H={hidden} I={inter}")
    layer = syn.build_experts(shape, seed=hidden)
    idx, w = skewed_routes(COUNTS, inter)
    assert idx.numel() / len(COUNTS) >= 44  # the large-tile kernel's range for every encoding
    assert plan_of(layer, idx.shape[0], 1).routed_tile == LARGE
    x = syn.hidden_states(shape, idx.shape[0], seed=3)
    got = mfma_on.moe_forward(to_dev(layer), x.to(DEV), idx.to(DEV), w.to(DEV))
    ref = om.streaming_reference(x, idx, w, 0, syn.DeviceLayerReader({0: layer}), num_experts=len(COUNTS))
    close(got, ref, f"{encoding} H={hidden} I={inter}")


@pytest.mark.parametrize("encoding", ["q4_group128", "q8_group128"])
def test_wide_scale_groups_and_dropped_routes(mfma_on, encoding):  # noqa: F811
    """Scale groups of 256 elements (two K groups share a scale), top-2 routes
    with ids out of range."""
    shape = syn.MoEShape("prefill_g256", 512, 5, 2, 256, encoding=encoding, group_size=256)
    note(f"prefill group 256 {encoding}")
    layer = syn.build_experts(shape, seed=9)
    g = torch.Generator().manual_seed(4)
    idx = torch.stack([torch.randperm(5, generator=g)[:2] for _ in range(333)])
    w = torch.rand(333, 2, generator=g).to(torch.bfloat16)
    x = syn.hidden_states(shape, 333, seed=5)
    assert plan_of(layer, 333, 2).routed_tile == LARGE
    dropped = idx.clone()
    dropped[::5, 1] = -1
    dropped[1::7, 0] = 5
    w_ref = w.clone()
    w_ref[::5, 1] = 0
    w_ref[1::7, 0] = 0
    got = mfma_on.moe_forward(to_dev(layer), x.to(DEV), dropped.to(DEV), w.to(DEV))
    ref = om.streaming_reference(x, idx, w_ref, 0, syn.DeviceLayerReader({0: layer}), num_experts=5)
    close(got, ref, f"group 256 {encoding}")


def test_infinities_and_nan_stay_in_their_token(mfma_on):  # noqa: F811
    """Non-finite activations poison their own token's output and no other."""
    shape = syn.MoEShape("prefill_nan", 256, 2, 1, 256, encoding="q4_group128")
    note("prefill non-finite")
    layer = to_dev(syn.build_experts(shape, seed=2))
    t = 150
    idx = (torch.arange(t) % 2).view(-1, 1)
    w = torch.ones(t, 1, dtype=torch.bfloat16)
    x = syn.hidden_states(shape, t, seed=6)
    assert plan_of(layer, t, 1).routed_tile == LARGE
    clean = mfma_on.moe_forward(layer, x.to(DEV), idx.to(DEV), w.to(DEV)).cpu()
    bad = x.clone()
    bad[0, 3] = float("nan")  # token 0 pads expert 0's last tile
    bad[7, 9] = float("inf")
    out = mfma_on.moe_forward(layer, bad.to(DEV), idx.to(DEV), w.to(DEV)).cpu()
    keep = torch.ones(t, dtype=torch.bool)
    keep[[0, 7]] = False
    assert torch.equal(out[keep], clean[keep])
    assert out[0].isnan().all() and not out[7].isfinite().all()


def test_silu_of_large_negative_gates(mfma_on):  # noqa: F811
    """g / (1 + exp(-g)) down to the largest finite exp(-g) (g = -88.5), where
    the reciprocal of 1 + exp(-g) is subnormal. Token t's gate is GATES[t % 8]
    in every row, its up value 2^100; row 0 of the down matrix picks one of
    them. The product keeps FP32's accuracy (exp's argument error included,
    below 1e-4), then bf16 rounds it and the output: 2^-7 relative. Where
    exp(-g) overflows the quotient is 0."""
    note("prefill silu of large negative gates")
    gates = torch.tensor([-80.0, -87.0, -87.5, -88.0, -88.5, -0.5, -89.0, -100.0])
    shape = syn.MoEShape("prefill_silu", 256, 2, 1, 256, encoding="bf16_le")
    t = 80
    x = torch.zeros(t, 256, dtype=torch.bfloat16)
    x[torch.arange(t), torch.arange(t) % 8] = 1
    gate = torch.zeros(2, 256, 256)
    gate[:, :, :8] = gates
    up = torch.zeros(2, 256, 256)
    up[:, :, :8] = 2.0 ** 100
    down = torch.zeros(2, 256, 256)
    down[:, 0, 17] = 1
    layer = replace(syn.build_experts(shape), gate=gate.to(torch.bfloat16), up=up.to(torch.bfloat16),
                    down=down.to(torch.bfloat16))
    idx = (torch.arange(t) // 8 % 2).view(-1, 1)
    assert plan_of(layer, t, 1).routed_tile == LARGE
    got = mfma_on.moe_forward(to_dev(layer), x.to(DEV), idx.to(DEV), torch.ones(t, 1, dtype=torch.bfloat16, device=DEV))
    g = gates.double()
    ref = g / (1 + torch.exp(-g)) * 2.0 ** 100
    out = got.cpu().double()[:, 0].view(-1, 8)
    assert ((out[:, :6] - ref[:6]).abs() <= 2.0 ** -7 * ref[:6].abs()).all(), out[0]
    assert (out[:, 6:].abs() <= ref[6:].abs()).all()


def test_block_replays_from_a_graph(mfma_on):  # noqa: F811
    """A whole block on the large tiles, captured and replayed with eager work
    in between, equals the eager call bit for bit."""
    shape = replace(syn.C2, num_experts=8, intermediate=384, shared_intermediate=512)
    note("prefill graph")
    ext = mfma_on
    layer = syn.build_experts(shape, device=DEV)
    dense = syn.build_dense(shape, device=DEV)
    x = syn.hidden_states(shape, 900, device=DEV)  # 3600 routes, 450 per expert
    assert plan_of(layer, 900, shape.top_k, shape.shared_intermediate).routed_tile == LARGE
    ws = ext.new_workspace(DEV, 900, shape.hidden, shape.intermediate, shape.shared_intermediate, 8, shape.top_k)
    ref = ext.moe_layer(layer, dense, x, shape.top_k, workspace=ws)[0].clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        res = ext.moe_layer(layer, dense, x, shape.top_k, workspace=ws)[0]
    for _ in range(3):
        res.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(res, ref)
        ext.moe_layer(layer, dense, x, shape.top_k, workspace=ws)


# rows: both sides of the first that takes the tiles (Q8 17, the others 25), of
# one 16-row tile, of the largest tile, several tiles; out features: not a
# multiple of the 128-row block (16, 1424), below it (64), and one the tiles do
# not take (1420)
@pytest.mark.parametrize("encoding", ["q4_group128", "q8_group128", "bf16_le"])
@pytest.mark.parametrize("rows,n,k", [(16, 64, 256), (17, 1424, 256), (24, 64, 2048), (25, 1424, 256), (33, 16, 640), (144, 64, 2048), (145, 1424, 384),
                                      (700, 1420, 256), (1000, 1424, 512)])
def test_linear_many_rows(hip_ext, encoding, rows, n, k):
    note(f"linear {encoding} rows={rows} n={n} k={k}")
    g = torch.Generator().manual_seed(rows + n + k)
    w = torch.randn(1, n, k, generator=g) * 0.02
    data, scales = syn.encode_projection(w, encoding)
    x = torch.randn(rows, k, generator=g).to(torch.bfloat16)
    xd, wd = x.to(DEV), data[0].to(DEV)
    if encoding == "q4_group128":
        deq = oc.q4_dequantize(data.numpy().tobytes(), scales.numpy().tobytes(), (n, k))
        got = hip_ext.q4_linear(xd, wd, scales[0].to(DEV), n, k, 128)
    elif encoding == "q8_group128":
        deq = oc.q8_dequantize(data.numpy().tobytes(), scales.numpy().tobytes(), (n, k))
        got = hip_ext.q8_linear(xd, wd, scales[0].to(DEV), n, k, 128)
    else:
        deq = data[0].float().numpy()
        got = hip_ext.bf16_linear(xd, wd)
    assert_bf16_rounded(got, x.float() @ torch.from_numpy(deq).T, "linear")


@pytest.mark.parametrize("encoding", ["q4_group128", "q8_group128"])
def test_lowest_codes_on_the_tiles(hip_ext, encoding):
    """The codecs never write the lowest code (-8, -128); the tiles' conversions
    take it as two's complement all the same."""
    note(f"lowest codes {encoding}")
    rows, n, k = 40, 64, 256
    g = torch.Generator().manual_seed(12)
    low = -8 if encoding == "q4_group128" else -128
    codes = torch.randint(low, -low, (n, k), generator=g, dtype=torch.int8)
    codes[:, ::5] = low
    scales = torch.rand(n * k // 128, generator=g) * 1e-2
    x = torch.randn(rows, k, generator=g).to(torch.bfloat16)
    data = (codes[:, 0::2] & 15 | codes[:, 1::2] << 4).view(torch.uint8) if low == -8 else codes
    linear = hip_ext.q4_linear if low == -8 else hip_ext.q8_linear
    got = linear(x.to(DEV), data.contiguous().to(DEV), scales.to(DEV), n, k, 128)
    deq = codes.float() * scales.repeat_interleave(128).view(n, k)
    assert_bf16_rounded(got, x.float() @ deq.T, "lowest codes")


def test_linear_to_an_unaligned_output(hip_ext):
    """An output that is not 8-byte aligned stays on the GEMV: bit for bit its
    rows in calls of four."""
    note("linear unaligned output")
    rows, n, k = 136, 64, 512
    g = torch.Generator().manual_seed(13)
    data, scales = syn.encode_projection(torch.randn(1, n, k, generator=g) * 0.02, "q4_group128")
    w, s = data[0].to(DEV), scales[0].to(DEV)
    x = torch.randn(rows, k, generator=g).to(torch.bfloat16).to(DEV)
    gemv = torch.cat([hip_ext.q4_linear(x[i:i + 4], w, s, n, k, 128) for i in range(0, rows, 4)])
    buf = torch.zeros(rows * n + 2, dtype=torch.bfloat16, device=DEV)
    _native.check(hip_ext.lib.uqm_q4_linear(x.data_ptr(), rows, w.data_ptr(), s.data_ptr(), n, k, 128,
                                            buf.data_ptr() + 2, torch.cuda.current_stream().cuda_stream), "linear")
    assert torch.equal(buf[1:-1].view(rows, n), gemv)
    assert buf[0] == 0 and buf[-1] == 0


@pytest.mark.parametrize("encoding", ["q4_group128", "q8_group128", "bf16_le"])
def test_linear_obeys_the_mfma_option(hip_ext, encoding):
    """With UQM_OPT_MFMA_MIN_TOKENS 0 (or above the rows) a linear of many rows
    is the GEMV: bit for bit its rows in calls of four."""
    note(f"linear option {encoding}")
    rows, n, k = 136, 256, 2048
    g = torch.Generator().manual_seed(8)
    data, scales = syn.encode_projection(torch.randn(1, n, k, generator=g) * 0.02, encoding)
    w, s = data[0].to(DEV), None if scales is None else scales[0].to(DEV)
    x = torch.randn(rows, k, generator=g).to(torch.bfloat16).to(DEV)

    def linear(v):
        if encoding == "bf16_le":
            return hip_ext.bf16_linear(v, w)
        return (hip_ext.q4_linear if encoding == "q4_group128" else hip_ext.q8_linear)(v, w, s, n, k, 128)

    gemv = torch.cat([linear(x[i:i + 4]) for i in range(0, rows, 4)])
    assert not torch.equal(linear(x), gemv)  # the tiles sum in another order
    try:
        for least in (0, rows + 1):
            hip_ext.set_option(_native.UQM_OPT_MFMA_MIN_TOKENS, least)
            assert torch.equal(linear(x), gemv), least
    finally:
        hip_ext.set_option(_native.UQM_OPT_MFMA_MIN_TOKENS, 2)


@pytest.mark.parametrize("which,t", [("ragged", 4300), ("ragged", 9700), ("c2", 2100)])
def test_dense_256_row_items(mfma_on, which, t):  # noqa: F811
    """The shared expert on 256 x 256 items. The planner takes them for the
    ragged shape's gate/up at 4300 tokens (1344 rows: the last 128-row half
    block half full; 17 token tiles, the last one partial) and for its down
    projection at 9700 (1088 rows: 64 in the last block), and for both c2
    projections at 2100 tokens (K split in two)."""
    shape = RAGGED if which == "ragged" else syn.C2
    note(f"dense 256 rows {which} t={t}")
    layer = syn.build_experts(shape, device=DEV)
    dense = syn.build_dense(shape, device=DEV)
    down = {4300: (128, 256, 1), 9700: (256, 256, 1), 2100: (256, 256, 2)}[t]
    assert dense_plan(layer, t, shape.top_k, shape.shared_intermediate) == ((256, 256), down)
    x = syn.hidden_states(shape, t, seed=t)
    out, _logits, weights, indices = mfma_on.moe_layer(layer, dense, x.to(DEV), shape.top_k)
    pick = torch.randperm(t, generator=torch.Generator().manual_seed(t))[:24]
    pick = torch.unique(torch.cat([pick, torch.tensor([0, t - 1])]))
    ref, *_ = om.qwen_block(x[pick], layout_of(shape, dense_cpu(dense)), syn.DeviceLayerReader({0: layer}), 0,
                            routes=(weights.cpu()[pick], indices.cpu()[pick]))
    close(out.cpu()[pick], ref, f"dense 256 rows {which} t={t}")
    assert torch.isfinite(out.float()).all()
