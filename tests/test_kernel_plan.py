"""Which kernels a call takes (uqm_moe_layer_plan): the rules on shapes, route
counts and options, on the host (256 compute units where there is no GPU)."""

from __future__ import annotations

import ctypes

import pytest

from uma_qmoe_amd import _native

ENC = {"q4": _native.UQM_Q4, "q8": _native.UQM_Q8, "bf16": _native.UQM_BF16}
P = 16  # any aligned address: the plan reads no device memory


def plan(enc, e, hidden, inter, k, tokens, shared=0):
    w = _native.ExpertWeights(ENC[enc], 128, e, hidden, inter, P, P, P, P, P, P)
    layer = _native.LayerWeights(w, P, k, 0, int(shared > 0), shared, P, P, P, P)
    out = _native.LayerPlan()
    _native.check(_native.library().uqm_moe_layer_plan(ctypes.byref(layer), tokens, ctypes.byref(out)), "plan")
    return out


def tile(*args, **kwargs):
    return plan(*args, **kwargs).routed_tile


# 60 experts of 2048 x 1408, top-4, with the shared expert; 64 of 2048 x 1024,
# top-8, without: both sides of every line
@pytest.mark.parametrize("args,shared,expected", [
    (("q4", 60, 2048, 1408, 4, 1), 5632, -1), (("q4", 60, 2048, 1408, 4, 2), 5632, -1),
    (("q4", 60, 2048, 1408, 4, 8), 5632, 1), (("q4", 60, 2048, 1408, 4, 9), 5632, 16),
    (("q4", 60, 2048, 1408, 4, 239), 5632, 16), (("q4", 60, 2048, 1408, 4, 240), 5632, 32),
    (("q4", 60, 2048, 1408, 4, 480), 5632, 32), (("q4", 60, 2048, 1408, 4, 481), 5632, 48),
    (("q4", 60, 2048, 1408, 4, 599), 5632, 48), (("q4", 60, 2048, 1408, 4, 600), 5632, 144),
    (("q8", 60, 2048, 1408, 4, 329), 5632, 32), (("q8", 60, 2048, 1408, 4, 330), 5632, 144),
    (("bf16", 60, 2048, 1408, 4, 59), 5632, 16), (("bf16", 60, 2048, 1408, 4, 60), 5632, 144),
    (("q4", 64, 2048, 1024, 8, 199), 0, 32), (("q4", 64, 2048, 1024, 8, 200), 0, 144),
])
def test_routed_tile(args, shared, expected):
    assert tile(*args, shared=shared) == expected


# Few experts make few large-tile items (row blocks x tiles): a serial chain of
# K stages on a part of the CUs, slower than the small tiles with their K split
# until there is enough work per CU.
@pytest.mark.parametrize("enc,e,hidden,inter,mean,large", [
    ("bf16", 8, 2048, 1408, 5, False), ("bf16", 8, 2048, 1408, 31, False), ("bf16", 8, 2048, 1408, 32, True),
    ("bf16", 16, 2048, 1408, 5, True), ("bf16", 4, 2048, 1408, 63, False), ("bf16", 4, 2048, 1408, 64, True),
    ("bf16", 4, 1024, 768, 127, False), ("bf16", 4, 1024, 768, 200, True),
    ("q8", 8, 2048, 1408, 35, False), ("q8", 8, 2048, 1408, 36, True), ("q8", 4, 4096, 4096, 26, False),
    ("q4", 6, 2048, 1408, 31, False), ("q4", 6, 2048, 1408, 32, True), ("q4", 4, 2048, 1408, 47, False),
    ("q4", 12, 2048, 1408, 25, True), ("q4", 4, 1024, 768, 64, False), ("q4", 8, 4096, 4096, 25, True),
])
def test_few_experts(enc, e, hidden, inter, mean, large):
    got = tile(enc, e, hidden, inter, 2, mean * e // 2)
    assert (got == 144) == large, got
    if not large:
        assert got in (16, 32, 48)


def test_shapes_without_small_tiles_keep_the_large_ones():
    """256 x 256 experts: the alternative is the GEMV, at any number of items.
    Below the line it stays the GEMV."""
    assert tile("bf16", 4, 256, 256, 2, 64) == 144
    assert tile("q4", 4, 256, 256, 2, 64) == 144
    assert tile("q4", 4, 256, 256, 2, 40) == 1
    # rows of 200 elements: neither
    assert tile("bf16", 8, 200, 256, 2, 64) == 1


def test_long_rows_take_smaller_tiles():
    """Scales of long rows leave no LDS for the widest grouped-GEMM items."""
    assert tile("q4", 44, 4096, 768, 4, 198) == 32
    assert tile("q8", 4, 5248, 768, 2, 36) == 16


def test_options_rule_the_plan():
    lib = _native.library()
    try:
        lib.uqm_set_option(_native.UQM_OPT_MFMA_MIN_TOKENS, 0)
        assert tile("q4", 60, 2048, 1408, 4, 2048, shared=5632) == 1
        assert plan("q4", 60, 2048, 1408, 4, 2048, shared=5632).gate_up_rows == 0
        lib.uqm_set_option(_native.UQM_OPT_MFMA_MIN_TOKENS, 1024)
        assert tile("q4", 60, 2048, 1408, 4, 1023) == 1 and tile("q4", 60, 2048, 1408, 4, 1024) == 144
        lib.uqm_set_option(_native.UQM_OPT_STREAM_MAX_ROUTES, 0)
        assert tile("q4", 60, 2048, 1408, 4, 1023) == 0
    finally:
        lib.uqm_set_option(_native.UQM_OPT_MFMA_MIN_TOKENS, 2)
        lib.uqm_set_option(_native.UQM_OPT_STREAM_MAX_ROUTES, 32)


def test_plan_validates_its_arguments():
    lib = _native.library()
    w = _native.ExpertWeights(_native.UQM_Q4, 128, 8, 256, 256, P, P, P, P, P, P)
    layer, out = _native.LayerWeights(w, P, 2, 0, 0, 0, None, None, None, None), _native.LayerPlan()
    assert lib.uqm_moe_layer_plan(None, 4, ctypes.byref(out)) == 1
    assert lib.uqm_moe_layer_plan(ctypes.byref(layer), 4, None) == 1
    assert lib.uqm_moe_layer_plan(ctypes.byref(layer), 0, ctypes.byref(out)) == 1
    layer.experts.gate = None
    assert lib.uqm_moe_layer_plan(ctypes.byref(layer), 4, ctypes.byref(out)) == 1


def dense(enc, e, hidden, inter, k, tokens, shared):
    p = plan(enc, e, hidden, inter, k, tokens, shared)
    return (p.gate_up_rows, p.gate_up_tokens), (p.down_rows, p.down_tokens, p.down_split)


# The shared expert's work items: the smallest from 128 tokens on, larger ones
# where they take less time in all (a last round of a few items counts)
@pytest.mark.parametrize("tokens,gate_up,down", [
    (127, (0, 0), (0, 0, 0)), (128, (128, 128), (128, 128, 4)), (384, (128, 256), (128, 128, 4)),
    (512, (128, 256), (128, 256, 4)), (640, (256, 256), (128, 256, 4)), (1025, (256, 256), (128, 256, 2)),
    (1280, (256, 256), (128, 256, 2)), (1535, (256, 256), (128, 256, 2)), (2048, (256, 256), (256, 256, 2)),
])
def test_dense_items_of_the_qwen_block(tokens, gate_up, down):
    assert dense("q4", 60, 2048, 1408, 4, tokens, 5632) == (gate_up, down)


def test_dense_items_where_large_ones_cost_more():
    """Shared expert 2816 x 2048 at 1025 tokens: a down projection on 256-row items
    split in four made the call 155 us against 150. 4096 x 1024 at 2048 tokens:
    256 gate/up items of 256 rows, a third of a second round of 192, 148 against
    143 us."""
    assert dense("q4", 32, 2048, 768, 4, 1025, 2816)[1] == (128, 256, 2)
    assert dense("q4", 32, 1024, 512, 4, 2048, 4096)[0] == (128, 256)
