"""RMSNorm launch against the CPU oracle: vector rows (multiples of 8, 128 to
8192, in one, two or four passes), the element-wise form for the others and for
unaligned pointers.

The FP32 sum of squares runs in another order than the oracle's (relative error
below 1e-5 here), so a value can round to the neighbouring bf16 once in the
normalised value and once in its product with the weight: at most 2 bf16 ulps."""

from __future__ import annotations

import pytest
import torch

from oracle import moe as om

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("rows,hidden,offset", [(1, 8, 0), (6, 2048, 0), (3, 2056, 0), (2, 8192, 0), (2, 8200, 0),
                                                (5, 2047, 0), (3, 2048, 1), (4, 120, 0), (4, 128, 0), (3, 136, 0),
                                                (2, 4096, 0), (2, 4104, 0)])
@pytest.mark.parametrize("weighted", [False, True])
def test_rmsnorm_rows(hip_ext, rows, hidden, offset, weighted):
    print(f"[case] rmsnorm {rows}x{hidden}+{offset} weighted={weighted}", flush=True)
    g = torch.Generator().manual_seed(hidden + rows)
    flat = torch.randn(rows * hidden + offset, generator=g).to(torch.bfloat16)
    w = (1 + 0.1 * torch.randn(hidden, generator=g)).to(torch.bfloat16) if weighted else None
    x = flat[offset:].view(rows, hidden)
    xd = flat.to(DEV)[offset:].view(rows, hidden)  # offset 1: not 16-byte aligned
    got = hip_ext.rmsnorm(xd, 1e-6, None if w is None else w.to(DEV)).cpu()
    ref = om.rmsnorm(x, 1e-6, w)
    ulp = torch.exp2(torch.floor(torch.log2(ref.float().abs().clamp_min(2.0 ** -126))) - 7)
    assert ((got.float() - ref.float()).abs() <= 2 * ulp).all()
