"""Decode attention at the edges of its tiles and splits: 1 to 16 query rows per KV group, row counts
around the 32-row wave tiles and 128-row block passes (mostly one pass a block: rows are split before
they are walked), three to four passes a block with a ragged end in every kernel (packed widths up to 96
and 160, wider keys with values up to 128, values up to 256), feature counts that leave part of a unit or
block empty, masked rows, and values that are infinite, in a first tile and in a later one. Reference: the oracle's float64 attention.

Tolerance: the output is bf16 (each within 2^-9 of its float32 value); scores, weights and sums are
float32 (P enters its products as three bf16 parts that add up to it), so the 2-norm error stays below
2^-8 of the result."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from harness import to_np
from logkv_amd.log_kv_pack import MidAttentionPlan, packed_attention, packed_dim
from oracle import readout as ro

pytestmark = pytest.mark.gpu

CASES = [
    # batch, groups, heads, tq, dk, dv, rows, causal
    (1, 1, 1, 1, 64, 64, 1, 1),
    (1, 2, 2, 2, 64, 64, 31, 2),
    (2, 1, 3, 1, 128, 128, 33, 0),
    (1, 2, 16, 2, 128, 128, 129, 2),
    (1, 1, 5, 1, 96, 96, 1000, 1),
    (3, 2, 4, 2, 128, 64, 2600, 2),
    (1, 1, 7, 2, 20, 12, 300, 2),
    (1, 1, 2, 1, 192, 128, 700, 1),
    (1, 1, 4, 2, 256, 256, 400, 2),
    (40, 16, 16, 1, 64, 64, 200, 1),
    (64, 4, 8, 1, 192, 128, 700, 1),        # 2 splits of three passes
    (1, 2, 4, 2, 168, 100, 300, 2),
]


# Lanes enough that a block walks several passes: (kernel's value limit, cases as above, passes of a block).
SEVERAL = [
    (64, (128, 4, 8, 1, 64, 64, 450, 1), 4),
    (128, (64, 4, 8, 2, 128, 128, 700, 2), 3),
    (128, (64, 4, 4, 1, 256, 128, 777, 1), 4),
    (256, (32, 4, 8, 1, 256, 256, 700, 1), 3),
    (256, (16, 8, 32, 2, 64, 200, 650, 2), 3),
]


def _rows(batch, groups, cap, dk, dv, g):
    dim = packed_dim(dk, dv)
    ka, va = torch.zeros(batch, groups, cap, dim), torch.zeros(batch, groups, cap, dim)
    ka[..., :dk] = torch.randn(batch, groups, cap, dk, generator=g)
    ka[..., dk] = torch.rand(batch, groups, cap, generator=g) * 4
    ka[:, :, :cap // 4, dk] = torch.where(torch.rand(batch, groups, cap // 4, generator=g) < 0.3, -10000.0,
                                          ka[:, :, :cap // 4, dk])
    va[..., :dv] = torch.randn(batch, groups, cap, dv, generator=g)
    return ka.to(torch.bfloat16).cuda(), va.to(torch.bfloat16).cuda()


@pytest.mark.parametrize("batch,groups,heads,tq,dk,dv,rows,causal", CASES)
def test_decode_matches_float64(batch, groups, heads, tq, dk, dv, rows, causal):
    g = torch.Generator().manual_seed(rows)
    ka, va = _rows(batch, groups, rows + 70, dk, dv, g)
    q = torch.randn(batch, heads, tq, dk, generator=g).to(torch.bfloat16).cuda()
    scale = dk ** -0.5
    plan = MidAttentionPlan(torch.tensor([rows - tq], dtype=torch.int32, device="cuda"), 0, 0)
    out, _ = packed_attention(q, ka, va, plan, tq, scale, causal, dv, groups)
    ref = ro.attention(to_np(q), to_np(ka)[:, :, :rows], to_np(va)[:, :, :rows], scale, causal, dv)
    err = np.linalg.norm(to_np(out).astype(np.float64) - ref)
    assert err <= 2.0 ** -8 * np.linalg.norm(ref), f"{err:.3e} of {np.linalg.norm(ref):.3e}"


@pytest.mark.parametrize("limit,case,passes", SEVERAL)
def test_several_passes_match_float64(limit, case, passes):
    batch, groups, _, _, _, dv, rows, _ = case
    assert dv <= limit
    splits = (512 if limit <= 128 else 256) // (batch * groups)
    assert -(-rows // (128 * splits)) == passes and rows % 32
    test_decode_matches_float64(*case)


@pytest.mark.parametrize("dk,dv,batch", [(64, 64, 128), (128, 128, 128), (192, 128, 128), (256, 256, 64)])
def test_infinite_values_in_a_later_tile(dk, dv, batch):
    """An infinity and a NaN in each wave's second or third tile reach their own feature only."""
    g = torch.Generator().manual_seed(dk)
    rows, groups = 515, 4   # one block a lane: five passes
    ka, va = _rows(batch, groups, rows, dk, dv, g)
    for wave, row in enumerate((130, 170, 330, 500)):
        va[:, :, row, 7 + wave], va[:, :, row, 40 + wave] = float("inf"), float("nan")
    q = torch.randn(batch, 2 * groups, 1, dk, generator=g).to(torch.bfloat16).cuda()
    plan = MidAttentionPlan(torch.tensor([rows - 1], dtype=torch.int32, device="cuda"), 0, 0)
    out, _ = packed_attention(q, ka, va, plan, 1, dk ** -0.5, 1, dv, groups)
    assert torch.isposinf(out[..., 7:11]).all() and torch.isnan(out[..., 40:44]).all()
    va[..., 7:11], va[..., 40:44] = 0.0, 0.0
    ref = ro.attention(to_np(q), to_np(ka), to_np(va), dk ** -0.5, 1, dv)
    rest = [d for d in range(dv) if not 7 <= d < 11 and not 40 <= d < 44]
    err = np.linalg.norm((to_np(out).astype(np.float64) - ref)[..., rest])
    assert err <= 2.0 ** -8 * np.linalg.norm(ref[..., rest])


def test_infinite_values_reach_only_their_feature():
    g = torch.Generator().manual_seed(5)
    ka, va = _rows(1, 1, 200, 128, 128, g)
    va[0, 0, 77, 5], va[0, 0, 199, 9] = float("inf"), float("inf")   # the second past the rows in use
    q = torch.randn(1, 4, 1, 128, generator=g).to(torch.bfloat16).cuda()
    plan = MidAttentionPlan(torch.tensor([150], dtype=torch.int32, device="cuda"), 0, 0)
    out, _ = packed_attention(q, ka, va, plan, 1, 128 ** -0.5, 1, 128, 1)
    assert torch.isposinf(out[..., 5]).all()
    va[0, 0, 77, 5] = 0.0
    ref = ro.attention(to_np(q), to_np(ka)[:, :, :151], to_np(va)[:, :, :151], 128 ** -0.5, 1, 128)
    rest = [d for d in range(128) if d != 5]
    err = np.linalg.norm((to_np(out).astype(np.float64) - ref)[..., rest])
    assert err <= 2.0 ** -8 * np.linalg.norm(ref[..., rest])
