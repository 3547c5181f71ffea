"""Chunk attention by split count: one split (below 2048 rows of capacity), a few, and the most there are,
with the packed rows filling the capacity or so few that most splits are empty. Reference: the oracle's
float64 attention.

Tolerance: the output is bf16 (each value within 2^-9) and P enters its product as fp16 (each weight within
2^-11, errors independent over the rows), sums are float32, so the 2-norm error stays below 2^-8 of the
result whatever the split count."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from harness import to_np
from logkv_amd.log_kv_pack import MidAttentionPlan, packed_attention, packed_dim
from oracle import readout as ro
from test_split_counts import forward_splits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,groups,heads,tq,dim,rows,cap,splits", [
    (1, 1, 1, 17, 64, 20, 20000, 16),         # one tile of rows: 15 empty splits
    (1, 2, 4, 40, 128, 200, 6000, 16),        # four tiles
    (1, 1, 1, 17, 64, 20000, 20000, 16),
    (2, 4, 8, 333, 64, 2466, 2466, 8),
    (1, 2, 2, 65, 96, 1100, 4100, 13),        # two tiles a split, the last four empty
    (1, 8, 32, 1000, 128, 900, 2100, 2),
    (1, 2, 2, 40, 128, 2000, 2047, 1),
    (1, 2, 2, 40, 128, 2000, 2048, 8),
    (1, 2, 2, 70, 32, 300, 400, 1),           # values of half the narrow kernel's width
    (2, 8, 8, 1024, 128, 3900, 4000, 4),     # the most splits that the combine for few of them takes
    (2, 4, 16, 333, 64, 6000, 6600, 5),       # and one more
    (2, 2, 4, 300, 96, 5000, 6000, 16),       # values of three quarters of the full kernel's
])
def test_split_counts_match_float64(batch, groups, heads, tq, dim, rows, cap, splits):
    assert forward_splits(batch, groups, heads, tq, dim, cap) == splits
    g = torch.Generator().manual_seed(rows + cap)
    wide = packed_dim(dim, dim)
    ka, va = torch.zeros(batch, groups, cap, wide), torch.zeros(batch, groups, cap, wide)
    ka[:, :, :rows, :dim] = torch.randn(batch, groups, rows, dim, generator=g)
    ka[:, :, :rows, dim] = torch.rand(batch, groups, rows, generator=g) * 4
    va[:, :, :rows, :dim] = torch.randn(batch, groups, rows, dim, generator=g)
    ka[:, :, rows:], va[:, :, rows:] = float("nan"), float("nan")   # rows past the packed ones are not read
    ka, va = ka.to(torch.bfloat16).cuda(), va.to(torch.bfloat16).cuda()
    q = torch.randn(batch, heads, tq, dim, generator=g).to(torch.bfloat16).cuda()
    tail = min(tq, rows)
    plan = MidAttentionPlan(torch.tensor([rows - tail], dtype=torch.int32, device="cuda"), 0, 0)
    causal = tq if tail == tq else 0
    out, _ = packed_attention(q, ka, va, plan, tail, dim ** -0.5, causal, dim, groups)
    ref = ro.attention(to_np(q), to_np(ka)[:, :, :rows], to_np(va)[:, :, :rows], dim ** -0.5, causal, dim)
    err = np.linalg.norm(to_np(out).astype(np.float64) - ref)
    assert err <= 2.0 ** -8 * np.linalg.norm(ref), f"{err:.3e} of {np.linalg.norm(ref):.3e}"
