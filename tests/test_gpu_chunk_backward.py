"""The matrix-core backward of packed attention at the edges of its tiles and splits: query rows around
the 256-row blocks and 64-row tiles, gradient rows around the 128-row blocks (fewer and more than the
queries), key ranges from one tile to many parts, every head dim, and rows whose strides rule out vector
loads. Reference: the oracle's float64 gradient.

Tolerance: outputs are bf16 (each within 2^-9 of its float32 value), P and dS enter their products as
two bf16 parts (2^-16), and the sums are float32, so the 2-norm error stays below 2^-8 of the result."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from harness import to_np
from logkv_amd.log_kv_pack import MidAttentionPlan, packed_attention, packed_attention_backward, packed_dim
from oracle import readout as ro

pytestmark = pytest.mark.gpu

CASES = [
    # batch, groups, heads, tq, dk, dv, rows, causal, grad_rows, padded feature stride
    (1, 1, 1, 1, 64, 64, 1, 1, 1, 0),
    (1, 2, 2, 65, 64, 64, 130, 65, 65, 0),
    (2, 1, 3, 100, 128, 128, 700, 100, 100, 0),
    (1, 2, 4, 128, 128, 128, 2049, 128, 128, 4),
    (1, 1, 2, 129, 96, 96, 1000, 129, 129, 3),
    (1, 1, 1, 257, 72, 64, 400, 257, 257, 0),
    (2, 2, 2, 31, 8, 32, 333, 0, 333, 1),
    (1, 1, 4, 16, 128, 64, 300, 16, 300, 0),
]


@pytest.mark.parametrize("batch,groups,heads,tq,dk,dv,rows,causal,grad_rows,pad", CASES)
def test_backward_matches_float64(batch, groups, heads, tq, dk, dv, rows, causal, grad_rows, pad):
    g = torch.Generator().manual_seed(rows)
    dim, cap = packed_dim(dk, dv), rows + 5
    ka, va = torch.zeros(batch, groups, cap, dim), torch.zeros(batch, groups, cap, dim)
    ka[..., :dk] = torch.randn(batch, groups, cap, dk, generator=g)
    ka[..., dk] = torch.rand(batch, groups, cap, generator=g) * 4
    ka[:, :, :rows // 4, dk] = torch.where(torch.rand(batch, groups, rows // 4, generator=g) < 0.3, -10000.0,
                                           ka[:, :, :rows // 4, dk])
    va[..., :dv] = torch.randn(batch, groups, cap, dv, generator=g)
    ka, va = ka.to(torch.bfloat16).cuda(), va.to(torch.bfloat16).cuda()

    def strided(*shape):   # contiguous features, rows padded by `pad` elements
        x = torch.randn(*shape[:-1], shape[-1] + pad, generator=g).to(torch.bfloat16).cuda()
        return x[..., :shape[-1]]

    q, dout = strided(batch, heads, tq, dk), strided(batch, heads, tq, dv)
    scale = dk ** -0.5
    plan = MidAttentionPlan(torch.tensor([rows - tq], dtype=torch.int32, device="cuda"), 0, 0)
    if grad_rows > tq:   # every row a gradient row: all of them in the tail
        plan, tail = MidAttentionPlan(torch.zeros(1, dtype=torch.int32, device="cuda"), 0, 0), rows
    else:
        tail = tq
    out, _ = packed_attention(q, ka, va, plan, tail, scale, causal, dv, groups)
    got = packed_attention_backward(q, ka, va, out, dout, plan, tail, scale, causal, dv, groups, grad_rows)
    ref = ro.attention_grad(to_np(q), to_np(ka)[:, :, :rows], to_np(va)[:, :, :rows], scale, causal, dv, to_np(dout),
                            grad_rows)
    for x, r, name in zip(got, ref, ("dq", "dk", "dv")):
        err = np.linalg.norm(to_np(x).astype(np.float64) - r)
        # A single visible row has p = 1 and dS = 0 exactly up to float32: an absolute floor for the zeros.
        assert err <= 2.0 ** -8 * np.linalg.norm(r) + 1e-6 * np.sqrt(r.size), f"{name}: {err:.3e} of {np.linalg.norm(r):.3e}"
