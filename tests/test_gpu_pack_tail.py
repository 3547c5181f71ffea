"""The rows a decode step adds to a packed prefix (recent rows from an offset on and the current rows) are
the rows a full pack writes there, bit for bit: one row up to several blocks of units, whole and partial
units, with and without an exact pool, current rows given as strided views."""

from __future__ import annotations

import pytest
import torch

from harness import feed, make_pair
from logkv_amd import log_kv_pack as lp
from workloads import Mixture

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,exact,back,cur", [(64, 0, 0, 1), (64, 32, 3, 2), (128, 32, 60, 5), (20, 0, 7, 1),
                                                (256, 0, 1, 0)])
def test_tail_rows_equal_a_full_pack(dim, exact, back, cur):
    gpu, ora = make_pair(batch=2, groups=3, dim=dim, K=4, B=8, recent=64, flush=64, max_seq=2048, s_h=0.25 * dim,
                         exact=exact, span=8, beta_novelty=bool(exact), beta_adaptive=bool(exact))
    mix = Mixture(2, 3, dim, clusters=4, seed=dim + exact)
    for blk in range(3):
        feed(gpu, ora, mix, blk * 64, 64, with_ends=bool(exact))
    k = torch.randn(2, 3, cur, 2 * dim, device="cuda").to(torch.bfloat16)[..., :dim]
    v = torch.randn(2, cur, 3, dim, device="cuda").to(torch.bfloat16).transpose(1, 2)
    packed = lp.packed_dim(dim, dim)
    plan = lp.semantic_mid_attention_plan(gpu)
    full_k, full_v = lp.pack_mid_kv(gpu, plan, k, v, packed)
    rows = full_k.size(2)
    buffers = tuple(torch.full((2, 3, rows + 4, packed), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    start = gpu.recent_count - back
    ka, va = lp.pack_mid_kv(gpu, plan, k, v, packed, buffers=buffers, skip_pooled=True, recent_start=start)
    at = rows - cur - back
    assert torch.equal(ka[:, :, at:], full_k[:, :, at:]) and torch.equal(va[:, :, at:], full_v[:, :, at:])
    for b in buffers:   # nothing else is written
        assert bool((b[:, :, :at] == 7.0).all()) and bool((b[:, :, rows:] == 7.0).all())


@pytest.mark.parametrize("dim,offset,stride,back,cur", [(64, 0, 64, 40, 3), (64, 4, 72, 40, 3), (64, 0, 68, 5, 2),
                                                        (72, 8, 80, 1, 1), (24, 4, 28, 64, 2)])
def test_tail_units_by_alignment(dim, offset, stride, back, cur):
    """Rows that allow 16-byte units and rows (by their first element or their stride) that allow 8-byte ones only."""
    gpu, ora = make_pair(batch=2, groups=3, dim=dim, K=4, B=8, recent=64, flush=64, max_seq=2048, s_h=0.25 * dim)
    mix = Mixture(2, 3, dim, clusters=4, seed=dim + offset)
    for blk in range(2):
        feed(gpu, ora, mix, blk * 64, 64)
    k, v = (torch.randn(2, 3, cur, stride + offset, device="cuda").to(torch.bfloat16).flatten()[offset:].as_strided(
        (2, 3, cur, dim), (3 * cur * stride, cur * stride, stride, 1)) for _ in range(2))
    packed = lp.packed_dim(dim, dim)
    plan = lp.semantic_mid_attention_plan(gpu)
    full_k, full_v = lp.pack_mid_kv(gpu, plan, k, v, packed)
    rows = full_k.size(2)
    buffers = tuple(torch.full((2, 3, rows + 4, packed), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    ka, va = lp.pack_mid_kv(gpu, plan, k, v, packed, buffers=buffers, skip_pooled=True,
                            recent_start=gpu.recent_count - back)
    at = rows - cur - back
    assert torch.equal(ka[:, :, at:], full_k[:, :, at:]) and torch.equal(va[:, :, at:], full_v[:, :, at:])
    for b in buffers:   # nothing else is written
        assert bool((b[:, :, :at] == 7.0).all()) and bool((b[:, :, rows:] == 7.0).all())
