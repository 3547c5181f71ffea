"""Key-range splits of the attention kernels, read off the workspace sizes the library asks for (no
GPU needed): the count a launch takes is one of those that were fastest on an MI355X, also where a flat
charge per split would trade a few tiles of the walk for gigabytes of float32 partials. Times beside each
case are of the whole call, in us, by count."""

from __future__ import annotations

import ctypes as C

import pytest

from logkv_amd import _lib
from logkv_amd.log_kv_pack import packed_dim


def _args(batch, groups, heads, tq, dim, cap):
    a = _lib.AttentionArgs()
    a.n_batch, a.n_heads, a.n_groups, a.tq, a.dk, a.dv, a.dim = batch, heads, groups, tq, dim, dim, packed_dim(dim, dim)
    a.cap, a.tail, a.causal_tail, a.scale = cap, tq, tq, dim ** -0.5
    return a


def _align256(n):
    return (n + 255) // 256 * 256


def forward_splits(batch, groups, heads, tq, dim, cap):
    """Splits of chunk attention: what its workspace holds beside V's fp16 copy and the lanes' shifts."""
    lanes, nq = batch * groups, heads // groups * tq
    a = _args(batch, groups, heads, tq, dim, cap)
    fixed = _align256(lanes * 64 * 2 * 4) + _align256(lanes * 4) + _align256(lanes * cap * dim * 2)
    part = _lib.lib().logkv_chunk_workspace_bytes(C.byref(a)) - fixed
    return max(1, round(part / (lanes * nq * (dim + 4) * 4)))


def backward_parts(batch, groups, heads, tq, dim, cap):
    """Parts of the key range in the backward, from the statistics' partials and dq's (dq's the larger
    of the two gradients here)."""
    lanes, nq = batch * groups, heads // groups * tq
    a = _args(batch, groups, heads, tq, dim, cap)
    floats = _lib.lib().logkv_chunk_backward_workspace_bytes(C.byref(a)) / 4 - lanes * nq * 2
    one = lanes * nq * 4
    return 1 if floats < lanes * nq * dim else round(floats / (one + lanes * nq * dim))


@pytest.mark.parametrize("shape,fast", [
    ((2, 8, 32, 1920, 128, 12000), {1}),            # 1: 883, 2: 961, 4: 1030, 9: 1229
    ((2, 8, 24, 1400, 128, 12000), {3, 4, 5}),      # 1: 848, 2: 698, 3: 656, 4: 652, 5: 650, 7: 681, 10: 748
    ((1, 8, 32, 1920, 128, 12000), {1}),            # 1: 457, 2: 489, 4: 527
    ((2, 8, 24, 700, 128, 12000), {4, 5, 6, 7}),    # 1: 373, 2: 402, 4: 350, 7: 351, 9: 373
    ((1, 8, 16, 2048, 128, 19000), {2}),            # 1: 681, 2: 408, 4: 429
    ((2, 8, 8, 1024, 128, 4000), {4}),              # 1: 141, 2: 97, 4: 73, 5: 104
    ((2, 4, 16, 333, 64, 6600), {5}),               # 1: 117, 4: 58, 5: 54, 10: 69
    ((2, 4, 8, 333, 64, 2466), {7, 8, 9}),          # 1: 81, 2: 55, 4: 42, 9: 40, 8: 38
    ((1, 2, 2, 40, 128, 2047), {1}),                # one split below 2048 rows of capacity
    ((1, 1, 1, 17, 64, 20000), {16}),               # one block: as many as there are
])
def test_forward_takes_a_fast_count(shape, fast):
    assert forward_splits(*shape) in fast


@pytest.mark.parametrize("shape,fast", [
    ((2, 8, 32, 1920, 128, 12000), {1, 2}),         # 1: 2907, 2: 2942, 4: 2982, 9: 3098
    ((2, 8, 32, 1100, 128, 5000), {3, 4, 5}),       # 1: 1104, 2: 909, 3: 862, 4: 857, 5: 880, 8: 967
    ((2, 8, 24, 1400, 128, 12000), {4, 5, 6, 7, 8}),   # 1: 2459, 2: 1906, 4: 1711, 5: 1663, 6: 1666, 8: 1682, 10: 1735
    ((2, 8, 16, 1024, 128, 13000), {2}),            # 1: 1004, 2: 599, 4: 628
    ((1, 8, 16, 333, 128, 4000), {8, 9}),           # 1: 326, 2: 188, 4: 123, 8: 97, 9: 95
    ((1, 8, 8, 64, 128, 19000), {16}),              # 1: 1557, 8: 235, 16: 145
])
def test_backward_takes_a_fast_count(shape, fast):
    assert backward_parts(*shape) in fast


@pytest.mark.parametrize("batch,groups,heads,tq,dk,dv,cap,splits", [
    (8, 8, 64, 2, 128, 128, 16896, 8),      # 512 blocks over 64 lanes
    (1, 2, 16, 2, 128, 128, 1000, 8),       # one per 128 rows
    (1, 1, 4, 4, 256, 256, 40000, 256),     # values wider than 128: one block per CU
    (1, 1, 4, 1, 4, 128, 40000, 313),
    (600, 1, 1, 1, 64, 64, 5000, 1),
])
def test_decode_workspace_is_what_its_splits_fill(batch, groups, heads, tq, dk, dv, cap, splits):
    a = _args(batch, groups, heads, tq, dv, cap)
    a.dk, a.dim = dk, packed_dim(dk, dv)
    need = _lib.lib().logkv_attention_workspace_bytes(C.byref(a))
    assert need == batch * groups * splits * (heads // groups * tq) * (dv + 2) * 4
