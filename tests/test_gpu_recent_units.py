"""The recent window's unit widths: rows of a multiple of 8 features move in 16-byte units, other widths and
sources whose rows are not 16-byte aligned in 8-byte ones; block sizes around a 256-unit block, and
moves of more units than a launch has threads. The window holds exactly the appended rows, and a flush moves
the rest to the front and clears the vacated rows."""

from __future__ import annotations

import ctypes as C

import pytest
import torch

from harness import make_pair
from logkv_amd import _lib
from logkv_amd._lib import stream_of
from workloads import Mixture

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,pad,sizes", [(64, 0, (31, 33, 64, 60)), (64, 4, (31, 33, 64, 60)), (20, 0, (51, 13, 64, 1)),
                                           (256, 0, (8, 9, 64, 47)), (12, 4, (64, 64, 2, 62))])
def test_window_rows_survive_append_and_shift(dim, pad, sizes):
    recent = 64
    gpu, _ = make_pair(batch=2, groups=3, dim=dim, K=4, B=8, recent=recent, flush=recent, max_seq=1024, s_h=16.0)
    mix, dev = Mixture(2, 3, dim, clusters=4, seed=dim), gpu.level_k.device
    held = [torch.zeros(2, 3, 0, dim, dtype=torch.bfloat16, device=dev) for _ in range(3)]
    start = 0
    for n in sizes:
        rows = []
        for i in range(3):
            t = torch.zeros(2, 3, n, dim + pad, dtype=torch.bfloat16, device=dev)[..., :dim]
            rows.append(t.copy_(mix.rows(n)))
            held[i] = torch.cat([held[i], t], dim=2)
        gpu.add_recent(rows[0], rows[1], k_raw=rows[2], input_pos=torch.arange(start, start + n, device=dev))
        start += n
        count = gpu.recent_count
        for i, name in enumerate(("recent_k", "recent_v", "recent_k_raw")):
            window = getattr(gpu, name)
            assert torch.equal(window[:, :, :count], held[i][:, :, start - count:]), name
            assert int(torch.count_nonzero(window[:, :, count:])) == 0, name
        assert gpu.recent_pos[:, :count].tolist() == [list(range(start - count, start))] * 2


def _window_args(window, rows, pos, recent_pos):
    """RecentArgs of a window and its source rows (keys, raw keys, values; ``[1, lanes, rows, d]`` each)."""
    a = _lib.RecentArgs()
    a.recent_k, a.recent_k_raw, a.recent_v = (w.data_ptr() for w in window)
    a.recent_pos, a.n_batch, a.n_groups, a.cap = recent_pos.data_ptr(), 1, window[0].size(1), window[0].size(2)
    a.dk, a.dkr, a.dv = (w.size(3) for w in window)
    a.k, a.k_raw, a.v = (r.data_ptr() for r in rows)
    (a.k_sb, a.k_sg, a.k_st), (a.kr_sb, a.kr_sg, a.kr_st), (a.v_sb, a.v_sg, a.v_st) = (r.stride()[:3] for r in rows)
    a.pos, a.pos_sb, a.pos_st = pos.data_ptr(), 0, 1
    return a


def _counted(lanes, rows, dim):
    """Rows whose 8-byte units count up from 1, as bf16 bits."""
    n = lanes * rows * dim // 4
    return torch.arange(1, n + 1, device="cuda").view(torch.bfloat16).view(1, lanes, rows, dim)


@pytest.mark.parametrize("lanes,cap,n,widths,take,count", [
    (23_000_000, 2, 1, (4, 4, 4), 1, 2),                             # one unit in each of many blocks
    (1, 22_600_000, 22_600_000, (256, 4, 4), 11_400_000, 22_600_000),   # one lane of many units
])
def test_moves_past_the_threads_of_a_launch(lanes, cap, n, widths, take, count):
    """Moves of more than 2^32 threads at one unit each."""
    print(f"case lanes {lanes} rows {n}", flush=True)
    rows = [_counted(lanes, n, d) for d in widths]
    window = [torch.zeros(1, lanes, cap, d, dtype=torch.bfloat16, device="cuda") for d in widths]
    pos, recent_pos = torch.arange(5, 5 + n, device="cuda"), torch.zeros(1, cap, dtype=torch.int64, device="cuda")
    args, stream = _window_args(window, rows, pos, recent_pos), stream_of(rows[0].device)
    at = count - n
    _lib.check(_lib.lib().logkv_recent_append(C.byref(args), at, n, stream), "append")
    bits = lambda t: t.reshape(lanes, -1).view(torch.int64)
    for w, r in zip(window, rows):
        assert torch.equal(bits(w[:, :, at:count].contiguous()), bits(r))
        assert not at or not bool(bits(w[:, :, :at].contiguous()).any())
    assert torch.equal(recent_pos[0, at:count], pos)
    _lib.check(_lib.lib().logkv_recent_shift(C.byref(args), take, count, stream), "shift")
    left = count - take
    for w, r in zip(window, rows):
        assert torch.equal(bits(w[:, :, :left].contiguous()), bits(r[:, :, n - left:].contiguous()))
        assert not bool(bits(w[:, :, left:].contiguous()).any())
    assert torch.equal(recent_pos[0, :left], pos[n - left:]) and not bool(recent_pos[0, left:].any())
