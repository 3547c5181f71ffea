"""The recent window's unit widths: rows of a multiple of 8 features move in 16-byte units, other widths and
sources whose rows are not 16-byte aligned in 8-byte ones; block sizes around a 256-unit block. The window
holds exactly the appended rows, and a flush moves the rest to the front and clears the vacated rows."""

from __future__ import annotations

import pytest
import torch

from harness import make_pair
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
