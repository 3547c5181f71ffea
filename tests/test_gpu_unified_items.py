"""The Lance-Williams phase on both sides of its item rule: with 8 merges or more per item the mirrors go
through LDS, with fewer they are written as the rows are computed. Flushes whose rounds fall on both sides (the
oracle reducer's own rounds say so), with full items, the least staged ones and a last item that is not full;
state bit for bit after every flush."""

from __future__ import annotations

import pytest
import torch

from harness import compare_state
from oracle import unified as U
from test_gpu_unified import _pair
from workloads import Mixture

pytestmark = pytest.mark.gpu

WAVES, COLUMNS, STAGED, MOST = 256, 128, 8, 16   # a lane's waves, columns of an item, merges of a staged / a full item


@pytest.mark.parametrize("rows", [1500, 2000, 3000])
def test_rounds_on_both_sides_of_the_staging_rule(rows, monkeypatch):
    print(f"case rows={rows}", flush=True)
    rounds, merge = [], U.Reducer._merge

    def counted(self, a, *rest):
        merge(self, a, *rest)
        rounds.append((len(a), int(self.alive.sum())))

    monkeypatch.setattr(U.Reducer, "_merge", counted)
    gpu, ora = _pair(1, 2, 32, 12, 16, rows, 4 * rows, 16.0)
    mix = Mixture(1, 2, 32, clusters=14, seed=rows, drift_every=rows)
    dev = gpu.level_k.device
    for i in range(2):
        k, v = mix.rows(rows), mix.rows(rows)
        pos = torch.arange(i * rows, (i + 1) * rows).unsqueeze(0)
        gpu.route_and_flush_batch(k.to(dev), v.to(dev), pos.to(dev))
        ora.flush_rows(k.float().numpy(), v.float().numpy(), pos.numpy())
        torch.cuda.synchronize()
        bad = compare_state(gpu, ora)
        assert not bad, f"flush {i}: " + "; ".join(bad)
    per_item = [(n, max(1, min(MOST, n * -(-live // COLUMNS) // WAVES))) for n, live in rounds]
    print(per_item)
    assert any(r < STAGED for _, r in per_item) and any(r >= STAGED for _, r in per_item)
    assert any(r >= STAGED and n % r for n, r in per_item), "no staged item short of its merges"
    assert rows != 3000 or any(r == MOST for _, r in per_item), "no full item"
