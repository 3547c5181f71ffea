"""Seeding of free clusters and the orphans' assignment at the edges of the row groups: 1 row up to
several passes of a block, every number of 64-wide feature slices with whole and partial ones, rows
whose strides rule out vector loads, lattice keys whose distances tie, and lanes that mix live and
free clusters. Decisions equal the oracle's exactly."""

from __future__ import annotations

import ctypes as C

import numpy as np
import pytest
import torch

from harness import make_pair, to_np
from logkv_amd._lib import check, lib, ptr, stream_of
from oracle import route
from workloads import Mixture

pytestmark = pytest.mark.gpu

CASES = [
    # dim, rows, live clusters left, lattice keys, padded row stride
    (64, 1, 0, False, 0),
    (128, 7, 0, True, 0),
    (128, 257, 0, True, 0),
    (128, 600, 5, False, 0),
    (128, 300, 3, True, 4),
    (96, 129, 0, False, 0),
    (20, 100, 4, True, 0),
    (192, 130, 0, False, 0),
    (256, 70, 2, True, 4),
]


@pytest.mark.parametrize("dim,rows,live,lattice,pad", CASES)
def test_seeds_and_orphans_match_oracle(dim, rows, live, lattice, pad):
    batch, groups, K = 2, 2, 12
    gpu, ora = make_pair(batch, groups, dim, K, 16, recent=64, flush=64, max_seq=4096, s_h=0.5 * dim)
    dev = gpu.level_k.device
    mix = Mixture(batch, groups, dim, clusters=K, seed=rows)
    if live:   # fill the clusters, then free all but `live` of them
        k, v = mix.rows(64), mix.rows(64)
        pos = torch.arange(64).unsqueeze(0).expand(batch, -1).contiguous()
        gpu.route_and_flush_batch(k.to(dev), v.to(dev), pos.to(dev))
        ora.flush_rows(k.float().numpy(), v.float().numpy(), pos.numpy())
        gpu.alive[:, :, live // 2:K - (live - live // 2)] = False
        ora.alive[:, :, live // 2:K - (live - live // 2)] = False
    if lattice:
        g = torch.Generator().manual_seed(rows)
        k = (torch.randint(0, 2, (batch, groups, rows, dim), generator=g) * 8.0).to(torch.bfloat16)
    else:
        k = mix.rows(rows)
    pos = torch.stack([100 + torch.randperm(rows, generator=torch.Generator().manual_seed(b)) for b in range(batch)])
    counts = torch.tensor([rows, max(1, rows - 3)], dtype=torch.int32)
    padded = torch.zeros(batch, groups, rows, dim + pad, dtype=torch.bfloat16, device=dev)
    k_dev, pos_dev, counts_dev = padded[..., :dim], pos.to(dev), counts.to(dev)
    k_dev.copy_(k)
    view, rv = gpu._ladder_view(), gpu._rows_view(k_dev, k_dev, pos_dev, counts_dev)
    ws = gpu._workspace_for(view, rows)
    assign = torch.empty(batch, groups, rows, dtype=torch.int8, device=dev)
    order = torch.empty(batch, rows, dtype=torch.int32, device=dev)
    check(lib().logkv_attach_assign(C.byref(view), C.byref(rv), C.byref(gpu._params), ptr(ws), ws.numel(),
                                    ptr(assign), ptr(order), stream_of(dev)), "attach")
    torch.cuda.synchronize()
    want, want_order = route.attach_assign(k.float().numpy(), pos.numpy(), counts.numpy(), ora.centroid, ora.alive,
                                           ora.p_hi_c, ora.s_h, ora.eta, ora.g0, ora.lam)
    for b in range(batch):
        n = int(counts[b])
        np.testing.assert_array_equal(to_np(order)[b, :n], want_order[b, :n])
        np.testing.assert_array_equal(to_np(assign)[b, :, :n], want[b, :, :n])
