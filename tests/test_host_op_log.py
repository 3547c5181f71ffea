"""The op-log's host side without a GPU: row tuples built on first read equal what an eager conversion gives
(lanes of unequal length, empty lanes), replay plans freeze them as nested tuples that compare, hash and slice
as such, and the cache's attribute is a plain one to its callers."""

from __future__ import annotations

import copy
import pickle

import pytest
import torch

from logkv_amd import LogStructuredKVCache
from logkv_amd.log_kv_cache import _HostOpLog, _SemanticReplayPlans

ROWS = torch.arange(2 * 3 * 5 * 4, dtype=torch.int32).view(2, 3, 5, 4)
LENGTHS = torch.tensor([[5, 0, 2], [1, 5, 3]], dtype=torch.int32)
WANT = [[[tuple(r) for r in ROWS[b, g, :LENGTHS[b, g]].tolist()] for g in range(3)] for b in range(2)]
FROZEN = tuple(tuple(map(tuple, batch)) for batch in WANT)


def taken():
    return _HostOpLog(ROWS.clone(), LENGTHS.clone())


def cache():
    """The attribute's owner without its device buffers (a cache proper lives on a GPU)."""
    c = LogStructuredKVCache.__new__(LogStructuredKVCache)
    torch.nn.Module.__init__(c)
    return c


def test_lists_equal_an_eager_conversion_and_are_fresh():
    log = taken()
    first = log.lists()
    assert first == WANT
    first[0][0].clear()
    assert log.lists() == WANT


@pytest.mark.parametrize("source", [taken, lambda: copy.deepcopy(WANT)])
def test_plans_freeze_nested_tuples(source):
    plans, other = _SemanticReplayPlans(source()), _SemanticReplayPlans(source())
    assert plans.host_log == FROZEN and type(plans.host_log) is tuple
    assert plans.host_log == other.host_log and hash(plans.host_log) == hash(other.host_log)
    assert plans.host_log is plans.host_log and plans.host_log[1:] == FROZEN[1:]
    assert [len(lane) for batch in plans.host_log for lane in batch] == LENGTHS.flatten().tolist()


def test_plans_hold_their_own_log_only():
    log = taken()
    plans = _SemanticReplayPlans(log)
    assert plans.holds(log)
    assert plans.holds(plans.host_log) and plans.holds(log)
    assert not plans.holds(None) and not plans.holds(taken()) and not plans.holds(FROZEN)
    rows = copy.deepcopy(WANT)
    plans = _SemanticReplayPlans(rows)
    rows[0][0].clear()
    assert plans.host_log == FROZEN
    assert plans.holds(plans.host_log) and not plans.holds(rows) and not plans.holds(None)
    with pytest.raises(RuntimeError, match="existing CPU op-log"):
        _SemanticReplayPlans(None)


def test_cache_attribute_reads_assigns_and_copies():
    c = cache()
    assert c._last_op_log_host is None
    c._last_op_log_host = taken()
    assert copy.deepcopy(c)._last_op_log_host == WANT
    rows = c._last_op_log_host
    assert rows == WANT and c._last_op_log_host is rows
    c._last_op_log_host = [[[(1, 2, 3, 4)]]]
    assert c._last_op_log_host == [[[(1, 2, 3, 4)]]]
    assert pickle.loads(pickle.dumps(c))._last_op_log_host == [[[(1, 2, 3, 4)]]]
    c._last_op_log_host = None
    assert c._last_op_log_host is None
