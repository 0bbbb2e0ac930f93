"""Traced launches, whose tasks all take positions of one ring: growing from
capacities that the tasks, or the items of a split task, do not fit."""
import pytest

import cuqc_amd as qc
import cuqc_amd.costmodel as cm
import oracle
from tests.graphs import planted

pytestmark = pytest.mark.gpu

COUNTERS = ["tasks", "branches", "children", "raw_cliques", "w_adj", "sum_t", "sum_t_written", "beyond"]


def rows(feats, subtree):
    return sorted(tuple(f.tolist()) + (int(s),) for f, s in zip(feats, subtree))


@pytest.fixture(scope="module")
def case():
    off, adj = planted(190, 0.20, [30, 26], 0.95, 41)
    ref = oracle.mine(off, adj, 0.9, 13, trace=True)
    return qc.Graph.from_csr(off, adj), ref, rows(ref["trace_feats"], cm.subtree_sizes(ref["trace_parent"], ref["trace_beyond"]))


@pytest.mark.parametrize("workgroups", [0, 3])
@pytest.mark.parametrize("chunk", [-1, 1, 64])
@pytest.mark.parametrize("cap", ["1", "5000"])
def test_growing(case, cap, chunk, workgroups, monkeypatch):
    g, ref, want = case
    monkeypatch.setenv("QCMINE_INITIAL_CAPACITY", cap)
    res = qc.mine(g, 0.9, 13, mode="persistent", lds_tile=64, split_min=1, split_chunk=chunk, workgroups=workgroups, trace=True)
    for k in COUNTERS:
        assert res.stats[k] == ref["stats"][k], k
    assert rows(res.trace_feats, res.trace_subtree) == want
