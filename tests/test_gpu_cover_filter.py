"""RemoveNonMax on lists long enough for the cover filter (8,192 raw sets):
several copies of a graph in one batch (equal sets in different instances,
equal sets of one length inside one), and the plain form's host sets."""
import sys

import pytest

import cuqc_amd as qc
import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cfg0():
    graphs = [qc.Graph.generate(0, s) for s in (1, 7)]
    refs = []
    for g in graphs:
        off, adj = g.csr()
        refs.append(oracle.mine(off, adj, g.gamma, g.min_size))
    return graphs, refs


# 2 copies stay below the filter's 8,192 sets, 3 pass it, 9 hold equal sets
# in nine key ranges
@pytest.mark.parametrize("copies", [1, 2, 3, 9])
def test_batch_of_equal_graphs(cfg0, copies):
    graphs, refs = cfg0
    gs = [graphs[i % 2] for i in range(copies)]
    print(f"[gpu] cover filter, batch of {copies}", flush=True)
    sys.stdout.flush()
    res = qc.mine_batch(gs, [g.gamma for g in gs], [g.min_size for g in gs])
    for i, r in enumerate(res):
        ref = refs[i % 2]
        assert r.stats["raw_cliques"] == ref["stats"]["raw_cliques"]
        assert r.maximal_sorted_tuples() == oracle.nonmax(ref["raw"])


@pytest.mark.parametrize("mode", ["plain", "persistent"])
def test_many_raw_sets(mode):
    """gamma 0.7 on a G(90, 0.3) with a planted set: 30,000 raw sets of which
    more than half are maximal, so the rounds give up early."""
    from tests.graphs import planted
    off, adj = planted(90, 0.30, [14], 0.95, 21)
    ref = oracle.mine(off, adj, 0.7, 7, threads=4)
    print(f"[gpu] cover filter, {len(ref['raw'])} raw sets, {mode}", flush=True)
    sys.stdout.flush()
    assert len(ref["raw"]) > 8192
    want = oracle.nonmax(ref["raw"])
    assert len(want) > 64
    res = qc.mine(qc.Graph.from_csr(off, adj), 0.7, 7, mode=mode)
    assert res.stats["raw_cliques"] == len(ref["raw"])
    assert res.maximal_sorted_tuples() == want
