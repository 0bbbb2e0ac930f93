"""Subtrees of at most 64 vertices run in registers: full searches whose
tasks cross 64 vertices, in every form, against the oracle (all counters, the
raw multiset and the maximal sets)."""
import sys

import pytest

import cuqc_amd as qc
import oracle
from tests.graphs import complete, planted

pytestmark = pytest.mark.gpu

COUNTERS = ["tasks", "branches", "children", "raw_cliques", "w_adj", "sum_t", "sum_t_written", "sum_clique_len",
            "beyond"]

# (builder, gamma, min_size): tasks just below and above 64 vertices, lookahead
# hits on all of them (complete graphs), min_size above 64 (every mindeg beyond
# the lane table), stale and negative exdegs (gamma 0.5), long failing removals
CASES = {
    "k64": (lambda: complete(64), 0.9, 5),
    "k65": (lambda: complete(65), 1.0, 60),
    "k66_ms66": (lambda: complete(66), 0.9, 66),
    "er66_dense": (lambda: planted(66, 0.75, [20], 0.97, 31), 0.95, 26),
    "er64_g05": (lambda: planted(64, 0.20, [9], 0.9, 32), 0.5, 9),
    "er63_g06": (lambda: planted(63, 0.25, [12], 0.9, 33), 0.6, 9),
    "er140_planted": (lambda: planted(140, 0.10, [33, 30], 0.93, 34), 0.85, 14),
    "er300": (lambda: planted(300, 0.05, [24, 22, 20], 0.95, 35), 0.9, 11),
}


@pytest.fixture(scope="module")
def refs():
    out = {}
    for name, (build, gamma, ms) in CASES.items():
        off, adj = build()
        out[name] = (off, adj, gamma, ms, oracle.mine(off, adj, gamma, ms, threads=4))
    return out


FORMS = {
    "plain": dict(mode="plain"),
    "plain_tile64": dict(mode="plain", lds_tile=64),
    "fifo": dict(mode="persistent"),
    "fifo_small_lds": dict(mode="persistent", lds_tile=64, lds_wide=-1),
    "static": dict(mode="persistent", scheduling=1),
    "one_wave": dict(mode="persistent", workgroups=1),
    "cost": dict(mode="persistent", order="cost"),
    "replays": dict(mode="persistent", replays=3),
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("form", list(FORMS))
def test_forms(refs, name, form):
    off, adj, gamma, ms, ref = refs[name]
    print(f"[gpu] tiny {name} {form}: {ref['stats']['tasks']} tasks", flush=True)
    sys.stdout.flush()
    kw = dict(FORMS[form])
    if kw.get("order") == "cost":
        kw["cost_model"] = qc.CostModel.create(seed=3)
    res = qc.mine(qc.Graph.from_csr(off, adj), gamma, ms, **kw)
    for k in COUNTERS:
        assert res.stats[k] == ref["stats"][k], k
    assert oracle.canon(res.raw) == oracle.canon(ref["raw"])
    assert res.maximal_sorted_tuples() == oracle.nonmax(ref["raw"])


@pytest.mark.parametrize("cap", ["1", "64", "4096"])
def test_growing_from_small_capacities(refs, monkeypatch, cap):
    off, adj, gamma, ms, ref = refs["er140_planted"]
    monkeypatch.setenv("QCMINE_INITIAL_CAPACITY", cap)
    res = qc.mine(qc.Graph.from_csr(off, adj), gamma, ms, mode="persistent")
    assert res.stats["w_adj"] == ref["stats"]["w_adj"]
    assert oracle.canon(res.raw) == oracle.canon(ref["raw"])


def test_fixed_clique_capacity_is_the_raw_sets_size(refs):
    """The waves take refs and slots of the clique stream several at a time;
    a capacity that holds the raw sets exactly is enough, one vertex less is not."""
    off, adj, gamma, ms, ref = refs["er140_planted"]
    g = qc.Graph.from_csr(off, adj)
    need = max(ref["stats"]["sum_clique_len"], 8 * (ref["stats"]["raw_cliques"] - 1024))
    res = qc.mine(g, gamma, ms, mode="persistent", clique_capacity=need)
    assert len(res.raw) == ref["stats"]["raw_cliques"]
    with pytest.raises(qc.QCError) as e:
        qc.mine(g, gamma, ms, mode="persistent", clique_capacity=ref["stats"]["sum_clique_len"] - 1)
    assert e.value.code == qc.QC_EOVERFLOW
