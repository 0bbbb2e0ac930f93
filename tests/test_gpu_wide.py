"""Tasks above 64 vertices: the layout in LDS and the one in the wave's HBM
slab, on both sides of the size where one passes to the other, in every form,
against the oracle (all counters, the raw multiset and the maximal sets)."""
import sys

import pytest

import cuqc_amd as qc
import oracle
from tests.graphs import complete, planted

pytestmark = pytest.mark.gpu

COUNTERS = ["tasks", "branches", "children", "raw_cliques", "w_adj", "sum_t", "sum_t_written", "sum_clique_len",
            "beyond"]

# (builder, gamma, min_size, window): root windows of one level keep the
# largest tasks to what the oracle does in a second.  "l2_13bit": the items of
# the last branches are small, while their vertices still carry the 2-hop
# counts of the whole root (4,300 vertices, 13 bits).
CASES = {
    "k130_odd_row_words": (lambda: complete(130), 0.95, 60, (0, -1, -1)),
    "er190": (lambda: planted(190, 0.20, [30, 26], 0.95, 41), 0.9, 13, (0, -1, -1)),
    "er200_g05": (lambda: planted(200, 0.10, [14], 0.9, 42), 0.6, 8, (-40, -1, 3)),
    "er700": (lambda: planted(700, 0.15, [40], 0.95, 43), 0.6, 20, (0, 6, 1)),
    "er960": (lambda: planted(960, 0.12, [40], 0.95, 44), 0.6, 20, (0, 4, 1)),
    "er1030": (lambda: planted(1030, 0.12, [40], 0.95, 45), 0.6, 20, (0, 4, 1)),
    "er2100": (lambda: planted(2100, 0.08, [40], 0.95, 46), 0.6, 20, (0, 3, 1)),
    "l2_13bit": (lambda: planted(4300, 0.03, [40], 0.95, 47), 0.5, 8, (-220, -1, 1)),
}


@pytest.fixture(scope="module")
def refs():
    out = {}
    for name, (build, gamma, ms, win) in CASES.items():
        off, adj = build()
        g = qc.Graph.from_csr(off, adj)
        b, e, d = win
        if b < 0:
            n = oracle.mine(off, adj, gamma, ms, max_depth=0)["stats"]["branches"]
            b, e = max(0, n + b), n
        ref = oracle.mine(off, adj, gamma, ms, root_begin=b, root_end=e, max_depth=d, threads=8)
        out[name] = (g, gamma, ms, (b, e, d), ref)
    return out


FORMS = {
    "plain": dict(mode="plain"),
    "fifo": dict(mode="persistent"),
    "small_lds": dict(mode="persistent", lds_tile=64, lds_wide=-1),
    "wide_lds": dict(mode="persistent", lds_wide=1024),
    "items": dict(mode="persistent", lds_tile=64, split_chunk=3, split_min=1),
    "unsplit": dict(mode="persistent", split_chunk=-1),
    "static": dict(mode="persistent", scheduling=1),
    "few_waves": dict(mode="persistent", workgroups=3),
    "cost": dict(mode="persistent", order="cost"),
    "trace": dict(mode="persistent", trace=True),
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("form", list(FORMS))
def test_forms(refs, name, form):
    g, gamma, ms, win, ref = refs[name]
    print(f"[gpu] wide {name} {form}: {ref['stats']['tasks']} tasks", flush=True)
    sys.stdout.flush()
    kw = dict(FORMS[form])
    if kw.get("order") == "cost":
        kw["cost_model"] = qc.CostModel.create(seed=3)
    res = qc.mine(g, gamma, ms, window=win, **kw)
    for k in COUNTERS:
        assert res.stats[k] == ref["stats"][k], k
    assert oracle.canon(res.raw) == oracle.canon(ref["raw"])
    assert res.maximal_sorted_tuples() == oracle.nonmax(ref["raw"])


# the level-synchronous form: tasks split into items across launches, against
# the unsplit form and with a caller's capacities (where nothing is split)
PLAIN = {
    "items_of_1": dict(split_chunk=1, split_min=1, lds_tile=64),
    "items_of_5": dict(split_chunk=5, lds_tile=64),
    "unsplit": dict(split_chunk=-1),
    "static": dict(scheduling=1),
    "capacities": dict(task_capacity=1 << 23, clique_capacity=1 << 22),
}


@pytest.mark.parametrize("name", ["er190", "er200_g05", "er960", "l2_13bit"])
@pytest.mark.parametrize("form", list(PLAIN))
def test_plain_splits(refs, name, form):
    g, gamma, ms, win, ref = refs[name]
    print(f"[gpu] plain {name} {form}", flush=True)
    res = qc.mine(g, gamma, ms, window=win, mode="plain", **PLAIN[form])
    for k in COUNTERS:
        assert res.stats[k] == ref["stats"][k], k
    assert oracle.canon(res.raw) == oracle.canon(ref["raw"])


def test_plain_clique_stream_overflows(refs, monkeypatch):
    """A launch whose raw sets do not fit the stream is made again with half the
    tasks: 65,536 vertices hold what two tasks of this graph emit, not a launch's."""
    g, gamma, ms, win, ref = refs["er190"]
    assert ref["stats"]["sum_clique_len"] > 3 * 65536
    monkeypatch.setenv("QCMINE_INITIAL_CAPACITY", "8192")
    res = qc.mine(g, gamma, ms, window=win, mode="plain")
    for k in COUNTERS:
        assert res.stats[k] == ref["stats"][k], k
    assert oracle.canon(res.raw) == oracle.canon(ref["raw"])
