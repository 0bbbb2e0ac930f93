"""A window near the end of a large root: the record that is left is small
enough for the LDS, while its vertices carry the 2-hop counts of the whole root
(more than 65,536 vertices), which a child's order compares."""
import numpy as np
import pytest

import cuqc_amd as qc

pytestmark = pytest.mark.gpu

COUNTERS = ["tasks", "branches", "children", "raw_cliques", "w_adj", "sum_t", "sum_t_written", "sum_clique_len",
            "beyond"]
GAMMA, MIN_SIZE = 0.5, 20


def hubs_over_ring(n: int = 66_000, hubs: int = 1_000, seed: int = 5):
    """`hubs` vertices joined with probability 0.35, each also to 0-200 vertices
    of a ring in which everyone has 12 neighbours: all n are in the root, the
    hubs last, with 2-hop counts of about 20,000 to 30,000."""
    rng = np.random.default_rng(seed)
    name = rng.permutation(n)
    ring = n - hubs
    iu = np.triu_indices(hubs, 1)
    m = rng.random(len(iu[0])) < 0.35
    parts = [np.stack([iu[0][m], iu[1][m]], 1)]
    at = np.arange(ring)
    for d in range(1, 7):
        parts.append(np.stack([hubs + at, hubs + (at + d) % ring], 1))
    w = rng.integers(0, 201, hubs)
    parts.append(np.stack([np.repeat(np.arange(hubs), w), hubs + rng.integers(0, ring, w.sum())], 1))
    e = name[np.concatenate(parts)]
    key = np.unique(np.concatenate([e[:, 0] * n + e[:, 1], e[:, 1] * n + e[:, 0]]))
    off = np.zeros(n + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(key // n, minlength=n))
    return off, (key % n).astype(np.uint32)


# the oracle's counters by window (oracle.mine on the graph above, 45 to 55 s each,
# so they are kept here; there are no raw sets): (branches left after the window's
# start, branches, max_depth) -> COUNTERS
BRANCHES = 65_417
REF = {
    (180, 1, 2): [533, 153655, 143890, 0, 4934783837, 225329, 29971975, 0, 143358],
    (180, 3, 1): [4, 1662, 1599, 0, 125173710, 67689, 476460, 0, 1596],
    (420, 1, 2): [774, 315593, 302014, 0, 9943448160, 389859, 86927222, 0, 301241],
}


@pytest.fixture(scope="module")
def graph():
    return qc.Graph.from_csr(*hubs_over_ring())


FORMS = {
    "plain": dict(mode="plain"),
    "plain_unsplit": dict(mode="plain", split_chunk=-1),
    "fifo": dict(mode="persistent"),
    "unsplit": dict(mode="persistent", split_chunk=-1),
    "unsplit_wide": dict(mode="persistent", split_chunk=-1, lds_wide=1024),
    "static_unsplit": dict(mode="persistent", scheduling=1, split_chunk=-1),
}


# (the covered block stays too: 180 branches leave 763 vertices, 420 leave 1,003)
@pytest.mark.parametrize("left,count,depth", list(REF))
@pytest.mark.parametrize("form", list(FORMS))
def test_two_hop_counts_of_the_whole_root(graph, left, count, depth, form, monkeypatch):
    monkeypatch.setenv("QCMINE_ROOT_CUT_WORDS", "1")
    print(f"[gpu] cut root {left} {count} {depth} {form}", flush=True)
    b = BRANCHES - left
    res = qc.mine(graph, GAMMA, MIN_SIZE, window=(b, b + count, depth), **FORMS[form])
    assert res.stats["root_size"] == 66_000 and res.stats["root_branches"] == BRANCHES
    assert [res.stats[k] for k in COUNTERS] == REF[left, count, depth]
