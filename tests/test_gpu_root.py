"""The root on the device: filter, peel, core ids, rows and Q order, against
the oracle (all counters of the search, which read every one of them)."""
import numpy as np
import pytest

import cuqc_amd as qc
import oracle
from tests.graphs import csr_from_edges

pytestmark = pytest.mark.gpu

COUNTERS = ["tasks", "branches", "children", "raw_cliques", "w_adj", "sum_t", "sum_t_written", "sum_clique_len",
            "beyond"]
DEVICE_MIN = 32768  # vertices from which the filter and the peel run on the device


def communities(n, seed, hubs=0, chain=0, size=(14, 30), keep=0.9, groups=40):
    """Dense groups, sparse noise, hubs with many neighbours of degree one, and
    a chain that the peel takes apart from one end, a vertex a round."""
    rng = np.random.default_rng(seed)
    edges = set()
    for _ in range(groups):
        k = int(rng.integers(*size))
        mem = rng.choice(n - chain, k, replace=False)
        for i in range(k):
            for j in range(i):
                if rng.random() < keep:
                    edges.add((int(min(mem[i], mem[j])), int(max(mem[i], mem[j]))))
    for u, v in rng.integers(0, n - chain, (2 * n, 2)):
        if u != v:
            edges.add((int(min(u, v)), int(max(u, v))))
    for h in range(hubs):
        for v in rng.choice(n - chain, 5000, replace=False):
            if v != h:
                edges.add((int(min(h, v)), int(max(h, v))))
    # w wide: vertex i of the chain has the w before and the w after it
    for i in range(n - chain, n):
        for j in range(i + 1, min(i + 8, n)):
            edges.add((i, j))
    return csr_from_edges(n, list(edges))


# (n, seed, gamma, min_size, depth, extra): both sides of the device's smallest graph,
# rounds beyond the device's limit (chain), hubs above a segment, an empty core,
# min_size with thr < min_size - 1 (second neighbours looked up)
CASES = {
    "below": (DEVICE_MIN - 1, 61, 0.8, 9, 3, {}),
    "at": (DEVICE_MIN, 61, 0.8, 9, 3, {}),
    "odd": (DEVICE_MIN + 4097, 62, 0.7, 10, -1, dict(hubs=3)),
    "chain": (DEVICE_MIN + 65, 63, 0.8, 10, 3, dict(chain=900)),
    "empty": (DEVICE_MIN + 1, 64, 0.9, 60, -1, {}),
    "g05": (DEVICE_MIN + 63, 65, 0.5, 14, 1, dict(hubs=2)),
}


@pytest.mark.parametrize("name", list(CASES))
def test_root(name):
    n, seed, gamma, ms, depth, kw = CASES[name]
    off, adj = communities(n, seed, **kw)
    ref = oracle.mine(off, adj, gamma, ms, max_depth=depth, threads=8)
    print(f"[gpu] root {name}: {ref['stats']['tasks']} tasks", flush=True)
    res = qc.mine(qc.Graph.from_csr(off, adj), gamma, ms, window=(0, -1, depth))
    for k in COUNTERS:
        assert res.stats[k] == ref["stats"][k], k
    assert oracle.canon(res.raw) == oracle.canon(ref["raw"])


def test_few_second_neighbours():
    """Cliques of exactly min_size - 1 vertices pass the degree threshold and
    have too few second neighbours: the core is then taken on the host."""
    n = DEVICE_MIN + 10
    edges = [(b + i, b + j) for b in range(0, 3000, 10) for i in range(9) for j in range(i)]
    edges += [(4000 + b + i, 4000 + b + j) for b in range(0, 300, 30) for i in range(12) for j in range(i)]
    off, adj = csr_from_edges(n, edges)
    gamma, ms = 0.7, 10
    ref = oracle.mine(off, adj, gamma, ms)
    res = qc.mine(qc.Graph.from_csr(off, adj), gamma, ms)
    assert res.stats["root_size"] == 120
    for k in COUNTERS:
        assert res.stats[k] == ref["stats"][k], k
    assert oracle.canon(res.raw) == oracle.canon(ref["raw"])
