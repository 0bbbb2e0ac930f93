"""The mining calls whose time matters, as a user's program makes them.

A case names a graph of the repository's generator (config, graph_seed,
instance), the search window, the execution form and its options; the seed
relabels the graph's vertices at random.  A relabelled graph is another input
(other ids, other ties in every vertex order, other sets in the answer) whose
search tree keeps its size within a few tens of percent, whereas graphs of
different generator seeds differ by orders of magnitude in the same window.

A pass returns the maximal sets (one offsets array, one vertex array, graph
after graph, in buffers of the state that are larger than any answer) and the
counters of the search, which do not depend on how the work was scheduled.
The raw sets come back to the program inside the result; their order is
unspecified, so they are not compared here.
"""
from __future__ import annotations

import numpy as np
import torch

import cuqc_amd as qc
from cuqc_amd import costmodel

COUNTERS = ("tasks", "branches", "children", "raw_cliques", "max_cliques", "sum_t", "sum_t_written",
            "sum_clique_len", "root_size", "beyond", "root_branches", "w_adj")

# room for the maximal sets of any case, and for their vertices
MOST_SETS, MOST_VERTS = 1 << 17, 1 << 21

OPTIONS = ("mode", "scheduling", "order", "lds_tile", "lds_wide", "mid_tile", "split_chunk", "split_min")


def listed() -> list[dict]:
    return [
        # the smallest calls: one small graph searched to the end, where the
        # fixed costs of a call and the depth of the tree count.  The command
        # line's default form ...
        dict(name="small graph", kind="mine", config=0, graph_seed=1, mode="persistent"),
        # ... and the Python binding's default form, one launch per level
        dict(name="small graph plain", kind="mine", config=0, graph_seed=7, mode="plain"),
        # the headline: root branches of an 8,000-gene co-expression network
        # (R = 5,489) that lead to tasks of 200-1,000 vertices
        dict(name="co-expression", kind="mine", config=1, graph_seed=2, begin=3600, end=3612, depth=3,
             mode="persistent"),
        # the same network, cost-ordered with a schedule as the autotuner
        # picks it, more branches of fewer levels
        dict(name="co-expression cost", kind="mine", config=1, graph_seed=2, begin=3560, end=3597, depth=2,
             mode="persistent", order="cost", lds_wide=512, mid_tile=512, split_chunk=128),
        # the same network under the command line's static scheduling toggle
        dict(name="co-expression static", kind="mine", config=1, graph_seed=2, begin=3589, end=3600, depth=2,
             mode="persistent", scheduling=1),
        # the same network level by level
        dict(name="co-expression plain", kind="mine", config=1, graph_seed=2, begin=3606, end=3612, depth=2,
             mode="plain"),
        # a sparse power-law network of 100,000 vertices at full depth: more
        # than half a million tasks of about 30 vertices
        dict(name="power law", kind="mine", config=2, graph_seed=3, begin=9263, end=9273, mode="persistent"),
        # the first branches of the same network's root: tasks of thousands
        # of vertices, where every full search begins
        dict(name="power law first", kind="mine", config=2, graph_seed=3, begin=0, end=3, depth=2,
             mode="persistent"),
        # the largest graph, 1,000,000 vertices: its root (R = 70,088) and a
        # window of large tasks
        dict(name="power law 1M", kind="mine", config=4, graph_seed=5, begin=41828, end=41846, depth=3,
             mode="persistent"),
        # one graph of 700 vertices searched to the end: 1.5 million tasks
        dict(name="full search", kind="mine", config=3, graph_seed=4, instance=15, mode="persistent"),
        # many graphs of 500-20,000 vertices, each with its own gamma and
        # min_size, through one call
        dict(name="batch of 61", kind="batch", config=3, graph_seed=4, instance=0, count=61, begin=-32, depth=2),
        # RemoveNonMax on a program's own sets
        dict(name="remove non-maximal", kind="nonmax", groups=301, sets=20011),
    ]


def draw(rng) -> dict:
    kind = rng.choice(["small", "co-expression", "co-expression", "power law", "batch", "batch", "nonmax"])

    def spread(lo, hi):  # spread over the logarithm
        return int(round(lo * (hi / lo) ** rng.random()))

    if kind == "small":
        return dict(kind="mine", config=0, graph_seed=rng.randrange(2, 1 << 30),
                    mode=rng.choice(["plain", "persistent", "persistent"]), scheduling=rng.randrange(2),
                    lds_tile=rng.choice([64, 128]))
    if kind == "co-expression":
        depth = rng.choice([2, 2, 3])
        begin = rng.randrange(3604, 3611) if depth == 3 else rng.randrange(500, 3600)
        return dict(kind="mine", config=1, graph_seed=2, begin=begin, end=begin + spread(2, 5 if depth == 3 else 24),
                    depth=depth, mode="persistent", scheduling=rng.choice([0, 0, 1]),
                    lds_wide=rng.choice([0, 256, 512]), mid_tile=rng.choice([0, 512]),
                    split_chunk=rng.choice([0, 32, 128]))
    if kind == "power law":
        begin = rng.randrange(3000, 11000)
        return dict(kind="mine", config=2, graph_seed=3, begin=begin, end=begin + spread(2, 30), depth=3,
                    mode="persistent")
    if kind == "batch":
        return dict(kind="batch", config=3, graph_seed=rng.randrange(5, 1 << 20), instance=rng.randrange(256),
                    count=spread(3, 60), begin=-spread(4, 32), depth=2)
    return dict(kind="nonmax", groups=spread(4, 400), sets=spread(50, 20000))


_BASE: dict = {}
_MODEL: list = []


def _base(config: int, graph_seed: int, instance: int):
    """The generator's graph: offsets, adjacency, gamma, min_size (the large
    ones take seconds to generate, so they are kept)."""
    key = (config, graph_seed, instance)
    if key not in _BASE:
        g = qc.Graph.generate(config, graph_seed, instance)
        off, adj = g.csr()
        got = (off, adj, g.gamma, g.min_size)
        if len(adj) < 1 << 20:
            return got
        _BASE[key] = got
    return _BASE[key]


def _relabelled(config: int, graph_seed: int, instance: int, seed: int):
    """A handle on the generator's graph with its vertices renamed by a random
    permutation, as a program builds one from its own CSR arrays."""
    off, adj, gamma, min_size = _base(config, graph_seed, instance)
    n = len(off) - 1
    dev = "cuda" if len(adj) >= 1 << 20 else "cpu"
    perm = torch.from_numpy(np.random.default_rng((seed, config, instance)).permutation(n)).to(dev)
    deg = torch.from_numpy(np.diff(off).astype(np.int64)).to(dev)
    key = torch.repeat_interleave(perm, deg) * n + perm[torch.from_numpy(adj.astype(np.int64)).to(dev)]
    key = torch.sort(key).values
    new_adj = (key % n).cpu().numpy().astype(np.uint32)
    new_deg = torch.zeros(n, dtype=torch.int64, device=dev)
    new_deg[perm] = deg
    new_off = np.zeros(n + 1, np.uint64)
    new_off[1:] = torch.cumsum(new_deg, 0).cpu().numpy()
    return qc.Graph.from_csr(new_off, new_adj), gamma, min_size


def _model():
    """A cost model trained on the traces of small graphs, kept by a program."""
    if not _MODEL:
        graphs = [qc.Graph.generate(0, s) for s in (1, 11)]
        _MODEL.append(costmodel.train_from_traces([(g, g.gamma, g.min_size, None) for g in graphs], steps=100)[0])
    return _MODEL[0]


def _sets(case: dict, seed: int) -> list[np.ndarray]:
    """Raw sets as a search emits them: most members of one of a few hundred
    dense groups of 30-80 vertices, many of them twice or inside another."""
    rng = np.random.default_rng(seed)
    perm = rng.permutation(100_000).astype(np.uint32)
    cut = np.concatenate(([0], np.cumsum(rng.integers(30, 81, case["groups"]))))
    groups = [perm[cut[i]:cut[i + 1]] for i in range(case["groups"])]
    which = rng.integers(0, case["groups"], case["sets"])
    lost = rng.integers(0, 7, case["sets"])
    out = []
    for g, k in zip(which, lost):
        m = groups[g]
        keep = np.ones(len(m), bool)
        keep[rng.integers(0, len(m), k)] = False
        out.append(m[keep])
    return out


def prepare(case: dict, seed: int) -> dict:
    out = dict(offsets=np.zeros(MOST_SETS + 1, np.int64), verts=np.zeros(MOST_VERTS, np.uint32))
    if case["kind"] == "nonmax":
        return dict(kind="nonmax", sets=_sets(case, seed), out=out)
    opts = {k: case[k] for k in OPTIONS if k in case}
    if case.get("order") == "cost":
        opts["cost_model"] = _model()
    window = (case.get("begin", 0), case.get("end", -1), case.get("depth", -1))
    first, count = case.get("instance", 0), case.get("count", 1)
    made = [_relabelled(case["config"], case["graph_seed"], first + i, seed) for i in range(count)]
    return dict(kind=case["kind"], graphs=[m[0] for m in made], gammas=[m[1] for m in made],
                min_sizes=[m[2] for m in made], window=window, opts=opts, out=out)


def _flat(sets: list[np.ndarray], out: dict) -> dict:
    """The sets one after another at the start of the state's buffers."""
    off = np.zeros(len(sets) + 1, np.int64)
    off[1:] = np.cumsum([len(s) for s in sets])
    out["offsets"][:len(off)] = off
    if sets:
        out["verts"][:off[-1]] = np.concatenate(sets)
    return dict(sets=len(sets), offsets=out["offsets"], verts=out["verts"])


def run(state: dict) -> dict:
    if state["kind"] == "nonmax":
        return _flat(qc.remove_nonmax(state["sets"]), state["out"])
    if state["kind"] == "batch":
        res = qc.mine_batch(state["graphs"], state["gammas"], state["min_sizes"],
                            windows=[state["window"]] * len(state["graphs"]), **state["opts"])
    else:
        res = [qc.mine(state["graphs"][0], state["gammas"][0], state["min_sizes"][0], window=state["window"],
                       **state["opts"])]
    got = _flat([s for r in res for s in r.maximal], state["out"])
    got["counters"] = np.array([[r.stats[k] for k in COUNTERS] for r in res], np.int64)
    return got


def work(case: dict) -> dict:
    """Bytes a pass cannot do without.  The size of a search's answer is not
    known before it, so a mining call counts the graphs it reads (8 bytes an
    offset, 4 bytes an adjacency entry); RemoveNonMax counts its sets (about
    52 vertices each), read once, and a survivor in four written once."""
    if case["kind"] == "nonmax":
        return {"bytes": case["sets"] * (8 + 52 * 4) * 1.25, "flops": 0}
    total = 0.0
    for i in range(case.get("count", 1)):
        off, adj, _, _ = _base(case["config"], case["graph_seed"], case.get("instance", 0) + i)
        total += 8.0 * len(off) + 4.0 * len(adj)
    return {"bytes": total, "flops": 0}


def exact(case: dict, seed: int):
    """Every output is a whole number: there is no rounding to measure."""
    return None
