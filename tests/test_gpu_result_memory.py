"""Raw sets are views of the memory the device wrote: they outlive the Result
that held them, several results are held at a time, and threads mine at once."""
import gc
import threading

import numpy as np
import pytest

import cuqc_amd as qc
import oracle
from tests.graphs import planted

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def graphs():
    # raw sets above and below a megabyte (the size from which blocks are pinned)
    out = []
    for n, p, sizes, keep, seed, gamma, ms in [(120, 0.10, [26, 24], 0.93, 51, 0.85, 11), (60, 0.30, [], 1.0, 11, 0.7, 6),
                                               (30, 0.10, [], 1.0, 52, 0.9, 20)]:
        off, adj = planted(n, p, sizes, keep, seed)
        ref = oracle.mine(off, adj, gamma, ms, threads=4)
        out.append((qc.Graph.from_csr(off, adj), gamma, ms, oracle.canon(ref["raw"])))
    assert sum(4 * len(s) for s in out[0][3]) > 1 << 20 and not out[2][3]
    return out


def test_arrays_outlive_their_result(graphs):
    held = []
    for _ in range(3):
        for g, gamma, ms, want in graphs:
            raw = qc.mine(g, gamma, ms).raw
            held.append((raw.offsets, raw.verts[1:], raw.verts[:1].copy(), want))
            del raw
            gc.collect()
    for off, tail, head, want in held:
        assert oracle.canon(qc.SetList(off, np.concatenate([head, tail]))) == want


def test_results_are_writable_and_separate(graphs):
    g, gamma, ms, want = graphs[0]
    a, b = qc.mine(g, gamma, ms), qc.mine(g, gamma, ms)
    a.raw.verts[:] = 0
    assert oracle.canon(b.raw) == want


def test_threads(graphs):
    bad = []

    def work(k):
        for i in range(4):
            g, gamma, ms, want = graphs[(k + i) % len(graphs)]
            if oracle.canon(qc.mine(g, gamma, ms).raw) != want:
                bad.append((k, i))

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad
