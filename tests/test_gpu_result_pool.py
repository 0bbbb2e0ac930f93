"""Pinned result blocks beyond what the pool keeps, freed by one thread while
others mine."""
import queue
import threading

import numpy as np
import pytest

import cuqc_amd as qc

pytestmark = pytest.mark.gpu


def digest(res):
    return len(res.raw), int(res.raw.verts.sum(dtype=np.int64)), len(res.raw.verts)


def test_blocks_freed_while_others_are_made():
    # 194 MB of raw sets a call; at most 1 GB of free blocks is kept
    g = qc.Graph.generate(3, 4, 15)
    want = digest(qc.mine(g, g.gamma, g.min_size, mode="persistent"))
    assert want[2] * 4 > 100 << 20
    held, bad = queue.Queue(), []

    def mine():
        for _ in range(6):
            res = qc.mine(g, g.gamma, g.min_size, mode="persistent")
            held.put(res)

    miners = [threading.Thread(target=mine) for _ in range(2)]
    [t.start() for t in miners]
    [t.join() for t in miners]  # 12 results, 2.3 GB
    more = threading.Thread(target=mine)
    more.start()
    while more.is_alive() or not held.empty():
        try:
            res = held.get(timeout=0.1)
        except queue.Empty:
            continue
        if digest(res) != want:
            bad.append(digest(res))
        del res
    more.join()
    assert not bad
