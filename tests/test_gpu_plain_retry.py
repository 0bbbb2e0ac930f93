"""The level-synchronous form where a launch's raw sets overflow the stream."""
import pytest

import cuqc_amd as qc
import oracle
from tests.graphs import planted

pytestmark = pytest.mark.gpu

COUNTERS = ["tasks", "branches", "children", "raw_cliques", "w_adj", "sum_t", "sum_t_written", "sum_clique_len"]


@pytest.fixture(scope="module")
def case():
    # two tasks below the root, of 5 and 19 raw sets; a window of one level
    off, adj = planted(80, 0.15, [], 1.0, 61)
    sets = [oracle.mine(off, adj, 0.5, 2, root_begin=b, root_end=b + 1, max_depth=1)["stats"]["raw_cliques"]
            for b in (0, 1)]
    assert sets == [19, 5]
    return qc.Graph.from_csr(off, adj), oracle.mine(off, adj, 0.5, 2, root_begin=0, root_end=2, max_depth=1)


def run(case, refs, monkeypatch):
    monkeypatch.setenv("QCMINE_INITIAL_CAPACITY", str(refs // 2))  # room for `refs` sets
    return qc.mine(case[0], 0.5, 2, window=(0, 2, 1), mode="plain")


@pytest.mark.parametrize("refs", [20, 22, 26])
def test_one_task_after_others(case, refs, monkeypatch):
    """Up to 22: both tasks overflow the stream, the first one alone leaves less
    than the second needs, which then runs on the emptied stream."""
    res = run(case, refs, monkeypatch)
    for k in COUNTERS:
        assert res.stats[k] == case[1]["stats"][k], k
    assert oracle.canon(res.raw) == oracle.canon(case[1]["raw"])


def test_one_task_too_large(case, monkeypatch):
    with pytest.raises(qc.QCError, match="overflowed"):
        run(case, 18, monkeypatch)
