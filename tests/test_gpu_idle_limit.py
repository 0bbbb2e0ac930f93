"""Waves that wait while one other works: the persistent launch is given up
only when tasks are pending and no wave works."""
import pytest

import cuqc_amd as qc
import oracle
from tests.graphs import planted

pytestmark = pytest.mark.gpu

COUNTERS = ["tasks", "branches", "children", "raw_cliques", "w_adj", "sum_t", "sum_t_written"]


@pytest.fixture(scope="module")
def case():
    off, adj = planted(960, 0.12, [40], 0.95, 44)
    return qc.Graph.from_csr(off, adj), oracle.mine(off, adj, 0.6, 20, root_begin=0, root_end=2, max_depth=1)


# Two tasks of about 950 vertices that are not split: some 9 ms on a wave each,
# against 64 looks of 14 us.
@pytest.mark.parametrize("form", [dict(), dict(scheduling=1), dict(workgroups=2), dict(workgroups=40), dict(trace=True)],
                         ids=["dynamic", "static", "2_waves", "40_waves", "trace"])
def test_long_tasks_on_few_waves(case, form, monkeypatch):
    monkeypatch.setenv("QCMINE_IDLE_LIMIT", "64")
    g, ref = case
    res = qc.mine(g, 0.6, 20, window=(0, 2, 1), mode="persistent", split_chunk=-1, **form)
    print(f"[gpu] {form}: {res.stats['t_kernel_ms']:.2f} ms", flush=True)
    for k in COUNTERS:
        assert res.stats[k] == ref["stats"][k], k
    assert res.stats["t_kernel_ms"] > 2.0
