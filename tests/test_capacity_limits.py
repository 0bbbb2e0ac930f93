"""Capacities whose bytes would not fit 64 bits are refused like any others that
no device holds, before anything is allocated or launched."""
import pytest

import cuqc_amd as qc
from tests.graphs import complete


@pytest.mark.parametrize("mode", ["plain", "persistent"])
@pytest.mark.parametrize("name", ["task_capacity", "clique_capacity"])
@pytest.mark.parametrize("value", [(1 << 64) - 1, 1 << 62, 1 << 60, (1 << 48) + 1])
def test_refused(mode, name, value):
    g = qc.Graph.from_csr(*complete(12))
    with pytest.raises(qc.QCError) as e:
        qc.mine(g, 0.9, 5, mode=mode, **{name: value})
    assert e.value.code == qc.QC_ENOMEM
    if mode == "persistent":
        with pytest.raises(qc.QCError) as e:
            qc.mine_batch([g, g], [0.9, 0.9], [5, 5], **{name: value})
        assert e.value.code == qc.QC_ENOMEM
