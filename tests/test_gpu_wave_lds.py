"""The waves of a persistent launch share the LDS of their CU between them,
however many the order of the search allows."""
import re

import pytest
import torch

import cuqc_amd as qc
from tests.graphs import planted

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", [dict(), dict(scheduling=1), dict(trace=True)], ids=["dynamic", "static", "trace"])
def test_lds_of_a_cu_is_used(form, monkeypatch, capfd):
    monkeypatch.setenv("QCMINE_PHASES", "1")
    g = qc.Graph.from_csr(*planted(700, 0.15, [40], 0.95, 43))
    qc.mine(g, 0.6, 20, window=(0, 1, 1), mode="persistent", **form)
    m = re.search(r"grid (\d+) waves, (\d+) B of LDS each", capfd.readouterr().err)
    per_cu = int(m[1]) // torch.cuda.get_device_properties(0).multi_processor_count
    # (160 KB a CU in granules of 1,280 B, less 1.1 KB of static LDS a wave)
    assert per_cu * (int(m[2]) + 1120 + 1280 + 256) >= 160 * 1024
    assert per_cu * (int(m[2]) + 1120) <= 160 * 1024
