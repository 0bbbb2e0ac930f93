"""The waves of a persistent launch share the LDS of their CU between them,
however many the order of the search allows."""
import re

import pytest

import cuqc_amd as qc
from tests.graphs import planted

pytestmark = pytest.mark.gpu


def test_lds_of_a_cu_is_used(monkeypatch, capfd):
    monkeypatch.setenv("QCMINE_PHASES", "1")
    g = qc.Graph.from_csr(*planted(700, 0.15, [40], 0.95, 43))
    lds = {}
    for order, form in (("dynamic", dict()), ("static", dict(scheduling=1)), ("trace", dict(trace=True))):
        qc.mine(g, 0.6, 20, window=(0, 1, 1), mode="persistent", **form)
        m = re.search(r"grid (\d+) waves, (\d+) B of LDS each", capfd.readouterr().err)
        lds[order] = (int(m[1]), int(m[2]))
    # (with 1.1 KB of static LDS a wave, in granules of 1,280 B a workgroup)
    whole = lds["dynamic"][0] * (lds["dynamic"][1] + 1120)
    for waves, each in lds.values():
        assert 0.95 * whole <= waves * (each + 1120) <= 1.05 * whole
    assert lds["static"][0] < lds["dynamic"][0]
