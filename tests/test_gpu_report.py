"""GPU: the DGQ_REPORT_FILE summary of a register whose last calls were measurements.

The report's probabilities and amplitudes are those of the collapsed state.  It
is computed here from the amplitudes read before: the ones that the outcomes
keep, over the root of what they add up to.  At most 12 roundings each on the
device: 1e-14 in FP64; in FP32 the collapses round to 2^-24 a few times: 1e-6.
"""
import json

import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4, 9, 13])
@pytest.mark.parametrize("prec", [1, 2])
def test_report_after_measurements(n, prec, quest, env, quest32, env32, tmp_path, monkeypatch):
    api, e = (quest, env) if prec == 2 else (quest32, env32)
    tol = 1e-14 if prec == 2 else 1e-6
    q = api.createQureg(n, e)
    api.initZeroState(q)
    api.apply_circuit(q, H.random_circuit(np.random.default_rng(n), n, 60))
    v = api.state_vector(q)
    api.seed([7, n])
    for k in (n - 1, 1, 2):
        out = api.measure(q, k)
        v = np.where((np.arange(1 << n) >> k) & 1 == out, v, 0.0)
    v /= np.sqrt((np.abs(v) ** 2).sum())
    path = tmp_path / "report.jsonl"
    monkeypatch.setenv("DGQ_REPORT_FILE", str(path))
    api.destroyQureg(q, e)
    monkeypatch.delenv("DGQ_REPORT_FILE")
    (row,) = [json.loads(x) for x in path.read_text().splitlines()]
    amps = np.array([complex(*a) for a in row["amps"]])
    w = np.abs(v) ** 2
    p1 = [w.reshape(-1, 2, 1 << k)[:, 1].sum() for k in range(n)]
    assert np.abs(amps - v[:16]).max() <= tol
    assert np.abs(np.array(row["p1"]) - p1).max() <= 4 * tol
    assert abs(row["total_prob"] - 1.0) <= 4 * tol
