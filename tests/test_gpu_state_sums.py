"""GPU: P(0) of every qubit from the sums that the last sweep of a flush writes,
against numpy on the state that the same flush stored.

The sums are trees of non-negative doubles as in test_gpu_probs: 1e-13 is allowed; a
sum without terms is exactly 0.  Sizes: the state in one tile, sums added up by the
host (up to 32 tiles) and on the device, the larger second stage (from 2^14 tiles), one
wave and several per tile, every number of register bits.
"""
import numpy as np
import pytest

from dgquest_amd import circuits

pytestmark = pytest.mark.gpu

SHAPES = [(7, (1, 1, 0)), (8, (2, 2, 0)), (9, (3, 3, 0)), (10, (3, 3, 0)), (14, (3, 3, 0)), (15, (3, 3, 0)), (23, (3, 3, 0)),
          (11, (4, 4, 0)), (11, (5, 5, 0)), (12, (5, 4, 1)), (13, (6, 4, 2)), (13, (7, 4, 3)), (14, (8, 5, 3)), (16, (7, 5, 2)),
          (17, (6, 3, 3)), (18, (6, 3, 3)), (22, (7, 4, 3))]


def _check(api, q, n):
    got = [float(api.calcProbOfOutcome(q, k, 0)) for k in range(n)] + [float(api.calcTotalProb(q))]
    v = api.state_vector(q)
    p = v.real ** 2 + v.imag ** 2
    want = [p.reshape(-1, 2, 1 << k)[:, 0].sum() for k in range(n)] + [p.sum()]
    tol = 1e-13 if api.prec == 2 else 1e-13 + 2.0 ** -24  # the API's real type rounds the result
    assert np.abs(np.array(got) - want).max() <= tol
    assert all(g == 0.0 for g, w in zip(got, want) if w == 0.0)


@pytest.mark.parametrize("n,shape", SHAPES)
@pytest.mark.parametrize("rotate", [0, 1])
@pytest.mark.parametrize("prec", [1, 2])
def test_probs_of_a_flush(n, shape, rotate, prec, quest, env, quest32, env32):
    api, e = (quest, env) if prec == 2 else (quest32, env32)
    q = api.createQureg(n, e)
    try:
        api.dgq_set_tuning(q, *shape, 4096)
        api.dgq_set_lane_rotation(q, rotate)
        api.initClassicalState(q, (1 << n) - 2)
        api.apply_circuit(q, [("hadamard", (n - 1,), ())])  # every other qubit keeps its value: exact zeros
        _check(api, q, n)
        api.apply_circuit(q, circuits.hea(n, 2, n) + [("swapGate", (0, n - 1), ())] + circuits.layered_u3_cz(n, 2, n))
        _check(api, q, n)
        api.pauliX(q, 0)  # one phase
        _check(api, q, n)
    finally:
        api.destroyQureg(q, e)
