"""CPU: plans for a state that is handed out in logical order next.

dgq_recorder_plan_home against dgq_recorder_plan, both run in the numpy model of
the descriptors: the same state in logical order to 1e-12 (the gates and their
order are the same; only where qubits lie differs), every block valid (the model
asserts its masks), and the map at the end: at home where the last tile holds the
six lane qubits, and never more than what one permutation pass of 12 bits undoes.
"""
import ctypes as C

import numpy as np
import pytest

from dgquest_amd import circuits
from dgquest_amd.quest import BLOCK_DT, OP_DT, PHASE_DT
from tests import helpers as H
from tests import plan_model as M


def _plan(api, q, home, shape):
    f = api.lib.dgq_recorder_plan_home if home else api.lib.dgq_recorder_plan
    f.argtypes = api.lib.dgq_recorder_plan.argtypes
    n = int(q.numQubitsRepresented)
    counts, l2p = (C.c_int * 3)(), (C.c_int * n)()
    f(q, *shape, 4096, 1, None, 0, None, 0, None, 0, counts, l2p)
    b, p, o = np.zeros(counts[0], BLOCK_DT), np.zeros(counts[1], PHASE_DT), np.zeros(counts[2], OP_DT)
    assert f(q, *shape, 4096, 1, b.ctypes.data, len(b), p.ctypes.data, len(p), o.ctypes.data, len(o), counts, l2p) == 0
    return b, p, o, list(l2p)


def _state(n, plan):
    b, p, o, l2p = plan
    psi = np.zeros(1 << n, dtype=np.complex128)
    M.run_plan(psi, n, b, p, o)
    i = np.arange(1 << n, dtype=np.int64)
    phys = np.zeros_like(i)
    for q in range(n):
        phys |= ((i >> q) & 1) << l2p[q]
    return psi[phys]


def _circuit(kind, n, rng):
    if kind == "qft":
        return circuits.ghz_qft(n)
    if kind == "hea":
        return circuits.hea(n, 4, 3)
    if kind == "layered":
        return circuits.layered_u3_cz(n, 6, 5)
    return H.random_circuit(rng, n, 120)  # swaps among its gates


@pytest.mark.parametrize("kind", ["qft", "hea", "layered", "random"])
@pytest.mark.parametrize("n,shape", [(7, (6, 3, 3)), (9, (3, 3, 0)), (12, (6, 3, 3)), (13, (3, 3, 0)), (14, (7, 4, 3)),
                                     (15, (4, 4, 0)), (16, (5, 4, 1)), (16, (3, 2, 1))])
@pytest.mark.parametrize("init", [0, 77, "plus"])
def test_home_plans_give_the_same_state(quest, kind, n, shape, init):
    rng = np.random.default_rng(n)
    q = quest.dgq_create_recorder(n)
    try:
        if init == "plus":
            quest.initPlusState(q)
        elif init:
            quest.initClassicalState(q, init)
        quest.apply_circuit(q, _circuit(kind, n, rng))
        plain, home = _plan(quest, q, False, shape), _plan(quest, q, True, shape)
    finally:
        quest.dgq_destroy_recorder(q)
    assert np.abs(_state(n, plain) - _state(n, home)).max() <= 1e-12
    assert len(home[0]) == len(plain[0])  # no block more
    l2p = home[3]
    assert sorted(l2p) == list(range(n))
    moved = {q for q in range(n) if l2p[q] != q} | set(range(min(n, 6)))
    assert len(moved) <= 12
    if n <= 6 + shape[1] + shape[2]:  # one tile: everything ends at home
        assert l2p == list(range(n))
