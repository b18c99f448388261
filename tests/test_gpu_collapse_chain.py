"""GPU: collapses one after another with no gate between them, whose P(0) comes from
the amplitudes that they keep.

Unlikely outcomes: every qubit of a product state is 0 with probability 2e-13 and
collapsed to it.  The kept amplitudes fall to 1e-165, their squares below the
smallest FP64 number.  P(0) of each is 2e-13 up to the rounding of the angle
(pi/2 to 2^-53 against 4.5e-7: 5e-10, doubled by the square): 1e-8 relative; the
state after 26 of them within 26 times that.
"""
import math

import pytest

pytestmark = pytest.mark.gpu


def test_unlikely_outcomes(quest, env):
    n, p = 26, 2e-13
    q = quest.createQureg(n, env)
    try:
        quest.initZeroState(q)
        for k in range(n):
            quest.rotateY(q, k, math.pi - 2.0 * math.asin(math.sqrt(p)))
        for k in range(n):
            assert abs(quest.collapseToOutcome(q, k, 0) / p - 1.0) <= 1e-8, k
        assert abs(quest.calcTotalProb(q) - 1.0) <= n * 1e-8
        a = quest.getAmp(q, 0)
        assert abs(a.real ** 2 + a.imag ** 2 - 1.0) <= n * 1e-8
    finally:
        quest.destroyQureg(q, env)


def test_a_collapse_repeated_many_times_stays_short(quest, env):
    q = quest.createQureg(10, env)
    try:
        quest.initZeroState(q)
        quest.hadamard(q, 3)
        for _ in range(300):
            quest.collapseToOutcome(q, 3, 1)
        quest.dgq_flush(q)
        assert quest.plan_stats(q)["gates_in"] <= 64
        assert abs(quest.getAmp(q, 8).real - 1.0) <= 1e-12
    finally:
        quest.destroyQureg(q, env)
