"""GPU: dq_permute_qubits moves every amplitude to its place, exactly.

Every amplitude holds its own index (exact in float up to 2^24).  Permutations:
the identity, one swap near and far, a reversal (an involution of every bit), a
rotation (one long cycle: two passes), few bits moved, random ones; registers
from one bit to some bits past the tile, and a larger one.  The number of passes is
checked without a GPU in test_permute_host.
"""
import ctypes as C

import numpy as np
import pytest

from dgquest_amd.engine import Engine

pytestmark = pytest.mark.gpu


def _perms(n, rng):
    ident = list(range(n))
    far = ident[:]
    far[0], far[n - 1] = far[n - 1], far[0]
    near = ident[:]
    if n > 2:
        near[1], near[2] = near[2], near[1]
    few = ident[:]
    pick = [int(x) for x in rng.permutation(n)[:3]]
    for a, b in zip(pick, pick[1:] + pick[:1]):
        few[a] = b
    top = ident[:]
    for i in range(n // 2, n):  # the upper half reversed, the coalesced bits stay
        top[i] = n - 1 - (i - n // 2)
    return [ident, far, near, ident[::-1], [(p + 1) % n for p in range(n)], few, top] + \
        [[int(x) for x in rng.permutation(n)] for _ in range(3)]


@pytest.mark.parametrize("n", [1, 2, 5, 6, 7, 9, 10, 11, 12, 13, 14, 15, 17, 20, 22])
@pytest.mark.parametrize("prec", [1, 2])
def test_permute_qubits(n, prec, quest, env, quest32, env32):
    api, e = (quest, env) if prec == 2 else (quest32, env32)
    L = Engine().lib
    L.dq_permute_qubits.argtypes = [C.c_void_p, C.c_int, C.c_int, C.POINTER(C.c_int), C.c_void_p]
    rng = np.random.default_rng(10 * n + prec)
    real = np.float64 if prec == 2 else np.float32
    i = np.arange(1 << n)
    re, im = i.astype(real), (-i).astype(real)
    q = api.createQureg(n, e)
    ptr = C.POINTER(api.qreal)
    try:
        for dest in _perms(n, rng):
            api.initStateFromAmps(q, re.ctypes.data_as(ptr), im.ctypes.data_as(ptr))
            st = api.dgq_state_pointer(q, None)
            assert L.dq_permute_qubits(st, n, prec, (C.c_int * n)(*dest), api.dgq_stream(q)) == 0
            to = np.zeros_like(i)
            for p in range(n):
                to |= ((i >> p) & 1) << dest[p]
            want = np.empty_like(i)
            want[to] = i
            got = api.state_vector(q)
            assert np.array_equal(got.real, want) and np.array_equal(got.imag, -want), (n, prec, dest)
    finally:
        api.destroyQureg(q, e)


@pytest.mark.parametrize("prec", [1, 2])
def test_state_after_relabelling(prec, quest, env, quest32, env32):
    """A program's own relabellings, undone when the state is handed out: equal
    amplitudes through the map before and in place after."""
    api, e = (quest, env) if prec == 2 else (quest32, env32)
    n = 19
    rng = np.random.default_rng(prec)
    q = api.createQureg(n, e)
    try:
        for rep in range(4):
            for k in range(n):
                api.rotateY(q, k, float(rng.uniform(0, 3)))
            for _ in range(rep * 5):
                a, b = (int(x) for x in rng.choice(n, 2, replace=False))
                api.swapGate(q, a, b)
                api.controlledPhaseShift(q, a, b, float(rng.uniform(0, 3)))
            through = api.state_vector(q)
            assert api.dgq_state_pointer(q, None)
            assert np.array_equal(api.state_vector(q), through)
    finally:
        api.destroyQureg(q, e)
