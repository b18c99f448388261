"""CPU: how many passes dq_permute_qubits takes, and what it refuses."""
import ctypes as C

import numpy as np
import pytest

from dgquest_amd.engine import Engine


def _launches(n, prec, dest):
    L = Engine().lib
    L.dq_permute_launches.argtypes = [C.c_int, C.c_int, C.POINTER(C.c_int)]
    return L.dq_permute_launches(n, prec, (C.c_int * len(dest))(*dest))


@pytest.mark.parametrize("prec", [1, 2])
@pytest.mark.parametrize("n", [1, 6, 12, 20, 30, 36, 40])
def test_passes(n, prec):
    ident = list(range(n))
    assert _launches(n, prec, ident) == 0
    if n > 1:
        assert _launches(n, prec, ident[::-1]) == 1  # an involution
        far = ident[:]
        far[0], far[-1] = far[-1], far[0]
        assert _launches(n, prec, far) == 1
    if n > 2:
        three = ident[:]
        three[0], three[n // 2], three[n - 1] = n // 2, n - 1, 0
        assert _launches(n, prec, three) == 1  # three bits fit any tile
        assert _launches(n, prec, [(p + 1) % n for p in ident]) == (1 if n <= (11 if prec == 2 else 12) else 2)
    rng = np.random.default_rng(n)
    for _ in range(20):
        assert _launches(n, prec, [int(x) for x in rng.permutation(n)]) in (0, 1, 2)


@pytest.mark.parametrize("n,prec,dest", [(3, 2, [0, 1, 1]), (3, 2, [0, 1, 3]), (3, 2, [-1, 1, 2]), (0, 2, [0]), (3, 3, [0, 1, 2]),
                                         (41, 2, list(range(41)))])
def test_refused(n, prec, dest):
    assert _launches(n, prec, dest) < 0
