"""GPU: P(0) of every qubit, over a whole state and over the amplitudes that a
set of collapsed qubits leaves (dq_prob_zero_all_fixed), against numpy.

The sums are trees of at most 2^n non-negative doubles, at most 48 additions
deep, so 48 * 2^-53 of the total (1) bounds their error; 1e-13 is allowed.
Sizes: below one workgroup, every number of loads per thread and its edges,
and the sizes where a workgroup starts to loop.
"""
import ctypes as C

import numpy as np
import pytest

from dgquest_amd.engine import Engine

pytestmark = pytest.mark.gpu


def _lib():
    L = Engine().lib
    vp = C.c_void_p
    L.dq_prob_ws_bytes.restype = C.c_size_t
    L.dq_prob_ws_bytes.argtypes = [C.c_int]
    L.dq_prob_zero_all_fixed.argtypes = [vp, C.c_int, C.c_int, C.c_uint64, C.c_uint64, C.c_double,
                                         C.POINTER(C.c_double), vp, C.c_size_t, vp]
    return L


def _expect(p, n, fixed, value, scale):
    i = np.arange(1 << n, dtype=np.uint64)
    p = np.where((i & np.uint64(fixed)) == np.uint64(value), p, 0.0)
    return scale * np.array([p.reshape(-1, 2, 1 << q)[:, 0].sum() for q in range(n)] + [p.sum()])


@pytest.mark.parametrize("n", [1, 2, 6, 7, 8, 9, 13, 16, 17, 19, 20, 21, 25, 26])
@pytest.mark.parametrize("prec", [1, 2])
def test_prob_zero_all_fixed(n, prec, quest, env, quest32, env32):
    L = _lib()
    api, e = (quest, env) if prec == 2 else (quest32, env32)
    rng = np.random.RandomState(100 * n + prec)
    real = np.float64 if prec == 2 else np.float32
    re, im = rng.standard_normal((2, 1 << n))
    s = 1.0 / np.sqrt((re ** 2 + im ** 2).sum())
    re, im = (re * s).astype(real), (im * s).astype(real)
    p = re.astype(np.float64) ** 2 + im.astype(np.float64) ** 2
    q = api.createQureg(n, e)
    ws = C.c_void_p()
    try:
        ptr = C.POINTER(api.qreal)
        api.initStateFromAmps(q, re.ctypes.data_as(ptr), im.ctypes.data_as(ptr))
        st = api.dgq_state_pointer(q, None)
        assert st
        wsb = L.dq_prob_ws_bytes(n)
        assert L.dq_malloc(C.byref(ws), wsb) == 0
        masks = [0, 1, 1 << (n - 1), (1 << n) - 1] + [int(rng.randint(1 << min(n, 30))) & int(rng.randint(1 << min(n, 30)))
                                                      for _ in range(2)]
        for fixed in masks:
            value = fixed & int(rng.randint(1 << min(n, 30)))
            got = (C.c_double * (n + 1))()
            rc = L.dq_prob_zero_all_fixed(st, n, prec, fixed, value, 1.5, got, ws, wsb, None)
            assert rc == 0, L.dq_last_error().decode()
            err = np.abs(np.array(got[:]) - _expect(p, n, fixed, value, 1.5)).max()
            assert err <= 1e-13, (n, prec, hex(fixed), hex(value), err)
        # refused: bits outside the register, a value outside the mask
        assert L.dq_prob_zero_all_fixed(st, n, prec, 1 << n, 0, 1.0, got, ws, wsb, None) != 0
        assert L.dq_prob_zero_all_fixed(st, n, prec, 0, 1, 1.0, got, ws, wsb, None) != 0
    finally:
        if ws:
            L.dq_free(ws)
        api.destroyQureg(q, e)


@pytest.mark.parametrize("prec", [1, 2])
def test_collapses_stay_recorded_until_read(prec, quest, env, quest32, env32):
    """Measurements answered from the kept amplitudes, then the state itself:
    it must be the collapse of the state before, whatever was measured last."""
    api, e = (quest, env) if prec == 2 else (quest32, env32)
    n, tol = 10, 1e-13 if prec == 2 else 4e-6
    rng = np.random.RandomState(7)
    q = api.createQureg(n, e)
    try:
        for k in range(n):
            api.rotateY(q, k, float(rng.uniform(0.5, 2.5)))
        for k in range(n):
            api.controlledPhaseShift(q, k, (k + 1) % n, float(rng.uniform(0, 6)))
            api.rotateX(q, (3 * k) % n, float(rng.uniform(0.5, 2.5)))
        before = api.state_vector(q)
        i = np.arange(1 << n)
        keep = np.ones(1 << n, dtype=bool)
        for k in (3, 0, 9, 3, 6):
            stat = api.qreal()
            out = api.measureWithStats(q, k, C.byref(stat))
            p = np.abs(np.where(keep, before, 0)) ** 2
            want = p[((i >> k) & 1) == out].sum() / p.sum()
            assert abs(stat.value - want) <= tol
            keep &= ((i >> k) & 1) == out
            if k == 9:  # a relabelling in between: the collapses are those of the qubits measured
                api.swapGate(q, 1, 2)
                swapped = (i & ~6) | ((i & 2) << 1) | ((i & 4) >> 1)
                before, keep = before[swapped], keep[swapped]
        assert abs(api.calcTotalProb(q) - 1.0) <= tol
        want = np.where(keep, before, 0)
        want /= np.linalg.norm(want)
        assert np.abs(api.state_vector(q) - want).max() <= tol
        assert abs(api.calcProbOfOutcome(q, 9, 0) - (np.abs(want) ** 2)[((i >> 9) & 1) == 0].sum()) <= tol
    finally:
        api.destroyQureg(q, e)
