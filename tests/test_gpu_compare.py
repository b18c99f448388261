"""GPU: dq_compare_states (inner product, norms, largest difference) against numpy.

Every sum is a tree of products of at most 2^n terms; a thread adds at most 2^9
step sums of 8, the trees above add 22 levels, so each result is within
600 * 2^-53 of the sum of the terms' magnitudes (at most 1): 1e-13 is allowed.
The largest difference has 3 roundings and a square root.
Sizes: below a workgroup, one load per thread, a share's edges and the first
size at which shares grow.
"""
import ctypes as C

import numpy as np
import pytest

from dgquest_amd.engine import Engine

pytestmark = pytest.mark.gpu


def _register(api, env, n, re, im):
    q = api.createQureg(n, env)
    real = np.float64 if api.prec == 2 else np.float32
    ptr = C.POINTER(api.qreal)
    re, im = np.ascontiguousarray(re, dtype=real), np.ascontiguousarray(im, dtype=real)
    api.initStateFromAmps(q, re.ctypes.data_as(ptr), im.ctypes.data_as(ptr))
    return q, re.astype(np.float64) + 1j * im.astype(np.float64)


@pytest.mark.parametrize("n", [1, 5, 8, 9, 10, 11, 12, 13, 17, 24, 25])
@pytest.mark.parametrize("precs", [(2, 2), (1, 1), (1, 2), (2, 1)])
def test_compare_states(n, precs, quest, env, quest32, env32):
    L = Engine().lib
    vp = C.c_void_p
    rng = np.random.RandomState(10 * n + precs[0])
    apis = [(quest, env) if p == 2 else (quest32, env32) for p in precs]
    regs, vecs = [], []
    for api, e in apis:
        re, im = rng.standard_normal((2, 1 << n))
        s = 1.0 / np.sqrt((re ** 2 + im ** 2).sum())
        q, v = _register(api, e, n, re * s, im * s)
        regs.append((api, e, q))
        vecs.append(v)
    ws, out = vp(), vp()
    try:
        ptrs = [api.dgq_state_pointer(q, None) for api, _, q in regs]
        wsb = L.dq_compare_ws_bytes(n)
        assert L.dq_malloc(C.byref(ws), wsb) == 0 and L.dq_malloc(C.byref(out), 40) == 0
        got = (C.c_double * 5)()
        assert L.dq_compare_states(ptrs[0], precs[0], ptrs[1], precs[1], n, out, ws, wsb, None) == 0
        assert L.dq_memcpy_async(got, out, 40, 2, None) == 0 and L.dq_stream_sync(None) == 0
        a, b = vecs
        z = np.vdot(a, b)
        want = [z.real, z.imag, np.vdot(a, a).real, np.vdot(b, b).real]
        assert np.abs(np.array(got[:4]) - want).max() <= 1e-13
        d = np.abs(a - b).max()
        assert abs(got[4] - d) <= 1e-14 * d
        if wsb > 256:
            assert L.dq_compare_states(ptrs[0], precs[0], ptrs[1], precs[1], n, out, ws, wsb - 256, None) != 0
    finally:
        for api, e, q in regs:
            api.destroyQureg(q, e)
        if ws:
            L.dq_free(ws)
        if out:
            L.dq_free(out)
