"""GPU: dense sweeps whose matrices are formed on the device
(dq_apply_dense_gates) against numpy.

One tile, one op per matrix: no gate (the identity), one, and many, of every
form (a 2x2 on each bit with no, some and all controls, phases with any
controls, a projection).  An output is a sum of 2^(k+1) real products of the
rounded matrix and the state, so its error is at most (2^(k+1) + 1) * 2^-24 of
the matrix row's norm (at most 1) times the norm of its 2^k amplitudes.
"""
import ctypes as C

import numpy as np
import pytest

from dgquest_amd.engine import Engine

pytestmark = pytest.mark.gpu

BLOCK = np.dtype([("n_qubits", "<u4"), ("tile_bits", "<u4"), ("op_begin", "<u4"), ("op_count", "<u4"),
                  ("nontile_mask", "<u8"), ("tile_q", "u1", 16)])
OP = np.dtype([("bits", "<u4", 8), ("mat", "<u8")])
GATE = np.dtype([("tmask", "<u4"), ("cmask", "<u4"), ("diag", "<u4"), ("pad", "<u4"), ("u", "<f8", 8)])


def _gates(rng, k, count):
    out = np.zeros(count, dtype=GATE)
    for i in range(count):
        g = out[i]
        t = i % k
        others = [b for b in range(k) if b != t]
        cm = sum(1 << b for b in others if rng.uniform() < (0.0, 0.3, 1.0)[i % 3])
        if i % 4 == 3:
            g["diag"], g["cmask"] = 1, cm
            g["u"][:2] = np.cos(i), np.sin(i)
            continue
        q, _ = np.linalg.qr(rng.standard_normal((2, 2)) + 1j * rng.standard_normal((2, 2)))
        if i == 5:
            q = np.array([[0, 0], [0, 1.25]])
        g["tmask"], g["cmask"] = 1 << t, cm
        g["u"][:] = np.ascontiguousarray(q.astype(complex)).view(float).reshape(-1)
    return out


def _matrix(gates, k):
    m = np.eye(1 << k, dtype=complex)
    i = np.arange(1 << k)
    for g in gates:
        tm, cm, u = int(g["tmask"]), int(g["cmask"]), g["u"][0::2] + 1j * g["u"][1::2]
        on = (i & cm) == cm
        if g["diag"]:
            m[on] *= u[0]
            continue
        lo = i[on & ((i & tm) == 0)]
        x, y = m[lo].copy(), m[lo | tm].copy()
        m[lo], m[lo | tm] = u[0] * x + u[1] * y, u[2] * x + u[3] * y
    return m


@pytest.mark.parametrize("k", [5, 6, 7])
@pytest.mark.parametrize("count", [0, 1, 23])
def test_dense_gates(k, count, quest32, env32):
    L = Engine().lib
    vp = C.c_void_p
    L.dq_dense_gates_ws_bytes.restype = C.c_size_t
    L.dq_dense_gates_ws_bytes.argtypes = [C.c_int] + [C.c_uint32] * 4
    L.dq_apply_dense_gates.argtypes = [C.c_int, vp, C.c_uint32, vp, C.c_uint32, vp, vp, C.c_uint32, vp, vp, C.c_size_t, vp]
    rng = np.random.default_rng(10 * k + count)
    n = 12
    gates = np.concatenate([_gates(rng, k, count), _gates(rng, k, 2)])
    begin = np.array([0, count, count + 2], dtype=np.uint32)
    block = np.zeros(1, dtype=BLOCK)
    block["n_qubits"], block["tile_bits"], block["op_count"], block["tile_q"][0, :n] = n, n, 2, np.arange(n)
    ops = np.zeros(2, dtype=OP)
    bits = [sorted(rng.permutation(n)[:k]) for _ in range(2)]
    for o in range(2):
        ops["bits"][o, :k], ops["mat"][o] = bits[o], o
    a = rng.standard_normal(1 << n) + 1j * rng.standard_normal(1 << n)
    a = (a / np.linalg.norm(a)).astype(np.complex64)
    re, im = np.ascontiguousarray(a.real), np.ascontiguousarray(a.imag)
    q = quest32.createQureg(n, env32)
    ws = vp()
    try:
        pf = C.POINTER(C.c_float)
        quest32.initStateFromAmps(q, re.ctypes.data_as(pf), im.ctypes.data_as(pf))
        st = quest32.dgq_state_pointer(q, None)
        wsb = L.dq_dense_gates_ws_bytes(k, 1, 2, 2, len(gates))
        assert L.dq_malloc(C.byref(ws), wsb) == 0
        args = [k, block.ctypes.data, 1, ops.ctypes.data, 2, gates.ctypes.data, begin.ctypes.data, 2, st, ws]
        assert L.dq_apply_dense_gates(*args, wsb, None) == 0, L.dq_last_error().decode()
        assert L.dq_stream_sync(None) == 0
        got = quest32.state_vector(q)
        # refused: a workspace too small, a control outside the op, a target under its own control
        assert L.dq_apply_dense_gates(*args, wsb - 1, None) != 0
        for bad in ((1 << k, 0), (1, 1)):
            wrong = gates.copy()
            wrong["cmask"][-1], wrong["tmask"][-1], wrong["diag"][-1] = bad[0], bad[1] or 1, 0
            args[5] = wrong.ctypes.data
            assert L.dq_apply_dense_gates(*args, wsb, None) != 0
    finally:
        if ws:
            L.dq_free(ws)
        quest32.destroyQureg(q, env32)
    want = a.astype(np.complex128)
    tol = 0.0
    for o in range(2):
        m = _matrix(gates[begin[o]:begin[o + 1]], k)
        axes = [n - 1 - b for b in reversed(bits[o])]
        t = np.moveaxis(want.reshape([2] * n), axes, range(k)).reshape(1 << k, -1)
        y = m @ t
        tol += ((2 << k) + 1) * 2.0 ** -24 * max(np.linalg.norm(m, axis=1).max(), 1.0) * np.linalg.norm(t, axis=0).max()
        want = np.moveaxis(y.reshape([2] * n), range(k), axes).reshape(-1)
    assert np.abs(got - want).max() <= tol
