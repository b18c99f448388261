"""GPU: read-outs through host result slots and descriptor uploads, at the sizes
where their paths change: one workgroup or two launches for P(0) (13 / 14 free
qubits), a result slot or a copy from the device (128 KiB: 2^13 amplitudes),
a copying kernel or the copy engine (64 KiB of descriptors), more threads than slots.

P(0): the bound of test_gpu_probs (1e-13).  Amplitudes are copied, so they are
equal; after a circuit FP64 amplitudes are within 1e-12 of the oracle.
"""
import ctypes as C
import threading

import numpy as np
import pytest

from dgquest_amd import circuits
from dgquest_amd.engine import Engine
from oracle.binding import Oracle

pytestmark = pytest.mark.gpu


def _random(n, real, seed):
    rng = np.random.RandomState(seed)
    re, im = rng.standard_normal((2, 1 << n))
    s = 1.0 / np.sqrt((re ** 2 + im ** 2).sum())
    return (re * s).astype(real), (im * s).astype(real)


@pytest.mark.parametrize("n", [5, 10, 11, 12, 13, 14, 15])
@pytest.mark.parametrize("prec", [1, 2])
def test_probs_and_amplitudes(n, prec, quest, env, quest32, env32):
    api, e = (quest, env) if prec == 2 else (quest32, env32)
    re, im = _random(n, np.float64 if prec == 2 else np.float32, n)
    p = re.astype(np.float64) ** 2 + im.astype(np.float64) ** 2
    L = Engine().lib
    L.dq_prob_ws_bytes.restype = C.c_size_t
    q = api.createQureg(n, e)
    ws = C.c_void_p()
    try:
        ptr = C.POINTER(api.qreal)
        api.initStateFromAmps(q, re.ctypes.data_as(ptr), im.ctypes.data_as(ptr))
        assert np.array_equal(api.state_vector(q), re.astype(np.float64) + 1j * im.astype(np.float64))
        api.swapGate(q, 0, n - 1)  # the map of the read
        i = np.arange(1 << n)
        j = (i & ~(1 | 1 << (n - 1))) | ((i & 1) << (n - 1)) | (i >> (n - 1))
        got = api.state_vector(q, 1, (1 << n) - 2)
        assert np.array_equal(got, (re[j].astype(np.float64) + 1j * im[j].astype(np.float64))[1:-1])
        api.swapGate(q, 0, n - 1)
        st = api.dgq_state_pointer(q, None)
        wsb = L.dq_prob_ws_bytes(n)
        assert L.dq_malloc(C.byref(ws), C.c_size_t(wsb)) == 0
        for fixed in (0, 1, 6, 1 << (n - 1), 0x15 & ((1 << n) - 1)):
            value = fixed & 0x14
            out = (C.c_double * (n + 1))()
            rc = L.dq_prob_zero_all_fixed(C.c_void_p(st), n, prec, C.c_uint64(fixed), C.c_uint64(value), C.c_double(1.0),
                                          out, ws, C.c_size_t(wsb), None)
            assert rc == 0
            w = np.where((i & fixed) == value, p, 0.0)
            want = [w.reshape(-1, 2, 1 << k)[:, 0].sum() for k in range(n)] + [w.sum()]
            assert np.abs(np.array(out[:]) - want).max() <= 1e-13, (n, prec, fixed)
    finally:
        if ws:
            L.dq_free(ws)
        api.destroyQureg(q, e)


@pytest.mark.parametrize("depth", [1, 4, 9, 40, 120])
def test_uploads_of_any_length(depth, quest, env):
    """Programs from a few KiB to several hundred, two registers in turn."""
    n = 10
    regs = [quest.createQureg(n, env) for _ in range(2)]
    try:
        for rep in range(3):
            for k, q in enumerate(regs):
                c = circuits.layered_u3_cz(n, depth, 10 * rep + k)
                quest.initZeroState(q)
                quest.apply_circuit(q, c)
                quest.dgq_flush(q)  # no wait: the other register's upload follows at once
            for k, q in enumerate(regs):
                ref = np.zeros(1 << n, dtype=np.complex128)
                ref[0] = 1.0
                Oracle().run(ref, circuits.layered_u3_cz(n, depth, 10 * rep + k))
                assert np.abs(quest.state_vector(q) - ref).max() <= 1e-12
    finally:
        for q in regs:
            quest.destroyQureg(q, env)


def test_more_threads_than_slots(quest, env):
    """24 threads read their own registers: every one gets its own results."""
    n, errs = 9, []

    def work(t):
        q = quest.createQureg(n, env)
        try:
            re, im = _random(n, np.float64, t)
            ptr = C.POINTER(quest.qreal)
            for _ in range(6):
                quest.initStateFromAmps(q, re.ctypes.data_as(ptr), im.ctypes.data_as(ptr))
                quest.rotateZ(q, 0, 0.0)
                if np.abs(quest.state_vector(q) - (re + 1j * im)).max() > 1e-15:
                    errs.append(t)
                if abs(quest.calcTotalProb(q) - 1.0) > 1e-13:
                    errs.append(t)
        finally:
            quest.destroyQureg(q, env)

    ts = [threading.Thread(target=work, args=(t,)) for t in range(24)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errs


def test_read_of_the_unwritten_word(quest, env):
    """An amplitude whose bits are those of a word that no kernel has stored is still read."""
    n = 4
    bits = np.array([0x7FF4DEAD00BEEF01], dtype=np.uint64)
    re, im = np.zeros(1 << n), np.zeros(1 << n)
    re[3:4], im[5:6] = bits.view(np.float64), bits.view(np.float64)
    q = quest.createQureg(n, env)
    ptr = C.POINTER(quest.qreal)
    try:
        quest.initStateFromAmps(q, re.ctypes.data_as(ptr), im.ctypes.data_as(ptr))
        for _ in range(2):
            v = quest.state_vector(q)
            assert v.real.copy().view(np.uint64)[3] == bits[0] and v.imag.copy().view(np.uint64)[5] == bits[0]
            assert np.count_nonzero(v.real.copy().view(np.uint64)) == 1
    finally:
        quest.destroyQureg(q, env)
