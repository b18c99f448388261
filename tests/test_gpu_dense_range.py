"""GPU: the dense form over the range of FP32, in the amplitudes and in the matrices.

FP32 keeps 24 bits down to 2^-126, and the kernel's split of a factor into bf16
pieces has to keep them too: registers scaled by powers of two against the FP64
oracle on the register's own (rounded) amplitudes, in the L2 norm relative to the
state's.  An op rounds its matrix, leaves out piece products below 2^-24 and adds
up at most 18 times, each 2^-24 of a result and independent: 2.7e-7, at most 8 ops
one after another 8e-7; 2e-6 is allowed.  Besides, each of 8 blocks may round
2^14 amplitudes of two parts to denormal numbers as it reads and writes them: 2^-150 each.

Matrix entries: k equal small rotations of k qubits in |0...0>, one op; the last
amplitude is the product of the sines, a matrix entry of 1e-37, within the 2^-24 of
each piece product (three are left out or rounded) and of the stored result: 1e-6.
"""
import ctypes as C
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [-124, -118, -112, -100, 0, 40, 62, 70, 100, 115])
@pytest.mark.parametrize("k", [5, 6, 7])
def test_scaled_registers(k, scale, quest32, env32, oracle):
    n = 14
    rng = np.random.default_rng(k)
    v = rng.standard_normal((2, 1 << n))
    v /= np.sqrt((v ** 2).sum())
    gates = [("u3Gate", (q,), tuple(float(np.float32(x)) for x in rng.uniform(0, 6, 3))) for q in range(n)]
    gates += [("controlledPhaseFlip", (q, (q + 3) % n), ()) for q in range(0, n, 2)]
    re, im = np.ldexp(v, scale).astype(np.float32)
    ref = oracle.run(np.ldexp(1.0, -scale) * (re.astype(np.float64) + 1j * im.astype(np.float64)), gates)
    q = quest32.createQureg(n, env32)
    try:
        quest32.initStateFromAmps(q, *(x.ctypes.data_as(C.POINTER(C.c_float)) for x in (re, im)))
        assert quest32.dgq_set_dense(q, k) == 0
        quest32.apply_circuit(q, gates)
        out = np.ldexp(1.0, -scale) * quest32.state_vector(q)
        assert quest32.dense_stats(q)["ops"] <= 8
    finally:
        quest32.destroyQureg(q, env32)
    denormal = 2 * 8 * np.sqrt(2 << n) * np.ldexp(1.0, -150 - scale)
    assert np.linalg.norm(out - ref) <= (2e-6 + denormal) * np.linalg.norm(ref)


@pytest.mark.parametrize("k", [5, 6, 7])
def test_small_matrix_entries(k, quest32, env32):
    n = 13
    angle = float(np.float32(2.0 * 10.0 ** (-37.0 / k)))
    q = quest32.createQureg(n, env32)
    try:
        quest32.initZeroState(q)
        assert quest32.dgq_set_dense(q, k) == 0
        quest32.apply_circuit(q, [("rotateY", (i,), (angle,)) for i in range(k)])
        a = quest32.getAmp(q, (1 << k) - 1)
        want = math.sin(angle / 2) ** k
        assert abs(a.real / want - 1.0) <= 1e-6 and a.imag == 0.0
    finally:
        quest32.destroyQureg(q, env32)
