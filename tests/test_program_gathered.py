"""CPU: device programs with gathered phases (op FAN) against the op semantics.

dq_build_program_gathered returns what dq_apply_blocks uploads.  The numpy
model of the FAN op follows gen_ops_asm.py: a thread's factor is the product
of the phases of the terms whose lane and workgroup condition hold, and it
multiplies the registers that the header's FM_* code selects.  Every other op
runs in the model of test_program_model.  The result must equal the ops
applied one at a time.

Tolerance: at most 160 ops, each a few roundings on values of order 1 to 10:
1e-12 in FP64 and 2e-5 with FP32 coefficients, as there.
"""
import ctypes as C

import numpy as np
import pytest

from dgquest_amd import circuits
from tests import helpers as H
from tests import test_program_model as M
from tests.test_program_model import GEN, eng, phases_of, run_ops  # noqa: F401  (eng is a fixture)


def build(eng, prec, R, ops):
    f = eng.dq_build_program_gathered
    f.argtypes = eng.dq_build_program.argtypes
    n = C.c_size_t()
    assert f(prec, R, ops.ctypes.data, len(ops), None, 0, C.byref(n)) == 0, eng.dq_last_error().decode()
    buf = np.zeros(n.value, dtype=np.uint8)
    assert f(prec, R, ops.ctypes.data, len(ops), buf.ctypes.data, len(buf) - 1, C.byref(n)) != 0
    assert f(prec, R, ops.ctypes.data, len(ops), buf.ctypes.data, len(buf), C.byref(n)) == 0
    return buf.tobytes()


def run_gathered(A, prog, prec, R, base):
    """Returns the number of FAN terms run."""
    ts = 8 if prec == 2 else 4
    codes = GEN.op_codes(R)
    end = np.array([codes.index(("END", ())), 0, 0, 0], dtype=np.uint32).tobytes()
    tid = np.arange(A.shape[0])
    at = terms = 0
    while True:
        code, mask, cthr, vthr = (int(x) for x in np.frombuffer(prog, dtype=np.uint32, count=4, offset=at))
        name, _ = codes[code]
        size = vthr if name == "FAN" else GEN.op_size(name, R, ts)
        assert not name.startswith("FM"), "reached through a FAN only"
        if name == "END":
            assert at + size == len(prog)
            return terms
        if name == "WG":
            c, v = np.frombuffer(prog, dtype=np.uint64, count=2, offset=at + 16)
            at += size + (vthr if (base & int(c)) != int(v) else 0)
            continue
        if name != "FAN":
            M.run_program(A, prog[at:at + size] + end, prec, R, base)
            at += size
            continue
        tb = GEN.FAN_TERM
        f = np.ones(A.shape[0], dtype=np.complex128)
        assert (size - 16) % tb == 0 and size > 16
        for k in range((size - 16) // tb):
            p = at + 16 + k * tb
            lane, wg = (int(x) for x in np.frombuffer(prog, dtype=np.uint32, count=2, offset=p))
            re, im = np.frombuffer(prog, dtype=np.float64, count=2, offset=p + 16)
            assert bool(wg & 0x400) == (p + tb == at + size)  # only the last term is marked
            terms += 1
            if wg & 0x100 and ((base >> (wg & 63)) ^ (wg >> 9)) & 1:
                continue
            f[(tid & (lane & 0xFFFF)) == lane >> 16] *= complex(re, im)
        fm, params = codes[mask]
        js = range(A.shape[1]) if fm == "FM_ALL" else [j for j in range(A.shape[1]) if ((j >> params[0]) & 1) == params[1]]
        for j in js:
            A[:, j] *= f
        at += size


def _circuit(kind, n, rng):
    if kind == "qft":
        return circuits.ghz_qft(n)
    if kind == "layered":
        return circuits.layered_u3_cz(n, 8, 5)
    if kind == "random":
        return H.random_circuit(rng, n, 160)
    out = []  # phases and flips: conditions on 0 too, several controls, signs
    for _ in range(60):
        a, b, c = (int(x) for x in rng.permutation(n)[:3])
        k = int(rng.integers(6))
        t = float(rng.uniform(-3, 3))
        out.append([("controlledPhaseShift", (a, b), (t,)), ("controlledRotateZ", (a, b), (t,)), ("pauliX", (a,), ()),
                    ("controlledPhaseFlip", (a, b), ()), ("multiControlledPhaseShift", (a, b, c), (t,)),
                    ("hadamard", (a,), ())][k])
    return out


@pytest.mark.parametrize("kind", ["qft", "layered", "random", "phases"])
@pytest.mark.parametrize("prec", [2, 1])
@pytest.mark.parametrize("shape", [(7, 4, 3), (6, 3, 3), (5, 4, 1), (4, 4, 0), (3, 2, 1), (7, 5, 2)])
def test_gathered_programs_match_ops(quest, quest32, eng, kind, prec, shape):  # noqa: F811
    lib = quest if prec == 2 else quest32
    rng = np.random.default_rng(100 * shape[0] + 10 * shape[1] + prec)
    n = 14
    tol = 1e-12 if prec == 2 else 2e-5
    terms = 0
    for R, W, ops, nontile in phases_of(lib, n, _circuit(kind, n, rng), shape):
        if len(ops) == 0:
            continue
        prog = build(eng, prec, R, ops)
        for _ in range(2):
            base = int(rng.integers(0, 1 << 62)) & nontile
            A0 = rng.normal(size=(64 << W, 1 << R)) + 1j * rng.normal(size=(64 << W, 1 << R))
            want = run_ops(A0.copy(), ops, prec, R, base)
            got = A0.copy()
            terms += run_gathered(got, prog, prec, R, base)
            assert np.abs(got - want).max() <= tol * max(1.0, np.abs(want).max())
    if kind == "qft":
        assert terms > 20  # the rewrite took place
