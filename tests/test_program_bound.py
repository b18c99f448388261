"""CPU: device programs stay within the workspace that dq_apply_ws_bytes reserves for them.

dq_apply_blocks refuses a plan whose programs outgrow that part of the
workspace, so no plan may.  Checked on the ops of plans with diagonal gates
left unmerged (every tile shape), and on the runs of diagonal ops that cost
most: tables made of a few plain phases, copied for two workgroup bits.
"""
import ctypes as C

import numpy as np
import pytest

from dgquest_amd import quest as Q
from tests.test_program_model import K_MAT, K_NEG, K_PHASE, K_SHEAR, eng  # noqa: F401  (eng is a fixture)

READ_AHEAD = 256  # of the interpreter, part of what is reserved


def align(x):
    return (x + 255) // 256 * 256


def room(eng, n_phases, n_ops):  # noqa: F811
    """Bytes reserved for the programs: what is left of the workspace of no blocks and jobs."""
    f = eng.dq_apply_ws_bytes
    f.restype = C.c_size_t
    return f(0, n_phases, n_ops, 0) - align(64 * n_phases) - align(104 * n_ops) - align(144 * 4 * n_phases)


def size(eng, prec, R, ops, gathered=True):  # noqa: F811
    f = eng.dq_build_program_gathered if gathered else eng.dq_build_program
    f.argtypes = [C.c_int, C.c_int, C.c_void_p, C.c_uint32, C.c_void_p, C.c_size_t, C.POINTER(C.c_size_t)]
    n = C.c_size_t()
    assert f(prec, R, ops.ctypes.data, len(ops), None, 0, C.byref(n)) == 0, eng.dq_last_error().decode()
    return n.value


def _op(kind, prec, c_reg=0, v_reg=0, c_wg=0, v_wg=0, c_thr=0, tbit=0):
    o = np.zeros(1, dtype=Q.OP_DT)
    o["kind"], o["tbit"], o["c_reg"], o["v_reg"], o["c_wg"], o["v_wg"], o["c_thr"] = kind, tbit, c_reg, v_reg, c_wg, v_wg, c_thr
    m = np.linspace(0.3, 0.8, 8)
    o["m"][0] = m if prec == 2 else np.frombuffer(m.astype(np.float32).tobytes() + bytes(32), dtype=np.float64)
    return o


def _phases(prec, R, plain, wg, end):
    """One run: `plain` unconditioned phases that make a table, `wg` with a workgroup bit each, then what ends it."""
    run = [_op(K_PHASE, prec, c_reg=1 << (i % R) if i > 1 else 0) for i in range(plain)]
    run += [_op(K_PHASE, prec, c_wg=1 << (20 + i), v_wg=1 << (20 + i)) for i in range(wg)]
    if end:
        run.append(_op(end, prec))
    return run


@pytest.mark.parametrize("prec", [1, 2])
@pytest.mark.parametrize("R", [1, 2, 3, 4, 5])
def test_tables_of_plain_phases(eng, prec, R):  # noqa: F811
    for plain in (2, 3, 4, 6):
        for wg in (0, 1, 2, 3):
            for end in (K_SHEAR, K_MAT):
                ops = np.concatenate(_phases(prec, R, plain, wg, end) * 20)
                for gathered in (False, True):
                    need = size(eng, prec, R, ops, gathered) + READ_AHEAD
                    assert need <= room(eng, 1, len(ops)), (plain, wg, end, gathered)
    ops = np.concatenate(_phases(prec, R, 2, 2, 0))  # the smallest run, nothing after it
    assert size(eng, prec, R, ops) + READ_AHEAD <= room(eng, 1, len(ops))


@pytest.mark.parametrize("prec", [1, 2])
@pytest.mark.parametrize("R", [1, 3, 5])
def test_random_runs(eng, prec, R):  # noqa: F811
    rng = np.random.default_rng(10 * R + prec)
    for _ in range(60):
        ops = []
        for _ in range(12):
            for _ in range(int(rng.integers(1, 9))):
                kind = K_PHASE if rng.integers(2) else K_NEG
                c = int(rng.integers(1 << R)) if rng.integers(2) else 0
                wg = 1 << int(rng.integers(20, 23)) if rng.integers(3) == 0 else 0
                thr = int(rng.integers(1, 64)) if rng.integers(4) == 0 else 0
                ops.append(_op(kind, prec, c_reg=c, v_reg=c & int(rng.integers(1 << R)), c_wg=wg, v_wg=wg * int(rng.integers(2)), c_thr=thr))
            for b in range(int(rng.integers(0, R + 1))):
                ops.append(_op(K_SHEAR if rng.integers(2) else K_MAT, prec, tbit=b))
        ops = np.concatenate(ops)
        assert size(eng, prec, R, ops) + READ_AHEAD <= room(eng, 1, len(ops))


@pytest.mark.parametrize("prec", [1, 2])
@pytest.mark.parametrize("fuse", [False, True])
@pytest.mark.parametrize("shape", [(5, 5, 0), (6, 5, 1), (7, 5, 2), (7, 4, 3), (6, 3, 3)])
def test_plans_of_phase_circuits(quest, quest32, eng, prec, fuse, shape):  # noqa: F811
    lib = quest if prec == 2 else quest32
    n = 20
    for seed in range(6):
        rng = np.random.default_rng(seed)
        circ = []
        for _ in range(300):
            a, b = (int(x) for x in rng.permutation(n)[:2])
            t = float(rng.uniform(0.1, 3))
            circ.append([("tGate", (a,), ()), ("phaseShift", (a,), (t,)), ("controlledPhaseShift", (a, b), (t,)),
                         ("controlledNot", (a, b), ())][int(rng.choice(4, p=[0.3, 0.3, 0.3, 0.1]))])
        r = lib.dgq_create_recorder(n)
        lib.apply_circuit(r, circ)
        blocks, phases, ops, _ = lib.recorder_plan(r, k=shape[0], R=shape[1], W=shape[2], fuse=fuse)
        lib.dgq_destroy_recorder(r)
        total = 0
        for blk in blocks:
            for p in phases[int(blk["phase_begin"]):int(blk["phase_begin"] + blk["phase_count"])]:
                part = ops[int(p["op_begin"]):int(p["op_begin"] + p["op_count"])].copy()
                total += size(eng, prec, int(blk["reg_bits"]), part) if len(part) else 16
        assert total + READ_AHEAD <= room(eng, len(phases), len(ops)), seed
