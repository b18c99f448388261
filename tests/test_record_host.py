"""apply_circuit records natively what apply() records gate by gate (no GPU)."""
import ctypes as C

import numpy as np
import pytest

from dgquest_amd import quest as Q
from dgquest_amd import serve as S

N = 6


def _gates():
    """One gate of every signature, distinct qubits, unitary parameters."""
    rs = np.random.RandomState(5)
    out = []
    for name, ks in Q.GATE_SIGNATURES.items():
        qubits = [int(x) for x in rs.permutation(N)]
        nq = sum(1 for k in ks if k == "q") + (3 if "qs" in ks else 0)
        par = []
        for k in ks:
            if k == "r":
                par += [float(rs.uniform(0, 6))]
            elif k == "c":  # (alpha, beta): the pair is unit
                par += [0.6, 0.0] if not par else [0.0, 0.8]
            elif k == "m":
                par += [0.0, 0.0, 1.0, 0.0, 0.0, 1.0, 0.0, 0.0]
            elif k == "v":
                par += [1.0, -2.0, 0.5]
        out.append((name, tuple(qubits[:nq]), tuple(par)))
    return out


def _rec(api, circuit):
    r = S.record(api, N, circuit)
    return r.gates.tobytes(), r.l2p.tobytes()


def _plain(api, circuit):
    """The same through apply() alone."""
    class Plain(type(api)):
        def apply(self, *a):
            return super().apply(*a)

    p = Plain.__new__(Plain)
    p.__dict__.update(api.__dict__)
    return _rec(p, circuit)


FORMS = {
    "tuples": lambda c: c,
    "lists": lambda c: [[g, list(q), list(p)] for g, q, p in c],
    "no params entry": lambda c: [(g, q) if not p else (g, q, p) for g, q, p in c],
    "numpy numbers": lambda c: [(g, tuple(np.int64(x) for x in q), tuple(np.float32(x) for x in p)) for g, q, p in c
                                if not set(Q.GATE_SIGNATURES[g]) & set("cm")],  # 32-bit pairs are not unitary to REAL_EPS
    "numpy arrays": lambda c: [(g, np.array(q), np.array(p)) for g, q, p in c],
    "integers and text as reals": lambda c: [(g, tuple(str(x) for x in q), tuple(int(x) for x in p)) for g, q, p in c
                                             if set(Q.GATE_SIGNATURES[g]) <= {"q", "r"}],
    "further entries": lambda c: [(g, q + (0,), p + (1.0,), "x") for g, q, p in c if "qs" not in Q.GATE_SIGNATURES[g]],
    "a generator": lambda c: (x for x in c),
}


@pytest.mark.parametrize("prec", [1, 2])
@pytest.mark.parametrize("form", sorted(FORMS))
def test_native_record_equals_gate_by_gate(prec, form):
    api = Q.load(prec)
    assert _rec(api, FORMS[form](_gates())) == _plain(api, FORMS[form](_gates()))


@pytest.mark.parametrize("bad,exc", [(("noSuchGate", (0,), ()), KeyError), (("rotateX", (0,), ()), IndexError),
                                     (("controlledNot", (0,), ()), IndexError), (("rotateX", (0,), ("x",)), ValueError),
                                     (("hadamard",), IndexError), (7, TypeError)])
def test_a_bad_entry_raises_after_the_ones_before_it(bad, exc):
    api = Q.load(2)
    q = api.dgq_create_recorder(N)
    S._bind(api.lib)
    try:
        with pytest.raises(exc):
            api.apply_circuit(q, [("hadamard", (0,), ()), bad, ("hadamard", (1,), ())])
        cnt = C.c_int()
        api.dgq_recorder_export(q, None, 0, C.byref(cnt), None, None, None, None)
        assert cnt.value == 1
    finally:
        api.dgq_destroy_recorder(q)
    with pytest.raises(TypeError):
        api.apply_circuit(q, 5)
