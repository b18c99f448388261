"""The work that users of this framework have it do, as measurable cases.

A case is one of
  circuit   record a circuit on a register that starts in a basis state, run it, read the result:
            the amplitudes on the host, P(0) of every qubit, or the state where it lies on the device
  step      one layer on a register that already holds a state, then P(0) of every qubit: the inner
            loop of a time evolution or of a variational search
  measure   a shallow circuit, then every qubit measured one after another
  sample    a circuit, then basis-state samples of its final state
  overlap   inner product of two registers
  dense     a grid circuit through the FP32 dense form (2^k x 2^k blocks on the matrix cores)
  serve     a batch of recorded circuits through the request server

Registers go from 10 to 30 qubits, as the request mix of dgquest_amd.circuits.serving_mix does, in both
precisions; circuit families and depths are those of that mix, of the benchmark (layered U3 + CZ, depth
24) and of the grid circuits of the tests.  Everything random comes from the seed: angles, pairings and
the basis state that a register starts in.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from dgquest_amd import quest as Q
from dgquest_amd import serve as S

F32, F64 = 1, 2
TWO_PI = 2.0 * math.pi


# --- cases --------------------------------------------------------------------
def listed():
    return [
        # a textbook program on a small register: launch and transfer latency
        {"name": "qft_n12_f64", "kind": "circuit", "circuit": "qft", "n": 12, "prec": F64, "depth": 1, "read": "amps"},
        # one energy evaluation of a variational search (odd size, FP32)
        {"name": "vqe_n17_f32", "kind": "circuit", "circuit": "hea", "n": 17, "prec": F32, "depth": 8, "read": "probs"},
        # a register that fits the caches, its state handed on on the device
        {"name": "layered_n21_f64", "kind": "circuit", "circuit": "layered", "n": 21, "prec": F64, "depth": 12, "read": "state"},
        # mostly diagonal work: a Fourier transform of a large odd register
        {"name": "qft_n27_f32", "kind": "circuit", "circuit": "qft", "n": 27, "prec": F32, "depth": 1, "read": "state"},
        # a random grid circuit in FP32, 4 x 7 qubits
        {"name": "grid_n28_f32", "kind": "circuit", "circuit": "grid", "n": 28, "prec": F32, "depth": 20, "read": "state"},
        # the benchmark circuit, with its expectation values
        {"name": "layered_n30_f64", "kind": "circuit", "circuit": "layered", "n": 30, "prec": F64, "depth": 24, "read": "probs"},
        # one Trotter step of a spin chain and its observables
        {"name": "step_n26_f64", "kind": "step", "n": 26, "prec": F64},
        # measuring a whole register, qubit by qubit
        {"name": "measure_n23_f64", "kind": "measure", "n": 23, "prec": F64, "depth": 2},
        # shots of a variational state
        {"name": "sample_n25_f64", "kind": "sample", "n": 25, "prec": F64, "depth": 4, "shots": 4096},
        # inner product of two variational states
        {"name": "overlap_n27_f64", "kind": "overlap", "n": 27, "prec": F64},
        # the dense form at its widest block
        {"name": "dense_n25_k7", "kind": "dense", "n": 25, "prec": F32, "depth": 20, "k": 7},
        # a burst of small requests that ask for expectation values, at the server's default precision
        {"name": "serve_64_f32", "kind": "serve", "n": 17, "prec": F32, "count": 64, "shots": 0},
    ]


def draw(rng):
    kind = rng.choice(["circuit", "circuit", "circuit", "circuit", "step", "measure", "sample", "overlap", "dense", "serve"])
    prec = rng.choice([F32, F64])
    if kind == "circuit":
        circuit = rng.choice(["qft", "hea", "layered", "grid"])
        n = rng.randint(10, 28)
        if circuit == "grid":
            n = rng.choice([12, 15, 16, 20, 21, 24, 25, 28])
        depth = {"qft": 1, "hea": rng.randint(4, 16), "layered": rng.randint(8, 24), "grid": rng.randint(6, 20)}[circuit]
        read = rng.choice(["probs", "state"] + (["amps"] if n <= 16 else []))
        return {"kind": kind, "circuit": circuit, "n": n, "prec": prec, "depth": depth, "read": read}
    if kind == "step":
        return {"kind": kind, "n": rng.randint(14, 29), "prec": prec}
    if kind == "measure":  # outcomes are whole numbers decided by P(0): FP64, where rounding does not decide them
        return {"kind": kind, "n": rng.randint(10, 25), "prec": F64, "depth": rng.randint(1, 4)}
    if kind == "sample":  # as above
        return {"kind": kind, "n": rng.randint(10, 27), "prec": F64, "depth": rng.randint(2, 8), "shots": int(2 ** rng.uniform(4, 13))}
    if kind == "overlap":
        return {"kind": kind, "n": rng.randint(12, 29), "prec": prec}
    if kind == "dense":
        return {"kind": kind, "n": rng.choice([15, 16, 20, 21, 24, 25]), "prec": F32, "depth": rng.randint(4, 20), "k": rng.choice([5, 6, 7])}
    shots = rng.choice([0, 64, 256]) if prec == F64 else 0
    return {"kind": kind, "n": rng.randint(12, 18), "prec": prec, "count": rng.randint(8, 96), "shots": shots}


# --- circuits: (gate, qubits, parameters), the names those of the QuEST API --------
def _angles(rs, prec, *shape):
    a = rs.uniform(0.0, TWO_PI, shape)
    return a.astype(np.float32).astype(np.float64) if prec == F32 else a  # what the API's real type holds


def _qft(n, prec):
    c = []
    for j in range(n):
        c.append(("hadamard", (j,), ()))
        for m in range(1, n - j):
            c.append(("controlledPhaseShift", (j, j + m), (math.pi / (1 << m),)))
    c += [("swapGate", (i, n - 1 - i), ()) for i in range(n // 2)]
    if prec == F32:
        c = [(g, q, tuple(float(np.float32(x)) for x in p)) for g, q, p in c]
    return c


def _hea(n, depth, rs, prec):
    c = []
    ay, az = _angles(rs, prec, depth, n), _angles(rs, prec, depth, n)
    for d in range(depth):
        c += [("rotateY", (q,), (float(ay[d, q]),)) for q in range(n)]
        c += [("rotateZ", (q,), (float(az[d, q]),)) for q in range(n)]
        c += [("controlledNot", (q, (q + 1) % n), ()) for q in range(n)]
    return c


def _layered(n, depth, rs, prec):
    c = []
    a = _angles(rs, prec, depth, n, 3)
    for d in range(depth):
        c += [("u3Gate", (q,), tuple(float(x) for x in a[d, q])) for q in range(n)]
        p = rs.permutation(n)
        c += [("controlledPhaseFlip", (int(p[k]), int(p[k + 1])), ()) for k in range(0, n - 1, 2)]
    return c


def _grid(n, depth, rs):
    rows = next(r for r in range(int(math.isqrt(n)), 0, -1) if n % r == 0)
    cols = n // rows
    last, c = [-1] * n, []
    for cyc in range(depth):
        for q in range(n):
            g = int(rs.randint(3)) if last[q] < 0 else (last[q] + 1 + int(rs.randint(2))) % 3
            last[q] = g
            c.append((("SqX", "SqY", "SqW")[g], (q,), ()))
        pat = cyc % 4
        if pat < 2:
            e = [(r * cols + k, r * cols + k + 1) for r in range(rows) for k in range(pat, cols - 1, 2)]
        else:
            e = [(r * cols + k, (r + 1) * cols + k) for r in range(pat - 2, rows - 1, 2) for k in range(cols)]
        c += [("controlledPhaseFlip", x, ()) for x in e]
    return c


def _trotter(n, rs, prec):
    """exp(-i dt (J sum Z Z + h sum X)) to first order on a ring, couplings of the seed."""
    j, h = 0.2 * rs.uniform(0.5, 1.5, n), 0.3 * rs.uniform(0.5, 1.5, n)
    if prec == F32:
        j, h = j.astype(np.float32).astype(np.float64), h.astype(np.float32).astype(np.float64)
    c = []
    for q in range(n):
        c.append(("controlledPhaseShift", (q, (q + 1) % n), (float(j[q]),)))
        c.append(("rotateZ", (q,), (float(j[q]),)))
    c += [("rotateX", (q,), (float(h[q]),)) for q in range(n)]
    return c


def _circuit(name, n, depth, rs, prec):
    if name == "qft":
        return _qft(n, prec)
    if name == "hea":
        return _hea(n, depth, rs, prec)
    if name == "layered":
        return _layered(n, depth, rs, prec)
    return _grid(n, depth, rs)


def _serve_circuits(case, rs):
    """(n, circuit) of each request: sizes 10..n and the families of the request mix, in an order that only the case decides."""
    out, mix = [], np.random.RandomState(case["n"] * 1000 + case["count"])
    for _ in range(case["count"]):
        n = int(mix.randint(10, case["n"] + 1))
        name = ("hea", "qft", "layered")[int(mix.choice(3, p=[0.4, 0.3, 0.3]))]
        depth = int(mix.randint(4, 17)) if name == "hea" else int(mix.randint(8, 25))
        out.append((n, _circuit(name, n, depth, rs, case["prec"])))
    return out


def _program(case, seed):
    """What the seed decides: the gates, the basis state at the start, and what else the kind needs."""
    rs = np.random.RandomState(int(seed) % (1 << 32))
    kind, n, prec = case["kind"], case["n"], case["prec"]
    if kind == "serve":
        return {"requests": _serve_circuits(case, rs), "seeds": [int(x) for x in rs.randint(1 << 31, size=case["count"])]}
    p = {"index": int(rs.randint(1 << min(n, 30)))}
    if kind == "circuit":
        p["gates"] = _circuit(case["circuit"], n, case["depth"], rs, prec)
    elif kind == "step":
        p["before"], p["gates"] = _layered(n, 1, rs, prec), _trotter(n, rs, prec)
    elif kind == "measure":
        p["gates"], p["key"] = _layered(n, case["depth"], rs, prec), int(rs.randint(1 << 31))
    elif kind == "sample":
        p["gates"], p["u"] = _hea(n, case["depth"], rs, prec), rs.uniform(0.0, 1.0, case["shots"])
    elif kind == "overlap":  # the same circuit, one of its layers turned a little
        p["gates"] = _layered(n, 1, rs, prec)
        p["other"] = p["gates"] + [("rotateX", (q,), (float(np.float32(0.1 * rs.uniform())),)) for q in range(n)]
    else:
        p["gates"] = _grid(n, case["depth"], rs)
    return p


# --- the framework's side -------------------------------------------------------
_env = {}


class _View:
    def __init__(self, register, ptr, prec):
        self.register = register
        self.__cuda_array_interface__ = {"shape": (int(register.q.numAmpsTotal),), "typestr": "<c16" if prec == F64 else "<c8",
                                         "data": (ptr, False), "version": 2}


class _Register:
    """A register that is given back with its last reference."""

    def __init__(self, case):
        self.api = Q.load(case["prec"])
        if case["prec"] not in _env:
            _env[case["prec"]] = self.api.createQuESTEnv()
        self.q = self.api.createQureg(case["n"], _env[case["prec"]])

    def __del__(self):
        self.api.destroyQureg(self.q, self.q.env)

    def state(self):
        """The state where it lies on the device, as a tensor that keeps the register: the memory is the register's."""
        prec = C.c_int()
        ptr = self.api.dgq_state_pointer(self.q, C.byref(prec))
        t = torch.as_tensor(_View(self, ptr, prec.value), device="cuda")
        t.register = self
        return t

    def probs(self):
        return np.array([self.api.calcProbOfOutcome(self.q, k, 0) for k in range(int(self.q.numQubitsRepresented))] +
                        [self.api.calcTotalProb(self.q)], dtype=np.float64 if self.api.prec == F64 else np.float32)


class _Serving:
    """A running server and the requests of one burst."""

    def __init__(self, case, p):
        api = Q.load(case["prec"])
        self.requests = S.RequestSet([S.record(api, n, c) for n, c in p["requests"]], [case["shots"]] * case["count"], p["seeds"])
        self.server = S.Server(api, prec=case["prec"], hbm_budget=4 << 30, recheck_fraction=0.0)

    def __del__(self):
        if hasattr(self, "server"):
            self.server.close()


def prepare(case, seed):
    p = _program(case, seed)
    kind = case["kind"]
    state = {"case": case, "p": p}
    if kind == "serve":
        state["serving"] = _Serving(case, p)
        return state
    r = state["reg"] = _Register(case)
    if kind == "step":
        r.api.initClassicalState(r.q, p["index"])
        r.api.apply_circuit(r.q, p["before"])
        r.api.dgq_flush(r.q)
    elif kind == "overlap":
        o = state["other"] = _Register(case)
        for reg, gates in ((r, p["gates"]), (o, p["other"])):
            reg.api.initClassicalState(reg.q, p["index"])
            reg.api.apply_circuit(reg.q, gates)
            reg.api.dgq_flush(reg.q)
    elif kind == "dense":
        r.api.dgq_set_dense(r.q, case["k"])
    if kind in ("step", "overlap"):
        r.api.dgq_sync(r.q)
        if kind == "overlap":
            state["other"].api.dgq_sync(state["other"].q)
    return state


def run(state):
    case, p = state["case"], state["p"]
    kind = case["kind"]
    if kind == "serve":
        v = state["serving"]
        res = v.server.replay(v.requests)
        real = np.float64 if case["prec"] == F64 else np.float32
        out = {"p0": np.concatenate([d["p0"] for d in res]).astype(real), "sum_z": np.array([d["sum_z"] for d in res], dtype=real)}
        if case["shots"]:
            out["samples"] = np.concatenate([d["samples"] for d in res]).astype(np.int64)
        return out
    r = state["reg"]
    api, q = r.api, r.q
    if kind == "overlap":
        z = api.calcInnerProduct(q, state["other"].q)
        return torch.tensor([z.real, z.imag], dtype=torch.float64 if case["prec"] == F64 else torch.float32)
    if kind != "step":
        api.initClassicalState(q, p["index"])
    if kind == "measure":
        api.seed([p["key"]])
    api.apply_circuit(q, p["gates"])
    if kind == "measure":
        outcomes, stats, prob = [], [], C.c_double()
        for k in range(case["n"]):
            outcomes.append(api.measureWithStats(q, k, C.byref(prob)))
            stats.append(prob.value)
        return {"outcomes": np.array(outcomes, dtype=np.int64), "probs": np.array(stats)}
    if kind == "sample":
        return S.sample(api, q, p["u"]).astype(np.int64)
    if kind == "dense" or case.get("read") == "state":
        return r.state()
    if case.get("read") == "amps":
        v = api.state_vector(q)
        return v if case["prec"] == F64 else v.astype(np.complex64)
    return r.probs()


# --- what a pass cannot do without ---------------------------------------------------
def _gate_flops(gates, n):
    """14 per amplitude for a 2x2 matrix, 7 with a control, 6 per amplitude that a diagonal touches."""
    per = 0.0
    for g, q, _ in gates:
        if g == "swapGate":
            continue
        if g == "controlledPhaseFlip":
            per += 0.25
        elif g == "controlledPhaseShift":
            per += 1.5
        elif g == "controlledNot":
            per += 0.0
        elif g == "rotateZ":
            per += 6.0
        else:
            per += 14.0
    return per * (1 << n)


def work(case):
    kind, n, prec = case["kind"], case["n"], case["prec"]
    amp = 16 if prec == F64 else 8
    state = amp << n
    p = _program(case, 1)
    if kind == "serve":
        return {"bytes": float(sum(2 * (amp << k) for k, _ in p["requests"])), "flops": sum(_gate_flops(c, k) for k, c in p["requests"])}
    if kind == "overlap":
        return {"bytes": 2.0 * state, "flops": 8.0 * (1 << n)}
    flops = _gate_flops(p["gates"], n)
    if kind == "step":  # read and written once; the observables while it is at hand
        return {"bytes": 2.0 * state, "flops": flops + 4.0 * (1 << n)}
    if kind == "measure":  # the probabilities need the state; a measured qubit halves what is left
        return {"bytes": 3.0 * state, "flops": flops + 8.0 * (1 << n)}
    if kind == "circuit" and case["read"] == "amps":
        return {"bytes": 2.0 * state, "flops": flops}
    if kind == "circuit" and case["read"] == "state" or kind == "dense":
        return {"bytes": 1.0 * state, "flops": flops}
    return {"bytes": 2.0 * state, "flops": flops + 4.0 * (1 << n)}  # written, and read for probabilities or samples


# --- the same in 64 bits, gate by gate --------------------------------------------------
def _matrix(g, p):
    h = 1.0 / math.sqrt(2.0)
    if g == "hadamard":
        return ((h, h), (h, -h))
    if g == "controlledNot":
        return ((0.0, 1.0), (1.0, 0.0))
    if g == "rotateX":
        c, s = math.cos(p[0] / 2), math.sin(p[0] / 2)
        return ((c, -1j * s), (-1j * s, c))
    if g == "rotateY":
        c, s = math.cos(p[0] / 2), math.sin(p[0] / 2)
        return ((c, -s), (s, c))
    if g == "u3Gate":
        t, f, l = p
        c, s = math.cos(t / 2), math.sin(t / 2)
        e = lambda x: complex(math.cos(x), math.sin(x))  # noqa: E731
        return ((c, -e(l) * s), (e(f) * s, e(f + l) * c))
    return {"SqX": ((h, -1j * h), (-1j * h, h)), "SqY": ((h, -h), (h, h)), "SqW": ((h, -0.5 - 0.5j), (0.5 - 0.5j, h))}[g]


def _simulate(v, n, gates):
    """The gates on the 2^n amplitudes v, in place; v[i] is the amplitude of basis state i of the qubits as the caller names them."""
    at = list(range(n))  # the bit of v's index that holds each qubit

    def part(bits, values):
        shape, index, top = [], [], n
        for b in sorted(bits, reverse=True):
            shape += [1 << (top - b - 1), 2]
            index += [slice(None), values[b]]
            top = b
        return v.view(shape + [1 << top])[tuple(index)]

    for g, q, p in gates:
        b = [at[x] for x in q]
        if g == "swapGate":
            at[q[0]], at[q[1]] = at[q[1]], at[q[0]]
        elif g == "controlledPhaseFlip":
            part(b, {b[0]: 1, b[1]: 1}).neg_()
        elif g == "controlledPhaseShift":
            part(b, {b[0]: 1, b[1]: 1}).mul_(complex(math.cos(p[0]), math.sin(p[0])))
        elif g == "rotateZ":
            part(b, {b[0]: 0}).mul_(complex(math.cos(p[0] / 2), -math.sin(p[0] / 2)))
            part(b, {b[0]: 1}).mul_(complex(math.cos(p[0] / 2), math.sin(p[0] / 2)))
        else:
            m = _matrix(g, p)
            on = {x: 1 for x in b[:-1]}
            x, y = part(b, {**on, b[-1]: 0}), part(b, {**on, b[-1]: 1})
            nx = x * m[0][0]
            nx.add_(y, alpha=m[0][1])
            y.mul_(m[1][1]).add_(x, alpha=m[1][0])
            x.copy_(nx)
    if at != list(range(n)):
        v = v.view([2] * n) if n <= 16 else v
        if v.dim() == 1:  # gather through the map, a piece at a time
            out = torch.empty_like(v)
            step = 1 << min(n, 22)
            for s in range(0, 1 << n, step):
                i = torch.arange(s, s + step, device=v.device)
                j = torch.zeros_like(i)
                for k in range(n):
                    j |= ((i >> k) & 1) << at[k]
                out[s:s + step] = v[j]
            return out
        return v.permute([n - 1 - at[n - 1 - d] for d in range(n)]).reshape(-1)
    return v


def _start(n, index):
    v = torch.zeros(1 << n, dtype=torch.complex128, device="cuda")
    v[index] = 1.0
    return v


def _probs(v, n):
    w = torch.view_as_real(v).square().sum(dim=1)
    return np.array([float(w.view(-1, 2, 1 << k)[:, 0].sum()) for k in range(n)] + [float(w.sum())])


def exact(case, seed):
    kind, n = case["kind"], case["n"]
    if n > 28:
        return None  # over about 20 seconds
    p = _program(case, seed)
    if kind == "sample":
        return None  # whole numbers
    if kind == "serve":
        probs = [_probs(_simulate(_start(k, 0), k, c), k) for k, c in p["requests"]]
        sum_z = [float(sum(2.0 * x[:-1] - x[-1])) for x in probs]
        return {"p0": np.concatenate(probs), "sum_z": np.array(sum_z), "samples": None}
    v = _start(n, p["index"])
    if kind == "overlap":
        a = _simulate(v, n, p["gates"])
        b = _simulate(_start(n, p["index"]), n, p["other"])
        z = torch.view_as_real(a.conj().mul(b)).sum(dim=0)
        return z.cpu()
    if kind == "step":
        v = _simulate(v, n, p["before"])
    v = _simulate(v, n, p["gates"])
    if kind == "measure":
        mt, stats = np.random.RandomState([p["key"]]), []
        for k in range(n):
            w = v.view(-1, 2, 1 << k)
            zero = float(torch.view_as_real(w[:, 0]).square().sum())
            if zero < 1e-13 or 1.0 - zero < 1e-13:
                out = 1 if zero < 1e-13 else 0
            else:
                out = int(int(mt.randint(0, 1 << 32, dtype=np.uint32)) * (1.0 / 4294967295.0) > zero)
            prob = zero if out == 0 else 1.0 - zero
            stats.append(prob)
            w[:, 1 - out] = 0
            w[:, out] *= 1.0 / math.sqrt(prob)
        return {"outcomes": None, "probs": np.array(stats)}
    if kind == "step" or case.get("read") == "probs":
        return _probs(v, n)
    return v
