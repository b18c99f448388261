// pyrecord.cpp -- records a Python circuit (a sequence of (name, qubits, params)
// entries) through the QuEST C API without a Python-level call per gate.
//
// Recording a gate is a few tens of nanoseconds of C; building its argument
// list in Python and passing it through ctypes took 0.75-1.0 us, which for
// registers up to about 21 qubits was more than the GPU's part of the pass
// (12 qubits, 84 gates: 66 of 140 us; 21 qubits, 372 gates: 386 of 745 us).
//
// Called through ctypes.PyDLL: the interpreter lock is held, but for a moment
// every kGatesPerTurn gates, and a Python exception left set on return is raised
// by the caller.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>

#include "QuEST.h"

namespace {

// Argument shapes recorded here; every other gate goes to the fallback.
enum Shape { Q, QR, QRR, QRRR, QQ, QQR, QQRR, NUM_SHAPES };
constexpr int kQubits[NUM_SHAPES] = {1, 1, 1, 1, 2, 2, 2};
constexpr int kReals[NUM_SHAPES] = {0, 1, 2, 3, 0, 1, 2};

// qreal is a parameter: both precisions share this library (Qureg holds no reals).
template <typename T>
void call(void *f, int shape, const Qureg &r, const int *q, const double *p) {
    switch (shape) {
        case Q: ((void (*)(Qureg, int))f)(r, q[0]); break;
        case QR: ((void (*)(Qureg, int, T))f)(r, q[0], (T)p[0]); break;
        case QRR: ((void (*)(Qureg, int, T, T))f)(r, q[0], (T)p[0], (T)p[1]); break;
        case QRRR: ((void (*)(Qureg, int, T, T, T))f)(r, q[0], (T)p[0], (T)p[1], (T)p[2]); break;
        case QQ: ((void (*)(Qureg, int, int))f)(r, q[0], q[1]); break;
        case QQR: ((void (*)(Qureg, int, int, T))f)(r, q[0], q[1], (T)p[0]); break;
        case QQRR: ((void (*)(Qureg, int, int, T, T))f)(r, q[0], q[1], (T)p[0], (T)p[1]); break;
    }
}

// Gates (under 0.1 us each) between two chances for other threads and signal handlers,
// which an interpreted loop gives at every gate.
constexpr unsigned kGatesPerTurn = 256;

bool plain_list(PyObject *o) { return PyTuple_CheckExact(o) || PyList_CheckExact(o); }

// The gate as C arguments if its entry holds nothing but plain tuples or lists
// of exact ints and floats (no Python code runs while it is read); false sends
// it to the fallback, which decides what it means or raises.
bool read_gate(PyObject *g, PyObject *table, void *&f, int &shape, int *q, double *p) {
    if (!plain_list(g) || PySequence_Fast_GET_SIZE(g) < 2) return false;
    PyObject **it = PySequence_Fast_ITEMS(g);
    if (!PyUnicode_CheckExact(it[0])) return false;
    PyObject *e = PyDict_GetItemWithError(table, it[0]);
    if (!e) return false;
    shape = (int)PyLong_AsLong(PyTuple_GET_ITEM(e, 0));
    f = PyLong_AsVoidPtr(PyTuple_GET_ITEM(e, 1));
    const int nq = kQubits[shape], nr = kReals[shape];
    if (!plain_list(it[1]) || PySequence_Fast_GET_SIZE(it[1]) < nq) return false;
    PyObject **qs = PySequence_Fast_ITEMS(it[1]);
    for (int i = 0; i < nq; i++) {
        if (!PyLong_CheckExact(qs[i])) return false;
        q[i] = (int)PyLong_AsUnsignedLongMask(qs[i]);  // wraps as a C int argument does
    }
    if (nr == 0) return true;
    if (PySequence_Fast_GET_SIZE(g) < 3 || !plain_list(it[2]) || PySequence_Fast_GET_SIZE(it[2]) < nr) return false;
    PyObject **ps = PySequence_Fast_ITEMS(it[2]);
    for (int i = 0; i < nr; i++) {
        if (!PyFloat_CheckExact(ps[i])) return false;
        p[i] = PyFloat_AS_DOUBLE(ps[i]);
    }
    return true;
}

}  // namespace

// Records every entry of the iterable `circuit` on *reg, in order.  table: gate
// name -> (shape, address of the gate's C function) of the precision `prec`.
// fallback(entry) applies an entry that is not in plain form.
extern "C" PyObject *dgq_py_record(PyObject *table, PyObject *fallback, int prec, const Qureg *reg, PyObject *circuit) {
    PyObject *iter = PyObject_GetIter(circuit);
    if (!iter) return nullptr;
    const Qureg r = *reg;
    unsigned turn = 0;
    while (PyObject *g = PyIter_Next(iter)) {
        void *f = nullptr;
        int shape = 0, q[2];
        double p[3];
        bool ok = true;
        if (read_gate(g, table, f, shape, q, p)) {
            if (prec == 2) call<double>(f, shape, r, q, p);
            else call<float>(f, shape, r, q, p);
        } else if (!PyErr_Occurred()) {
            PyObject *res = PyObject_CallFunctionObjArgs(fallback, g, nullptr);
            ok = res != nullptr;
            Py_XDECREF(res);
        } else {
            ok = false;
        }
        Py_DECREF(g);
        if (!ok) break;
        if (++turn % kGatesPerTurn == 0) {
            if (PyErr_CheckSignals()) break;
            Py_BEGIN_ALLOW_THREADS
            Py_END_ALLOW_THREADS
        }
    }
    Py_DECREF(iter);
    if (PyErr_Occurred()) return nullptr;
    Py_RETURN_NONE;
}
