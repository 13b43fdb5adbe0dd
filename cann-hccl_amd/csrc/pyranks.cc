// The loop over the ranks of one process, for the Python mirror (module _hccl_ranks).
//
// A program that drives all p ranks from one thread makes p calls of the C API per collective.  Through ctypes each of
// them costs 0.5 us and more of argument conversion, several times the call itself.  Here the sequences are read once and
// the p calls are made in C++, in rank order, without the interpreter's lock (a rank may block in its call).  Measured
// per collective: 8-rank all-reduce of 8 KiB 7.6 us through ctypes, 4.4 us here; 64-rank all-to-all-v of short blocks,
// tables as numpy arrays, 80 us and 29 us.
//
// Whatever this loop does not recognise (other sequence or pointer types than lists or tuples of integers, None and
// c_void_p) it leaves alone: call() then returns -1 before any call was made and the caller goes through ctypes.
//
// The functions are those of the library that the mirror has loaded, handed over by bind(): were this module linked
// against the library, a libhccl.so elsewhere on the loader's search path could be taken for it.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>
#include <cstring>

#include "hccl/hccl.h"
#include "hccl/hccl_amd_ext.h"

namespace {

enum Kind : long {
    ALL_REDUCE = 0, REDUCE_SCATTER, REDUCE_SCATTER_NO_ALLOC, ALL_GATHER, ALL_TO_ALL, BROADCAST, REDUCE, SCATTER, ALL_TO_ALL_V,
    KIND_COUNT
};

// in the order of Kind
struct Functions {
    decltype(&HcclAllReduce) allReduce;
    decltype(&HcclReduceScatter) reduceScatter;
    decltype(&HcclAmdReduceScatterNoAlloc) reduceScatterNoAlloc;
    decltype(&HcclAllGather) allGather;
    decltype(&HcclAlltoAll) allToAll;
    decltype(&HcclBroadcast) broadcast;
    decltype(&HcclReduce) reduce;
    decltype(&HcclScatter) scatter;
    decltype(&HcclAlltoAllV) allToAllV;
};
static_assert(sizeof(Functions) == KIND_COUNT * sizeof(void *), "one function per kind");
Functions g_fn = {};

constexpr Py_ssize_t kMostRanks = 64;
PyObject *g_valueName = nullptr;      // "value"
PyTypeObject *g_voidPointer = nullptr;   // ctypes.c_void_p

// None, an integer, or a ctypes.c_void_p; 1 = converted.
int AsPointer(PyObject *o, void **out)
{
    if (o == Py_None) {
        *out = nullptr;
        return 1;
    }
    if (PyLong_CheckExact(o)) {
        *out = reinterpret_cast<void *>(static_cast<uintptr_t>(PyLong_AsUnsignedLongLongMask(o)));
        if (PyErr_Occurred()) {
            PyErr_Clear();
            return 0;
        }
        return 1;
    }
    if (Py_TYPE(o) == g_voidPointer) {
        PyObject *v = PyObject_GetAttr(o, g_valueName);
        if (v == nullptr) {
            PyErr_Clear();
            return 0;
        }
        const int ok = (v == Py_None || PyLong_CheckExact(v)) ? AsPointer(v, out) : 0;
        Py_DECREF(v);
        return ok;
    }
    return 0;
}

int AsNumber(PyObject *o, uint64_t *out)
{
    if (!PyLong_CheckExact(o)) {
        return 0;
    }
    *out = PyLong_AsUnsignedLongLongMask(o);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        return 0;
    }
    return 1;
}

bool Plain(PyObject *o) { return PyList_CheckExact(o) || PyTuple_CheckExact(o); }

// A p x p table of 64-bit unsigned integers, row by row without gaps (a numpy array, for one).
struct Table {
    Py_buffer view = {};
    bool held = false;
    ~Table() { Drop(); }
    void Drop()
    {
        if (held) {
            PyBuffer_Release(&view);
            held = false;
        }
    }
    bool Take(PyObject *o, Py_ssize_t p)
    {
        if (!PyObject_CheckBuffer(o) || PyObject_GetBuffer(o, &view, PyBUF_FORMAT | PyBUF_C_CONTIGUOUS) != 0) {
            PyErr_Clear();
            return false;
        }
        held = true;
        const char *f = view.format;
        return f != nullptr && (f[0] == 'L' || f[0] == 'Q') && f[1] == 0 && view.itemsize == 8 && view.ndim == 2 && view.shape[0] == p &&
            view.shape[1] == p;
    }
};

// call(kind, comms, sends, recvs, count, dtype, op, root, stream, tables) -> HcclResult of the first call that failed, 0, or
// -1 (not recognised, nothing called).  tables: None, or the four p x p tables of an all-to-all-v.
PyObject *Call(PyObject *, PyObject *const *args, Py_ssize_t nargs)
{
    PyObject *const no = PyLong_FromLong(-1);
    if (no == nullptr || nargs != 10 || g_fn.allReduce == nullptr || !PyLong_CheckExact(args[0])) {
        return no;
    }
    const long kind = PyLong_AsLong(args[0]);
    if (kind < 0 || kind >= KIND_COUNT || !Plain(args[1]) || !Plain(args[2]) || !Plain(args[3])) {
        PyErr_Clear();
        return no;
    }
    // as zip() does: as many ranks as the shortest of the three
    Py_ssize_t p = PySequence_Fast_GET_SIZE(args[1]);
    for (int i = 2; i <= 3; i++) {
        const Py_ssize_t n = PySequence_Fast_GET_SIZE(args[i]);
        p = n < p ? n : p;
    }
    uint64_t count = 0, dtype = 0, op = 0, root = 0;
    void *stream = nullptr;
    if (p > kMostRanks || !AsNumber(args[4], &count) || !AsNumber(args[5], &dtype) || !AsNumber(args[6], &op) || !AsNumber(args[7], &root) ||
        !AsPointer(args[8], &stream)) {
        return no;
    }
    void *comm[kMostRanks], *send[kMostRanks], *recv[kMostRanks];
    for (Py_ssize_t r = 0; r < p; r++) {
        if (!AsPointer(PySequence_Fast_GET_ITEM(args[1], r), &comm[r]) || !AsPointer(PySequence_Fast_GET_ITEM(args[2], r), &send[r]) ||
            !AsPointer(PySequence_Fast_GET_ITEM(args[3], r), &recv[r])) {
            return no;
        }
    }
    Table table[4];
    const uint64_t *t[4] = {};
    if (kind == ALL_TO_ALL_V) {
        if (!Plain(args[9]) || PySequence_Fast_GET_SIZE(args[9]) != 4 || p != PySequence_Fast_GET_SIZE(args[1])) {
            return no;
        }
        for (int i = 0; i < 4; i++) {
            if (!table[i].Take(PySequence_Fast_GET_ITEM(args[9], i), p)) {
                return no;
            }
            t[i] = static_cast<const uint64_t *>(table[i].view.buf);
        }
    }
    Py_DECREF(no);
    const HcclDataType dt = static_cast<HcclDataType>(static_cast<int32_t>(dtype));
    const HcclReduceOp ro = static_cast<HcclReduceOp>(static_cast<int32_t>(op));
    const uint32_t rt = static_cast<uint32_t>(root);
    HcclResult res = HCCL_SUCCESS;
    Py_BEGIN_ALLOW_THREADS
    for (Py_ssize_t r = 0; r < p && res == HCCL_SUCCESS; r++) {
        switch (kind) {
            case ALL_REDUCE: res = g_fn.allReduce(send[r], recv[r], count, dt, ro, comm[r], stream); break;
            case REDUCE_SCATTER: res = g_fn.reduceScatter(send[r], recv[r], count, dt, ro, comm[r], stream); break;
            case REDUCE_SCATTER_NO_ALLOC: res = g_fn.reduceScatterNoAlloc(send[r], recv[r], count, dt, ro, comm[r], stream); break;
            case ALL_GATHER: res = g_fn.allGather(send[r], recv[r], count, dt, comm[r], stream); break;
            case ALL_TO_ALL: res = g_fn.allToAll(send[r], count, dt, recv[r], count, dt, comm[r], stream); break;
            case BROADCAST: res = g_fn.broadcast(send[r], count, dt, rt, comm[r], stream); break;
            case REDUCE: res = g_fn.reduce(send[r], recv[r], count, dt, ro, rt, comm[r], stream); break;
            case SCATTER: res = g_fn.scatter(send[r], recv[r], count, dt, rt, comm[r], stream); break;
            default:
                res = g_fn.allToAllV(send[r], t[0] + r * p, t[1] + r * p, dt, recv[r], t[2] + r * p, t[3] + r * p, dt, comm[r], stream);
                break;
        }
    }
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(static_cast<long>(res));
}

// bind(addresses): the library's functions, in the order of Kind, as integers.
PyObject *Bind(PyObject *, PyObject *addresses)
{
    if (!PyTuple_CheckExact(addresses) || PyTuple_GET_SIZE(addresses) != KIND_COUNT) {
        PyErr_SetString(PyExc_TypeError, "bind: a tuple of one address per collective");
        return nullptr;
    }
    void *address[KIND_COUNT];
    for (long k = 0; k < KIND_COUNT; k++) {
        address[k] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(addresses, k));
        if (address[k] == nullptr) {
            if (!PyErr_Occurred()) {
                PyErr_SetString(PyExc_ValueError, "bind: null address");
            }
            return nullptr;
        }
    }
    std::memcpy(&g_fn, address, sizeof(g_fn));
    Py_RETURN_NONE;
}

PyMethodDef g_methods[] = {
    {"call", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(Call)), METH_FASTCALL, "one collective, called for every rank"},
    {"bind", Bind, METH_O, "the functions that call() calls"},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_hccl_ranks", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__hccl_ranks()
{
    PyObject *ctypes = PyImport_ImportModule("ctypes");
    if (ctypes == nullptr) {
        return nullptr;
    }
    g_voidPointer = reinterpret_cast<PyTypeObject *>(PyObject_GetAttrString(ctypes, "c_void_p"));
    Py_DECREF(ctypes);
    g_valueName = PyUnicode_InternFromString("value");
    if (g_voidPointer == nullptr || g_valueName == nullptr) {
        return nullptr;
    }
    return PyModule_Create(&g_module);
}
