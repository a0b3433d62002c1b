// Ragged Python lists to flat arrays.  A batch of rollouts reaches the packer as lists of Python numbers;
// walking them through numpy's iterator protocol takes about 10 ns per number, most of it in calls per element.
// Here exact lists of exact numbers are read straight from the list storage.  Anything else is left to the
// caller's general path: every function returns a negative number for it and promises nothing about its outputs.
//
// Called with the interpreter lock held (ctypes.PyDLL).  Nothing here runs Python code or gives the lock up, so
// a list cannot change while it is read; it may have changed since its length was taken, which is checked.
#include <Python.h>

#include <cstdint>

namespace {
constexpr Py_ssize_t AHEAD = 16;  // numbers lie scattered on the heap: their cache lines are requested early

// sequence i of `seqs`, when it is an exact list of the length that `offsets` says
PyObject* row(PyObject* seqs, Py_ssize_t i, const int64_t* offsets) {
    PyObject* s = PyList_GET_ITEM(seqs, i);
    return PyList_CheckExact(s) && PyList_GET_SIZE(s) == offsets[i + 1] - offsets[i] ? s : nullptr;
}
bool as_int(PyObject* o, int64_t* v) {
    if (PyLong_CheckExact(o)) {
        int overflow = 0;
        *v = PyLong_AsLongLongAndOverflow(o, &overflow);
        return overflow == 0;
    }
    if (!PyBool_Check(o)) return false;
    *v = o == Py_True;
    return true;
}
// each(sequence, position in the flat array, value) for every element; false: not lists of numbers
template <class Read, class Each>
bool walk(PyObject* seqs, const int64_t* offsets, int64_t n, Read&& read, Each&& each) {
    if (!PyList_CheckExact(seqs) || PyList_GET_SIZE(seqs) != n) return false;
    for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject* s = row(seqs, i, offsets);
        if (!s) return false;
        PyObject** items = reinterpret_cast<PyListObject*>(s)->ob_item;
        const Py_ssize_t len = PyList_GET_SIZE(s);
        for (Py_ssize_t k = 0; k < len; ++k) {
            __builtin_prefetch(items[k + AHEAD < len ? k + AHEAD : k]);
            if (!read(items[k], [&](auto v) { each(i, offsets[i] + k, v); })) return false;
        }
    }
    return true;
}
const auto read_int = [](PyObject* o, auto&& give) {
    int64_t v;
    if (!as_int(o, &v)) return false;
    give(v);
    return true;
};
}  // namespace

extern "C" {
// offsets[0 .. n] of the n sequences laid back to back
int oi_py_offsets(PyObject* seqs, int64_t n, int64_t* offsets) {
    if (!PyList_CheckExact(seqs) || PyList_GET_SIZE(seqs) != n) return -1;
    offsets[0] = 0;
    for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject* s = PyList_GET_ITEM(seqs, i);
        if (!PyList_CheckExact(s)) return -1;
        offsets[i + 1] = offsets[i] + PyList_GET_SIZE(s);
    }
    return 0;
}
// integers; others[i] = how many of sequence i differ from `skip`
int oi_py_flatten_ints(PyObject* seqs, int64_t n, const int64_t* offsets, int64_t skip, int64_t* out, int64_t* others) {
    for (int64_t i = 0; i < n; ++i) others[i] = 0;
    return walk(seqs, offsets, n, read_int, [&](int64_t i, int64_t at, int64_t v) {
        out[at] = v;
        others[i] += v != skip;
    }) ? 0 : -1;
}
// integers as flags: 1 where not 0
int oi_py_flatten_flags(PyObject* seqs, int64_t n, const int64_t* offsets, uint8_t* out) {
    return walk(seqs, offsets, n, read_int, [&](int64_t, int64_t at, int64_t v) { out[at] = v != 0; }) ? 0 : -1;
}
// floats, rounded to fp32
int oi_py_flatten_floats(PyObject* seqs, int64_t n, const int64_t* offsets, float* out) {
    const auto read = [](PyObject* o, auto&& give) {
        if (!PyFloat_CheckExact(o)) return false;
        give(PyFloat_AS_DOUBLE(o));
        return true;
    };
    return walk(seqs, offsets, n, read, [&](int64_t, int64_t at, double v) { out[at] = (float)v; }) ? 0 : -1;
}
}
