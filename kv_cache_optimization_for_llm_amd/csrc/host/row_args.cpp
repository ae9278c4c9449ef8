// Per-row arguments of a sampling, read from the rows' Python objects into the staging array that goes up to the device.
// Four list comprehensions over 64 rows took 23 us of a call whose kernels take 18; this takes 4.  Called with the
// interpreter's lock held (ctypes.PyDLL).  The comprehensions are what a row's values mean: they run where an exception is set
// here, and where the function is absent because the interpreter's headers were.
#if __has_include(<Python.h>)
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <climits>
#include <cstdint>

namespace {

struct Names {
    PyObject *temperature = PyUnicode_InternFromString("temperature"), *rng_key = PyUnicode_InternFromString("rng_key"),
             *rng_step = PyUnicode_InternFromString("rng_step"), *seat = PyUnicode_InternFromString("seat"),
             *apply_penalty = PyUnicode_InternFromString("apply_penalty");
};

bool real(PyObject *row, PyObject *name, double *out) {
    PyObject *v = PyObject_GetAttr(row, name);
    if (!v) return false;
    *out = PyFloat_AsDouble(v);
    Py_DECREF(v);
    return !(*out == -1.0 && PyErr_Occurred());
}

// int(value), its low 32 bits
bool low_bits(PyObject *row, PyObject *name, uint32_t *out) {
    PyObject *v = PyObject_GetAttr(row, name);
    if (!v) return false;
    PyObject *whole = PyNumber_Long(v);
    Py_DECREF(v);
    if (!whole) return false;
    const unsigned long long bits = PyLong_AsUnsignedLongLongMask(whole);
    Py_DECREF(whole);
    if (bits == (unsigned long long)-1 && PyErr_Occurred()) return false;
    *out = (uint32_t)bits;
    return true;
}

bool whole32(PyObject *row, PyObject *name, int32_t *out) {
    PyObject *v = PyObject_GetAttr(row, name);
    if (!v) return false;
    PyObject *index = PyNumber_Index(v);
    Py_DECREF(v);
    if (!index) return false;
    const long value = PyLong_AsLong(index);
    Py_DECREF(index);
    if (value == -1 && PyErr_Occurred()) return false;
    if (value < INT_MIN || value > INT_MAX) {
        PyErr_SetString(PyExc_OverflowError, "a row's seat does not fit 32 bits");
        return false;
    }
    *out = (int32_t)value;
    return true;
}

bool truth(PyObject *row, PyObject *name, bool *out) {
    PyObject *v = PyObject_GetAttr(row, name);
    if (!v) return false;
    const int t = PyObject_IsTrue(v);
    Py_DECREF(v);
    *out = t > 0;
    return t >= 0;
}

} // namespace

enum { READ_SAMPLED = 1, READ_PENALTY = 2, READ_SEATS = 4, READ_AS_USED = 8, READ_KEYS = 16 };

// One pass over the rows: READ_KEYS the keys and steps alone, whatever else is asked for as below.
static int read_rows(PyObject *list, long long n, int32_t *staging, long long stride, int want) {
    static const Names names;
    int flags = 0;
    for (long long i = 0; i < n && flags >= 0; ++i) {
        if (i >= PySequence_Fast_GET_SIZE(list)) {
            PyErr_SetString(PyExc_ValueError, "fewer rows than logits");
            return -1;
        }
        PyObject *row = PySequence_Fast_GET_ITEM(list, i);
        Py_INCREF(row);
        double temperature = 0.0;
        bool penalty = false, ok = true;
        if (want & READ_SAMPLED) ok = real(row, names.temperature, &temperature);
        if (ok && want & READ_PENALTY) ok = truth(row, names.apply_penalty, &penalty);
        if (ok && staging && want & READ_SAMPLED) {
            const float inverse = temperature > 0.0 ? (float)(1.0 / temperature) : 0.f;
            __builtin_memcpy(&staging[i], &inverse, sizeof inverse);
        }
        if (ok && staging && want & READ_KEYS) {
            uint32_t key = 0, step = 0;
            ok = low_bits(row, names.rng_key, &key) && low_bits(row, names.rng_step, &step);
            staging[stride + i] = (int32_t)key;
            staging[2 * stride + i] = (int32_t)step;
        }
        if (ok && staging && want & READ_SEATS) {
            int32_t seat = 0;
            ok = whole32(row, names.seat, &seat);
            if (want & READ_PENALTY) staging[3 * stride + i] = penalty ? seat : -1;
            staging[4 * stride + i] = seat;
        }
        Py_DECREF(row);
        flags = ok ? flags | (temperature > 0.0 ? 1 : 0) | (penalty ? 2 : 0) : -1;
    }
    return flags;
}

// Returns bit 0: a row has a temperature (asked for with READ_SAMPLED), bit 1: a row asks for the penalty (READ_PENALTY); -1: an
// exception is set.  With `staging` ([5][stride], n <= stride) its rows get, with READ_SAMPLED, 1 / temperature (0: greedy) in fp32
// and the low 32 bits of key and step, with READ_SEATS the seat and, with READ_PENALTY too, the seat of rows that ask for the penalty
// (else -1).  Nothing else of a row is looked at.  READ_AS_USED, with `staging`: keys and steps only where a row has a temperature,
// the penalty's seats only where a row asks for it.
extern "C" int kva_sample_rows(PyObject *rows, long long n, int32_t *staging, long long stride, int want) {
    PyObject *list = PySequence_Fast(rows, "the rows of a sampling are a sequence");
    if (!list) return -1;
    int flags;
    if (want & READ_AS_USED && staging) {
        flags = read_rows(list, n, staging, stride, want & (READ_SAMPLED | READ_PENALTY));
        const int rest = (flags & 1 ? READ_KEYS : 0) | (want & READ_SEATS ? READ_SEATS | (flags & 2 ? READ_PENALTY : 0) : 0);
        if (flags >= 0 && rest && read_rows(list, n, staging, stride, rest) < 0) flags = -1;
    } else {
        flags = read_rows(list, n, staging, stride, want | (want & READ_SAMPLED ? READ_KEYS : 0));
    }
    Py_DECREF(list);
    return flags;
}
#endif
