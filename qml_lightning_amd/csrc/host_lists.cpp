// Host side of a batch given as Python lists of per-molecule numpy arrays (BaseKernel.format_data): the arrays are walked
// here, through numpy's C interface, straight into the buffer that is uploaded.  np.concatenate over the same lists costs 130 ns
// an array, the index arithmetic and scatters behind it as much again: 2048 molecules of 3 to 29 atoms 0.72 ms in all, 0.1 ms
// this way (the padding itself is qmll_format_batch, on the device).  Called with the interpreter lock held (ctypes.PyDLL).
// Lists of anything but plain arrays are refused with -1: the caller has a general route for them.
#define NPY_NO_DEPRECATED_API NPY_1_7_API_VERSION
#include <Python.h>
#include <numpy/arrayobject.h>

namespace {

bool plain(PyObject* o, int ndim, npy_intp width) {
    if (!PyArray_CheckExact(o)) return false;
    PyArrayObject* a = reinterpret_cast<PyArrayObject*>(o);
    return PyArray_ISCARRAY_RO(a) && PyArray_NDIM(a) == ndim && (ndim == 1 || PyArray_DIM(a, 1) == width);
}
PyArrayObject* array_at(PyObject* seq, Py_ssize_t i) { return reinterpret_cast<PyArrayObject*>(PySequence_Fast_GET_ITEM(seq, i)); }
bool is_list(PyObject* o) { return PyList_Check(o) || PyTuple_Check(o); }
bool is_real(int t) { return t == NPY_DOUBLE || t == NPY_FLOAT; }

template <typename To, typename From>
void cast(const void* from, npy_intp n, To* to) {
    const From* p = static_cast<const From*>(from);
    for (npy_intp i = 0; i < n; ++i) to[i] = static_cast<To>(p[i]);
}
template <typename To>
bool cast_any(PyArrayObject* a, npy_intp n, To* to) {
    const void* p = PyArray_DATA(a);
    switch (PyArray_TYPE(a)) {
        case NPY_DOUBLE: cast<To, double>(p, n, to); return true;
        case NPY_FLOAT: cast<To, float>(p, n, to); return true;
        case NPY_LONG: cast<To, npy_long>(p, n, to); return true;
        case NPY_LONGLONG: cast<To, npy_longlong>(p, n, to); return true;
        case NPY_INT: cast<To, npy_int>(p, n, to); return true;
        case NPY_SHORT: cast<To, npy_short>(p, n, to); return true;
        case NPY_BYTE: cast<To, npy_byte>(p, n, to); return true;
        case NPY_UBYTE: cast<To, npy_ubyte>(p, n, to); return true;
        default: return false;
    }
}

// whether molecule i is three plain arrays of the same number of atoms, and that number
bool molecule(PyObject* X, PyObject* Q, PyObject* F, Py_ssize_t i, int qtype, npy_intp& atoms) {
    PyObject* x = PySequence_Fast_GET_ITEM(X, i);
    PyObject* q = PySequence_Fast_GET_ITEM(Q, i);
    if (!plain(x, 2, 3) || !plain(q, 1, 0) || !is_real(PyArray_TYPE(array_at(X, i))) || PyArray_TYPE(array_at(Q, i)) != qtype) return false;
    atoms = PyArray_DIM(array_at(X, i), 0);
    if (PyArray_DIM(array_at(Q, i), 0) != atoms) return false;
    if (F != Py_None) {
        PyObject* f = PySequence_Fast_GET_ITEM(F, i);
        if (!plain(f, 2, 3) || !is_real(PyArray_TYPE(array_at(F, i))) || PyArray_DIM(array_at(F, i), 0) != atoms) return false;
    }
    return true;
}

bool lists(PyObject* X, PyObject* Q, PyObject* F, Py_ssize_t n) {
    return is_list(X) && is_list(Q) && (F == Py_None || is_list(F)) && n > 0 && PySequence_Fast_GET_SIZE(X) == n &&
           PySequence_Fast_GET_SIZE(Q) == n && (F == Py_None || PySequence_Fast_GET_SIZE(F) == n) &&
           PyArray_CheckExact(PySequence_Fast_GET_ITEM(Q, 0));
}

}  // namespace

// once, before the others: 0, or -1 with a Python exception set
extern "C" int qmll_lists_init(void) {
    import_array1(-1);
    return 0;
}

// the molecules' atom counts and the number of atoms in all; -1: not lists of n plain arrays each
extern "C" long long qmll_lists_measure(PyObject* X, PyObject* Q, PyObject* F, long long n, int* counts) {
    if (!lists(X, Q, F, n)) return -1;
    const int qtype = PyArray_TYPE(array_at(Q, 0));
    long long total = 0;
    for (Py_ssize_t i = 0; i < n; ++i) {
        npy_intp atoms;
        if (!molecule(X, Q, F, i, qtype, atoms) || atoms > 0x7fffffff) return -1;
        counts[i] = (int)atoms;
        total += atoms;
        if (total > 0x7fffffff) return -1;
    }
    return total;
}

// the atoms of all molecules one behind the other: x [total, 3], q [total], f [total, 3] (F not None), and each molecule's first
// atom; 0, or -1 when the lists are no longer what they measured (another thread may have had them in between)
extern "C" int qmll_lists_pack(PyObject* X, PyObject* Q, PyObject* F, long long n, const int* counts, long long total, float* x, float* q,
                               double* f, int* starts) {
    if (!lists(X, Q, F, n)) return -1;
    const int qtype = PyArray_TYPE(array_at(Q, 0));
    long long at = 0;
    for (Py_ssize_t i = 0; i < n; ++i) {
        npy_intp atoms;
        if (!molecule(X, Q, F, i, qtype, atoms) || atoms != counts[i] || at + atoms > total) return -1;
        starts[i] = (int)at;
        if (!cast_any(array_at(X, i), 3 * atoms, x + 3 * at) || !cast_any(array_at(Q, i), atoms, q + at)) return -1;
        if (F != Py_None && !cast_any(array_at(F, i), 3 * atoms, f + 3 * at)) return -1;
        at += atoms;
    }
    return at == total ? 0 : -1;
}
