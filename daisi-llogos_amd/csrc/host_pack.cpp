// What the sampler packs on the host for every step, from Python's own lists: each row's window of recent tokens, one behind the other, and its
// uniform number.  4,000 small integers take Python 0.1 ms to gather and convert, most of a step of the sampler; read where they lie they
// take 10 us.  Called with the interpreter's lock held (ctypes.PyDLL).  Whatever is no list or tuple of plain integers in range is left to
// Python: -1, and no error set.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>

namespace {

struct Items {
    PyObject** at = nullptr;
    Py_ssize_t n = -1;                  // -1: neither a list nor a tuple
};

Items items_of(PyObject* o) {
    Items s;
    if (PyList_CheckExact(o) || PyTuple_CheckExact(o)) {
        s.at = PySequence_Fast_ITEMS(o);
        s.n = PySequence_Fast_GET_SIZE(o);
    }
    return s;
}

uint64_t splitmix64(uint64_t x) {
    uint64_t z = x + 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// an integer modulo 2^64; false for anything else
bool masked(PyObject* o, uint64_t& v) {
    if (!PyLong_CheckExact(o)) return false;
    v = PyLong_AsUnsignedLongLongMask(o);
    return !(v == (uint64_t)-1 && PyErr_Occurred());
}

}  // namespace

extern "C" {

// Tokens in the windows of all histories together: the last `count` of each, or all of it where count is 0 or not below its length.
__attribute__((visibility("default"))) long long llogos_host_windows_size(PyObject* histories, long long count) {
    const Items rows = items_of(histories);
    long long total = rows.n < 0 ? -1 : 0;
    for (Py_ssize_t r = 0; r < rows.n; ++r) {
        const Items h = items_of(rows.at[r]);
        if (h.n < 0) return -1;
        total += count > 0 && count < h.n ? count : h.n;
    }
    return total;
}

// Writes them to flat (room for `room` tokens) and each row's place to starts [rows + 1]: their number, or -1.
__attribute__((visibility("default"))) long long llogos_host_windows(PyObject* histories, long long count, long long n_rows, int32_t* starts, int32_t* flat, long long room) {
    const Items rows = items_of(histories);
    if (rows.n != n_rows) return -1;
    long long n = 0;
    starts[0] = 0;
    for (Py_ssize_t r = 0; r < rows.n; ++r) {
        const Items h = items_of(rows.at[r]);
        if (h.n < 0) return -1;
        const Py_ssize_t first = count > 0 && count < h.n ? h.n - (Py_ssize_t)count : 0;
        if (n + (h.n - first) > room) return -1;
        for (Py_ssize_t i = first; i < h.n; ++i) {
            if (!PyLong_CheckExact(h.at[i])) return -1;
            int overflow = 0;
            const long v = PyLong_AsLongAndOverflow(h.at[i], &overflow);
            if (overflow != 0 || v < INT32_MIN || v > INT32_MAX) return -1;
            flat[n++] = (int32_t)v;
        }
        starts[r + 1] = (int32_t)n;
    }
    return n;
}

// sampling/rng.py: uniform(seed, requests[r], indices[r]) for n rows; 0, or -1.
__attribute__((visibility("default"))) int llogos_host_uniforms(PyObject* seed, PyObject* requests, PyObject* indices, long long n, float* out) {
    const Items r = items_of(requests), i = items_of(indices);
    uint64_t s;
    if (r.n != n || i.n != n || !masked(seed, s)) { PyErr_Clear(); return -1; }
    const uint64_t h0 = splitmix64(s);
    for (Py_ssize_t k = 0; k < n; ++k) {
        uint64_t a, b;
        if (!masked(r.at[k], a) || !masked(i.at[k], b)) { PyErr_Clear(); return -1; }
        uint64_t h = splitmix64(h0 ^ (a + 1) * 0xD6E8FEB86659FD93ull);
        h = splitmix64(h ^ (b + 1) * 0xA0761D6478BD642Full);
        out[k] = (float)(h >> 40) / 16777216.0f;
    }
    return 0;
}

}  // extern "C"
