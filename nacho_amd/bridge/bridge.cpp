// The call path between the Python classes and the C ABI (include/nacho_hip.h), in C++: fills
// the operands' descriptors from their torch buffers, calls the entry point without the
// interpreter lock, and hands the result buffers to torch in place (no copy, released with
// nacho_free on the stream that produced them when the last tensor over them dies), as the
// reference's generated nanobind wrapper does (src/backend/generate_bindings.cpp:288-327,
// runtime/nacho_nb.h:37-58).
//
// The same steps through ctypes and __cuda_array_interface__ cost about 11 us more per call, as
// much as the kernels of a small merge: csr_add of 200 rows 25.2 -> 14.5 us.
//
// An operand that does not pass the checks here (lengths, devices) makes invoke() return None:
// the caller (ops.py) then raises the exception that names what is wrong.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <exception>
#include <string>

#include "../../include/nacho_hip.h"

namespace {

enum Kind { kCsr = 0, kCoo, kCoo3, kDcsr, kCsf3, kCsr64, kScalar };
constexpr int kMaxBuffers = 6;

// Number of buffers and dimensions of a kind.
constexpr int kBuffers[] = {3, 3, 4, 4, 6, 3, 1};
constexpr int kDims[] = {2, 2, 3, 2, 3, 2, 0};

// Buffers that hold offsets: one entry more than the level above.
constexpr bool kIsOffsets[][kMaxBuffers] = {{true},        {false}, {false}, {false, true},
                                            {false, true, false, true}, {true}, {false}};

union Desc {
    nacho_csr csr;
    nacho_coo coo;
    nacho_coo3 coo3;
    nacho_dcsr dcsr;
    nacho_csf3 csf3;
    nacho_csr64 csr64;
    nacho_scalar scalar;
};

using FreeFn = int (*)(void *, void *);
FreeFn g_free = nullptr;

struct Buffer {
    void *ptr;
    int64_t n;
};

// The operand's buffers and dimensions; false when a buffer is not on `device`.
bool read_operand(int kind, PyObject *buffers, PyObject *dims, int device, Buffer *out,
                  int32_t *size) {
    if (!PyTuple_CheckExact(buffers) || PyTuple_GET_SIZE(buffers) != kBuffers[kind]) return false;
    if (!PyTuple_CheckExact(dims) || PyTuple_GET_SIZE(dims) != kDims[kind]) return false;
    for (int i = 0; i < kBuffers[kind]; ++i) {
        PyObject *o = PyTuple_GET_ITEM(buffers, i);
        if (!THPVariable_Check(o)) return false;
        const at::Tensor &t = THPVariable_Unpack(o);
        if (!t.is_cuda() || t.get_device() != device) return false;
        out[i].n = t.numel();
        out[i].ptr = out[i].n > 0 ? t.data_ptr() : nullptr;
    }
    for (int i = 0; i < kDims[kind]; ++i) {
        size[i] = static_cast<int32_t>(PyLong_AsLong(PyTuple_GET_ITEM(dims, i)));
    }
    return !PyErr_Occurred();
}

template <typename T>
T *as(const Buffer &b) {
    return static_cast<T *>(b.ptr);
}

// The operand's descriptor; false when its lengths do not fit each other or 32 bits.
bool fill(int kind, const Buffer *b, const int32_t *s, Desc *d) {
    for (int i = 0; i < kBuffers[kind]; ++i) {
        if (b[i].n > INT32_MAX + int64_t{kIsOffsets[kind][i]}) {
            return false;
        }
    }
    const int32_t n0 = static_cast<int32_t>(b[0].n), n1 = static_cast<int32_t>(b[1].n);
    switch (kind) {
        case kCsr:
            if (b[0].n != static_cast<int64_t>(s[0]) + 1 || b[2].n != n1) return false;
            d->csr = nacho_csr{s[0], s[1], as<int32_t>(b[0]), n1, as<int32_t>(b[1]),
                               as<float>(b[2]), n1};
            return true;
        case kCoo:
            if (b[1].n != n0 || b[2].n != n0) return false;
            d->coo = nacho_coo{s[0], s[1], n0, as<int32_t>(b[0]), n0, as<int32_t>(b[1]),
                               as<float>(b[2]), n0};
            return true;
        case kCoo3:
            if (b[1].n != n0 || b[2].n != n0 || b[3].n != n0) return false;
            d->coo3 = nacho_coo3{s[0], s[1], s[2], n0, as<int32_t>(b[0]), n0, as<int32_t>(b[1]),
                                 n0, as<int32_t>(b[2]), as<float>(b[3]), n0};
            return true;
        case kDcsr: {
            const int32_t n2 = static_cast<int32_t>(b[2].n);
            if (b[1].n != b[0].n + 1 || b[3].n != n2) return false;
            d->dcsr = nacho_dcsr{s[0], s[1], n0, as<int32_t>(b[0]), as<int32_t>(b[1]), n2,
                                 as<int32_t>(b[2]), as<float>(b[3]), n2};
            return true;
        }
        case kCsf3: {
            const int32_t n2 = static_cast<int32_t>(b[2].n), n4 = static_cast<int32_t>(b[4].n);
            if (b[1].n != b[0].n + 1 || b[3].n != b[2].n + 1 || b[5].n != n4) return false;
            d->csf3 = nacho_csf3{s[0], s[1], s[2], n0, as<int32_t>(b[0]), as<int32_t>(b[1]), n2,
                                 as<int32_t>(b[2]), as<int32_t>(b[3]), n4, as<int32_t>(b[4]),
                                 as<float>(b[5]), n4};
            return true;
        }
        default: return false;
    }
}

PyObject *wrap(void *ptr, int64_t n, at::ScalarType type, int device, void *stream) {
    const auto options = at::TensorOptions().dtype(type).device(at::kCUDA, device);
    if (!ptr) return THPVariable_Wrap(at::empty({0}, options));
    return THPVariable_Wrap(at::from_blob(
        ptr, {n}, [stream](void *p) { (void)g_free(p, stream); }, options,
        at::Device(at::kCUDA, static_cast<c10::DeviceIndex>(device))));
}

// The result's tensors and dimensions: ((tensor, ...), (size, ...)).
PyObject *adopt(int kind, const Desc &z, int device, void *stream) {
    const auto I = at::kInt, L = at::kLong, F = at::kFloat;
    struct {
        void *p;
        int64_t n;
        at::ScalarType t;
    } b[kMaxBuffers] = {};
    int64_t s[3] = {0, 0, 0};
    auto put = [&](int i, void *p, int64_t n, at::ScalarType t) { b[i] = {p, n, t}; };
    switch (kind) {
        case kCsr:
            put(0, z.csr.dim_j_offsets, z.csr.dim_i_size + int64_t{1}, I);
            put(1, z.csr.dim_j_indices, z.csr.dim_j_length, I);
            put(2, z.csr.values, z.csr.dim_j_length, F);
            s[0] = z.csr.dim_i_size, s[1] = z.csr.dim_j_size;
            break;
        case kCsr64:
            put(0, z.csr64.dim_j_offsets, z.csr64.dim_i_size + int64_t{1}, L);
            put(1, z.csr64.dim_j_indices, z.csr64.dim_j_length, I);
            put(2, z.csr64.values, z.csr64.dim_j_length, F);
            s[0] = z.csr64.dim_i_size, s[1] = z.csr64.dim_j_size;
            break;
        case kCoo:
            put(0, z.coo.dim_i_indices, z.coo.nnz, I);
            put(1, z.coo.dim_j_indices, z.coo.nnz, I);
            put(2, z.coo.values, z.coo.nnz, F);
            s[0] = z.coo.dim_i_size, s[1] = z.coo.dim_j_size;
            break;
        case kCoo3:
            put(0, z.coo3.dim_i_indices, z.coo3.nnz, I);
            put(1, z.coo3.dim_j_indices, z.coo3.nnz, I);
            put(2, z.coo3.dim_k_indices, z.coo3.nnz, I);
            put(3, z.coo3.values, z.coo3.nnz, F);
            s[0] = z.coo3.dim_i_size, s[1] = z.coo3.dim_j_size, s[2] = z.coo3.dim_k_size;
            break;
        case kDcsr:
            put(0, z.dcsr.dim_i_indices, z.dcsr.dim_i_length, I);
            put(1, z.dcsr.dim_j_offsets, z.dcsr.dim_i_length + int64_t{1}, I);
            put(2, z.dcsr.dim_j_indices, z.dcsr.dim_j_length, I);
            put(3, z.dcsr.values, z.dcsr.dim_j_length, F);
            s[0] = z.dcsr.dim_i_size, s[1] = z.dcsr.dim_j_size;
            break;
        case kCsf3:
            put(0, z.csf3.dim_i_indices, z.csf3.dim_i_length, I);
            put(1, z.csf3.dim_j_offsets, z.csf3.dim_i_length + int64_t{1}, I);
            put(2, z.csf3.dim_j_indices, z.csf3.dim_j_length, I);
            put(3, z.csf3.dim_k_offsets, z.csf3.dim_j_length + int64_t{1}, I);
            put(4, z.csf3.dim_k_indices, z.csf3.dim_k_length, I);
            put(5, z.csf3.values, z.csf3.dim_k_length, F);
            s[0] = z.csf3.dim_i_size, s[1] = z.csf3.dim_j_size, s[2] = z.csf3.dim_k_size;
            break;
        default: put(0, z.scalar.values, 1, F); break;
    }
    PyObject *tensors = PyTuple_New(kBuffers[kind]);
    PyObject *dims = tensors ? PyTuple_New(kDims[kind]) : nullptr;
    int done = 0;
    if (dims) {
        for (; done < kBuffers[kind]; ++done) {
            PyObject *t = wrap(b[done].p, b[done].n, b[done].t, device, stream);
            if (!t) break;
            PyTuple_SET_ITEM(tensors, done, t);
        }
        for (int i = 0; i < kDims[kind] && done == kBuffers[kind]; ++i) {
            PyObject *v = PyLong_FromLongLong(s[i]);
            if (!v) break;
            PyTuple_SET_ITEM(dims, i, v);
        }
    }
    if (done != kBuffers[kind] || PyErr_Occurred()) {  // out of memory
        for (int i = done; i < kBuffers[kind]; ++i) {
            if (b[i].p) (void)g_free(b[i].p, stream);
        }
        Py_XDECREF(tensors);
        Py_XDECREF(dims);
        return nullptr;
    }
    return Py_BuildValue("NN", tensors, dims);
}

// invoke(entry, result_kind, num_blocks, threads_per_block, stream, device,
//        kind, buffers, dims, kind, buffers, dims[, kind, buffers, dims])
//   -> ((tensor, ...), (size, ...)), an int error code, or None
PyObject *invoke(PyObject *, PyObject *const *args, Py_ssize_t n) {
    const int operands = static_cast<int>((n - 6) / 3);
    if (n != 6 + 3 * operands || operands < 2 || operands > 3) {
        PyErr_SetString(PyExc_TypeError, "invoke: two or three operands");
        return nullptr;
    }
    void *entry = PyLong_AsVoidPtr(args[0]);
    const long kind = PyLong_AsLong(args[1]);
    const int32_t nb = static_cast<int32_t>(PyLong_AsUnsignedLongLongMask(args[2]));
    const int32_t tpb = static_cast<int32_t>(PyLong_AsUnsignedLongLongMask(args[3]));
    void *stream = PyLong_AsVoidPtr(args[4]);
    const int device = static_cast<int>(PyLong_AsLong(args[5]));
    if (PyErr_Occurred()) return nullptr;
    if (!entry || !g_free || kind < kCsr || kind > kScalar) {
        PyErr_SetString(PyExc_ValueError, "invoke: no such entry point or result");
        return nullptr;
    }
    try {
        Desc d[3], z;
        for (int i = 0; i < operands; ++i) {
            const long k = PyLong_AsLong(args[6 + 3 * i]);
            Buffer b[kMaxBuffers];
            int32_t s[3];
            if (k < kCsr || k > kCsf3 ||
                !read_operand(static_cast<int>(k), args[7 + 3 * i], args[8 + 3 * i], device, b, s) ||
                !fill(static_cast<int>(k), b, s, &d[i])) {
                PyErr_Clear();
                Py_RETURN_NONE;
            }
        }
        int rc = 0;
        std::string failure;  // an exception must not pass the point where the lock is taken again
        Py_BEGIN_ALLOW_THREADS
        try {
            if (operands == 2) {
                using Fn = int (*)(const void *, const void *, void *, int32_t, int32_t, void *,
                                   const nacho_allocator *);
                rc = reinterpret_cast<Fn>(entry)(&d[0], &d[1], &z, nb, tpb, stream, nullptr);
            } else {
                using Fn = int (*)(const void *, const void *, const void *, void *, int32_t,
                                   int32_t, void *, const nacho_allocator *);
                rc = reinterpret_cast<Fn>(entry)(&d[0], &d[1], &d[2], &z, nb, tpb, stream,
                                                 nullptr);
            }
        } catch (const std::exception &e) {
            failure = std::string("the entry point threw: ") + e.what();
        }
        Py_END_ALLOW_THREADS
        if (!failure.empty()) {
            PyErr_SetString(PyExc_RuntimeError, failure.c_str());
            return nullptr;
        }
        if (rc != 0) return PyLong_FromLong(rc);
        return adopt(static_cast<int>(kind), z, device, stream);
    } catch (const std::exception &e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

// set_free(address of nacho_free)
PyObject *set_free(PyObject *, PyObject *arg) {
    void *p = PyLong_AsVoidPtr(arg);
    if (PyErr_Occurred()) return nullptr;
    g_free = reinterpret_cast<FreeFn>(p);
    Py_RETURN_NONE;
}

PyMethodDef g_methods[] = {
    {"invoke", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(invoke)), METH_FASTCALL,
     "Call a C entry point on torch buffers and adopt its result."},
    {"set_free", set_free, METH_O, "Address of nacho_free."},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_bridge", nullptr, -1, g_methods,
                        nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__bridge() { return PyModule_Create(&g_module); }
