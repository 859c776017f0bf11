// mindrl_amd/_native.so - the host side of the buffer classes' calls: checks the arguments, allocates the results and
// calls the C ABI (include/mrb.h, include/mrb_more.h), in one step from Python.
//
// A call on a small buffer is 4 to 8 us of kernels, and through ctypes its host side took two to four times as long: a
// torch.empty for each result (1.1 us each, seven to nine of them), the checks of the arguments and the pointer arrays in
// Python. Here results come straight from torch's caching allocator, and a call's host time is theirs, the library's and the
// runtime's launch.
//
// A rollout's returns with gradients went through a Python autograd function, whose backward half the engine's thread
// runs under the interpreter's lock; ReturnBackward needs neither (forward and backward of [1000, 4096] 84 -> 52 us).
//
// Every method returns None, having done nothing, when an argument is not what the fast path takes (another dtype or
// device, not contiguous, rows that do not match): the Python classes then convert it and call again, or raise.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/hip/impl/HIPCachingAllocatorMasqueradingAsCUDA.h>
#include <c10/core/Allocator.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>

#include <cstring>
#include <mutex>
#include <new>

#include "../../include/mrb.h"
#include "../../include/mrb_more.h"

namespace {

constexpr int kMaxDims = 62;  // of a field: results of two more are what torch's own operations take at most

struct Field {
    at::ScalarType type;
    int64_t item, numel, bytes;  // per element, elements and bytes per row
    int ndim;
    int64_t shape[kMaxDims];
};

struct Rows {  // one buffer: its handle and its fields
    PyObject_HEAD
    int64_t handle;
    int nfields;
    int device;
    PyObject* check;  // _lib.check: status code -> exception
    Field f[MRB_MAX_FIELDS];
};

// ---- results -----------------------------------------------------------------------------------------------------

struct Output {
    at::ScalarType type;
    int64_t bytes;
    int ndim;
    int64_t shape[kMaxDims + 2];
    at::Tensor t;
    void* ptr;
};

c10::Storage new_storage(int64_t bytes) {
    // torch's allocator for what it calls CUDA tensors on this platform
    c10::Allocator* allocator = c10::hip::HIPCachingAllocatorMasqueradingAsCUDA::get();
    return c10::Storage(c10::make_intrusive<c10::StorageImpl>(c10::StorageImpl::use_byte_size_t(), bytes, allocator->allocate(bytes),
                                                              allocator, /*resizable=*/true));
}

void make(Output& o, c10::Storage storage) {
    o.ptr = storage.mutable_data();
    o.t = at::detail::make_tensor<c10::TensorImpl>(std::move(storage), c10::DispatchKeySet(c10::DispatchKey::CUDA),
                                                   c10::scalarTypeToTypeMeta(o.type));
    o.t.unsafeGetTensorImpl()->set_sizes_contiguous(c10::IntArrayRef(o.shape, o.ndim));
}

// A storage each: a result can be grown, saved, kept or marked as used on another stream without the call's others.
void allocate(Output* o, int n, int device) {
    c10::OptionalDeviceGuard guard;
    if (c10::hip::current_device() != device) guard.reset_device(c10::Device(c10::DeviceType::CUDA, (c10::DeviceIndex)device));
    for (int i = 0; i < n; ++i) make(o[i], new_storage(o[i].bytes));
}

// [lead..., *shape_i]; nlead 0..2
void describe(Output& o, const Field& f, const int64_t* lead, int nlead) {
    o.type = f.type;
    o.bytes = f.bytes;
    o.ndim = nlead + f.ndim;
    for (int i = 0; i < nlead; ++i) {
        o.shape[i] = lead[i];
        o.bytes *= lead[i];
    }
    for (int i = 0; i < f.ndim; ++i) o.shape[nlead + i] = f.shape[i];
}

void describe(Output& o, at::ScalarType type, int64_t item, const int64_t* lead, int nlead) {
    o.type = type;
    o.bytes = item;
    o.ndim = nlead;
    for (int i = 0; i < nlead; ++i) {
        o.shape[i] = lead[i];
        o.bytes *= lead[i];
    }
}

PyObject* as_tuple(Output* o, int n) {
    PyObject* out = PyTuple_New(n);
    if (!out) return nullptr;
    for (int i = 0; i < n; ++i) {
        PyObject* t = THPVariable_Wrap(std::move(o[i].t));
        if (!t) {
            Py_DECREF(out);
            return nullptr;
        }
        PyTuple_SET_ITEM(out, i, t);
    }
    return out;
}

// ---- arguments ---------------------------------------------------------------------------------------------------

void* stream_of_current_device() { return c10::hip::getCurrentHIPStream().stream(); }

// A contiguous tensor of `type` on the buffer's device: its address and number of elements.
bool on_device(const Rows* r, PyObject* x, at::ScalarType type, void** ptr, int64_t* numel) {
    if (!THPVariable_Check(x)) return false;
    const at::Tensor& t = THPVariable_Unpack(x);
    if (!t.is_cuda() || t.get_device() != r->device || t.scalar_type() != type || !t.is_contiguous() || t.layout() != c10::kStrided)
        return false;
    *ptr = t.data_ptr();
    *numel = t.numel();
    return true;
}

// None, or such a tensor of `want` elements.
bool optional_on_device(const Rows* r, PyObject* x, at::ScalarType type, int64_t want, void** ptr) {
    *ptr = nullptr;
    if (x == Py_None) return true;
    int64_t n;
    return on_device(r, x, type, ptr, &n) && n == want;
}

// The element type of a buffer's format string ('f', '<f', '=f', '@f'), or Undefined.
at::ScalarType type_of_format(const char* s, int64_t item) {
    if (!s) return at::ScalarType::Byte;
    if (*s == '<' || *s == '=' || *s == '@') ++s;
    if (!s[0] || s[1]) return at::ScalarType::Undefined;
    switch (s[0]) {
        case 'e': return at::ScalarType::Half;
        case 'f': return at::ScalarType::Float;
        case 'd': return at::ScalarType::Double;
        case '?': return at::ScalarType::Bool;
        case 'B': return at::ScalarType::Byte;
        case 'b': return at::ScalarType::Char;
        case 'h': return at::ScalarType::Short;
        case 'i': case 'l': case 'q':
            return item == 8 ? at::ScalarType::Long : item == 4 ? at::ScalarType::Int : at::ScalarType::Undefined;
        default: return at::ScalarType::Undefined;
    }
}

PyTypeObject* ndarray_type = nullptr;  // numpy.ndarray

// The rows a call brings: device tensors where they lie; host tensors and arrays copied into the buffer's pinned
// staging memory (mrb_stage), which the kernels read.
struct Source {
    const void* ptr[MRB_MAX_FIELDS] = {};
    int64_t nrows = -1;
    const void* host[MRB_MAX_FIELDS] = {};  // rows in host memory
    at::Tensor held[MRB_MAX_FIELDS];        // the host tensors among them: they are read without the interpreter's lock
    int64_t staged = 0;                     // bytes of staging memory they take
    Py_buffer view[MRB_MAX_FIELDS];
    bool viewed[MRB_MAX_FIELDS] = {};
    int nviews = 0;
    ~Source() {
        for (int i = 0; i < nviews; ++i)
            if (viewed[i]) PyBuffer_Release(&view[i]);
    }
    // false: not what the fast path takes (no Python error is left behind)
    bool take(const Rows* r, PyObject* fields) {
        PyObject** items;
        if (PyTuple_Check(fields) && PyTuple_GET_SIZE(fields) == r->nfields) items = &PyTuple_GET_ITEM(fields, 0);
        else if (PyList_Check(fields) && PyList_GET_SIZE(fields) == r->nfields) items = &PyList_GET_ITEM(fields, 0);
        else return false;
        for (int i = 0; i < r->nfields; ++i) {
            const Field& f = r->f[i];
            int64_t n;
            nviews = i + 1;
            if (THPVariable_Check(items[i])) {
                const at::Tensor& t = THPVariable_Unpack(items[i]);
                if (t.scalar_type() != f.type || !t.is_contiguous() || t.layout() != c10::kStrided) return false;
                ptr[i] = t.data_ptr();
                n = t.numel();
                if (t.is_cpu()) {
                    if (t.is_neg()) return false;  // (a view that negates: a plain copy of its memory is not its values)
                    host[i] = ptr[i];
                    held[i] = t;
                } else if (!t.is_cuda() || t.get_device() != r->device) {
                    return false;
                }
            } else {
                if (!PyObject_TypeCheck(items[i], ndarray_type)) return false;
                if (PyObject_GetBuffer(items[i], &view[i], PyBUF_C_CONTIGUOUS | PyBUF_FORMAT) != 0) {
                    PyErr_Clear();
                    return false;
                }
                viewed[i] = true;
                if (view[i].itemsize != f.item || type_of_format(view[i].format, view[i].itemsize) != f.type) return false;
                n = view[i].len / view[i].itemsize;
                host[i] = view[i].buf;
            }
            if (n % f.numel || (nrows >= 0 && n / f.numel != nrows)) return false;
            nrows = n / f.numel;
            if (host[i]) staged += (nrows * f.bytes + 15) / 16 * 16;
        }
        return true;
    }
    // Copies host rows into the staging memory; false where they do not fit it. Page-locked rows may be what work queued
    // on the stream fills (a non-blocking copy from the device): they are read when that work is done. Called WITHOUT the
    // interpreter's lock: both may wait for the device, and what the device is waiting for may be another Python thread.
    bool stage(const Rows* r, void* stream) {
        if (staged == 0 || nrows <= 0) return true;
        void* to = nullptr;
        if (mrb_stage(r->handle, staged, &to, stream) != MRB_OK || mrb_host_settled(host, r->nfields, stream) != MRB_OK) return false;
        char* at = static_cast<char*>(to);
        for (int i = 0; i < r->nfields; ++i) {
            if (!host[i]) continue;
            const int64_t bytes = nrows * r->f[i].bytes;
            memcpy(at, host[i], (size_t)bytes);
            ptr[i] = at;
            at += (bytes + 15) / 16 * 16;
        }
        return true;
    }
};

bool integer(PyObject* x, int64_t* v) {
    *v = PyLong_AsLongLong(x);
    return !(*v == -1 && PyErr_Occurred());
}
bool real(PyObject* x, float* v) {
    const double d = PyFloat_AsDouble(x);
    *v = (float)d;
    return !(d == -1.0 && PyErr_Occurred());
}

// Raises what _lib.check raises for a status.
PyObject* failed(Rows* r, int rc) {
    PyObject* res = PyObject_CallFunction(r->check, "i", rc);
    if (res) {
        Py_DECREF(res);
        PyErr_Format(PyExc_RuntimeError, "libmrb status %d", rc);
    }
    return nullptr;
}

// (the library's calls run without the interpreter's lock, as they do through ctypes)
#define CALL(expr)                                \
    int rc;                                       \
    Py_BEGIN_ALLOW_THREADS rc = (expr);           \
    Py_END_ALLOW_THREADS if (rc != MRB_OK) return failed(r, rc)
// the same for a call that brings rows (`src`); None where they do not fit the staging memory
#define CALL_WITH_ROWS(expr)                              \
    int rc = MRB_OK;                                      \
    bool ready;                                           \
    Py_BEGIN_ALLOW_THREADS ready = src.stage(r, stream);  \
    if (ready) rc = (expr);                               \
    Py_END_ALLOW_THREADS if (!ready) Py_RETURN_NONE;      \
    if (rc != MRB_OK) return failed(r, rc)

#define ARGS(count)                                                                                    \
    Rows* const r = reinterpret_cast<Rows*>(self);                                                     \
    if (nargs != (count)) {                                                                            \
        PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", (int)(count), nargs);          \
        return nullptr;                                                                                \
    }

// A sample of no rows (the library has its own words for it).
PyObject* refused(Rows* r, int64_t rows) {
    const int rc = mrb_per_sample(r->handle, rows, 0.0f, nullptr, nullptr, nullptr, nullptr, nullptr);
    return failed(r, rc != MRB_OK ? rc : MRB_EINVAL);
}

// ---- prioritized -------------------------------------------------------------------------------------------------

// Result tensors of a sample: indices, weights, fields.
struct Sampled {
    Output o[MRB_MAX_FIELDS + 3];
    void* fields[MRB_MAX_FIELDS];
    int n = 0;
    bool prepare(const Rows* r, const int64_t* lead, int nlead) {  // false: no rows to sample
        for (int i = 0; i < nlead; ++i)
            if (lead[i] <= 0) return false;
        describe(o[0], at::ScalarType::Long, 8, lead, nlead);
        describe(o[1], at::ScalarType::Float, 4, lead, nlead);
        for (int i = 0; i < r->nfields; ++i) describe(o[2 + i], r->f[i], lead, nlead);
        n = 2 + r->nfields;
        return true;
    }
    void finish(const Rows* r) {
        allocate(o, n, r->device);
        for (int i = 0; i < r->nfields; ++i) fields[i] = o[2 + i].ptr;
    }
    int64_t* indices() { return static_cast<int64_t*>(o[0].ptr); }
    float* weights() { return static_cast<float*>(o[1].ptr); }
};

// per_sample(batch, beta, uniforms or None)
PyObject* per_sample(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    ARGS(3)
    int64_t batch;
    float beta;
    void* u;
    if (!integer(args[0], &batch) || !real(args[1], &beta)) return nullptr;
    if (!optional_on_device(r, args[2], at::ScalarType::Float, batch, &u)) Py_RETURN_NONE;
    Sampled s;
    if (!s.prepare(r, &batch, 1)) return refused(r, batch);
    s.finish(r);
    void* const stream = stream_of_current_device();
    CALL(mrb_per_sample(r->handle, batch, beta, static_cast<float*>(u), s.indices(), s.weights(), s.fields, stream));
    return as_tuple(s.o, s.n);
    END_HANDLE_TH_ERRORS
}

// The tensors a sample of `batch` rows goes to: indices and weights that hold them, and the fields, whose shapes the caller
// has checked.
bool given_outputs(const Rows* r, PyObject* indices, PyObject* weights, PyObject* fields, int64_t batch, void** idx, void** w,
                   void** to) {
    int64_t ni, nw, n;
    if (!on_device(r, indices, at::ScalarType::Long, idx, &ni) || !on_device(r, weights, at::ScalarType::Float, w, &nw) || ni < batch ||
        nw < batch || !PyList_Check(fields) || PyList_GET_SIZE(fields) != r->nfields)
        return false;
    for (int i = 0; i < r->nfields; ++i)
        if (!on_device(r, PyList_GET_ITEM(fields, i), r->f[i].type, &to[i], &n)) return false;
    return true;
}

// per_sample_into(batch, beta, uniforms or None, indices, weights, fields): results written to given tensors
PyObject* per_sample_into(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    ARGS(6)
    int64_t batch;
    float beta;
    void *u, *idx, *w, *fields[MRB_MAX_FIELDS];
    if (!integer(args[0], &batch) || !real(args[1], &beta)) return nullptr;
    if (!optional_on_device(r, args[2], at::ScalarType::Float, batch, &u)) Py_RETURN_NONE;
    if (!given_outputs(r, args[3], args[4], args[5], batch, &idx, &w, fields)) Py_RETURN_NONE;
    void* const stream = stream_of_current_device();
    CALL(mrb_per_sample(r->handle, batch, beta, static_cast<float*>(u), static_cast<int64_t*>(idx), static_cast<float*>(w), fields,
                        stream));
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// per_sample_many(nbatch, batch, beta, uniforms or None)
PyObject* per_sample_many(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    ARGS(4)
    int64_t lead[2];
    float beta;
    void* u;
    if (!integer(args[0], &lead[0]) || !integer(args[1], &lead[1]) || !real(args[2], &beta)) return nullptr;
    if (!optional_on_device(r, args[3], at::ScalarType::Float, lead[0] * lead[1], &u)) Py_RETURN_NONE;
    Sampled s;
    if (!s.prepare(r, lead, 2)) return refused(r, lead[0] <= 0 ? lead[0] : lead[1]);
    s.finish(r);
    void* const stream = stream_of_current_device();
    CALL(mrb_per_sample_many(r->handle, lead[0], lead[1], beta, static_cast<float*>(u), s.indices(), s.weights(), s.fields, stream));
    return as_tuple(s.o, s.n);
    END_HANDLE_TH_ERRORS
}

// per_sample_next(batch, beta, uniforms or None, slot_field, row_field)
PyObject* per_sample_next(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    ARGS(5)
    int64_t batch, slot, row;
    float beta;
    void* u;
    if (!integer(args[0], &batch) || !real(args[1], &beta) || !integer(args[3], &slot) || !integer(args[4], &row)) return nullptr;
    if (row < 0 || row >= r->nfields || !optional_on_device(r, args[2], at::ScalarType::Float, batch, &u)) Py_RETURN_NONE;
    Sampled s;
    if (!s.prepare(r, &batch, 1)) return refused(r, batch);
    describe(s.o[s.n++], r->f[row], &batch, 1);
    s.finish(r);
    void* const stream = stream_of_current_device();
    CALL(mrb_per_sample_next(r->handle, batch, beta, static_cast<float*>(u), (int)slot, (int)row, s.indices(), s.weights(), s.fields,
                             s.o[s.n - 1].ptr, stream));
    return as_tuple(s.o, s.n);
    END_HANDLE_TH_ERRORS
}

// The entries of an update: indices and priorities of equal length.
bool entries(const Rows* r, PyObject* indices, PyObject* priorities, void** idx, void** pr, int64_t* n) {
    int64_t m;
    return on_device(r, indices, at::ScalarType::Long, idx, n) && on_device(r, priorities, at::ScalarType::Float, pr, &m) && m == *n;
}

// per_update(indices, priorities)
PyObject* per_update(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    ARGS(2)
    void *idx, *pr;
    int64_t n;
    if (!entries(r, args[0], args[1], &idx, &pr, &n)) Py_RETURN_NONE;
    void* const stream = stream_of_current_device();
    CALL(mrb_per_update(r->handle, static_cast<int64_t*>(idx), static_cast<float*>(pr), n, stream));
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// per_push(fields, priorities or None)
PyObject* per_push(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    ARGS(2)
    void* const stream = stream_of_current_device();
    void* pr;
    Source src;
    if (args[1] != Py_None && !THPVariable_Check(args[1])) Py_RETURN_NONE;
    if (!src.take(r, args[0]) || !optional_on_device(r, args[1], at::ScalarType::Float, src.nrows, &pr)) Py_RETURN_NONE;
    CALL_WITH_ROWS(mrb_per_push(r->handle, src.ptr, src.nrows, static_cast<float*>(pr), stream));
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// per_update_push(indices, priorities, fields, push priorities or None)
PyObject* per_update_push(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    ARGS(4)
    void* const stream = stream_of_current_device();
    void *idx, *pr, *ppr;
    int64_t n;
    Source src;
    if (!entries(r, args[0], args[1], &idx, &pr, &n) || !src.take(r, args[2]) ||
        !optional_on_device(r, args[3], at::ScalarType::Float, src.nrows, &ppr))
        Py_RETURN_NONE;
    CALL_WITH_ROWS(mrb_per_update_push(r->handle, static_cast<int64_t*>(idx), static_cast<float*>(pr), n, src.ptr, src.nrows,
                                       static_cast<float*>(ppr), stream));
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// per_step(indices, priorities, fields, push priorities or None, batch, beta, uniforms or None, out or None); `out`:
// (indices, weights, [fields]) given tensors
PyObject* per_step(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    ARGS(8)
    void* const stream = stream_of_current_device();
    void *idx, *pr, *ppr, *u;
    int64_t n, batch;
    float beta;
    Source src;
    if (!integer(args[4], &batch) || !real(args[5], &beta)) return nullptr;
    if (!entries(r, args[0], args[1], &idx, &pr, &n) || !optional_on_device(r, args[6], at::ScalarType::Float, batch, &u) ||
        !src.take(r, args[2]) || !optional_on_device(r, args[3], at::ScalarType::Float, src.nrows, &ppr))
        Py_RETURN_NONE;
    Sampled s;
    void *oidx, *w;
    const bool given = args[7] != Py_None;
    if (given) {
        if (!PyTuple_Check(args[7]) || PyTuple_GET_SIZE(args[7]) != 3) Py_RETURN_NONE;
        if (!given_outputs(r, PyTuple_GET_ITEM(args[7], 0), PyTuple_GET_ITEM(args[7], 1), PyTuple_GET_ITEM(args[7], 2), batch, &oidx, &w,
                           s.fields))
            Py_RETURN_NONE;
    } else {
        if (!s.prepare(r, &batch, 1)) return refused(r, batch);
        s.finish(r);
        oidx = s.o[0].ptr;
        w = s.o[1].ptr;
    }
    CALL_WITH_ROWS(mrb_per_update_push_sample(r->handle, static_cast<int64_t*>(idx), static_cast<float*>(pr), n, src.ptr, src.nrows,
                                              static_cast<float*>(ppr), batch, beta, static_cast<float*>(u),
                                              static_cast<int64_t*>(oidx), static_cast<float*>(w), s.fields, stream));
    if (given) Py_RETURN_TRUE;
    return as_tuple(s.o, s.n);
    END_HANDLE_TH_ERRORS
}

// ---- gathers: [n, *shape_i] for given slots, a uniform or a reservoir buffer's draws ----------------------------------

struct Gathered {
    Output o[MRB_MAX_FIELDS + 1];
    void* fields[MRB_MAX_FIELDS];
    void* indices = nullptr;
    int n = 0;
    void prepare(const Rows* r, int64_t rows, bool with_indices) {
        for (int i = 0; i < r->nfields; ++i) describe(o[i], r->f[i], &rows, 1);
        n = r->nfields;
        if (with_indices) describe(o[n++], at::ScalarType::Long, 8, &rows, 1);
        allocate(o, n, r->device);
        for (int i = 0; i < r->nfields; ++i) fields[i] = o[i].ptr;
        if (with_indices) indices = o[n - 1].ptr;
    }
    PyObject* result(const Rows* r) {  // fields, or (indices, fields)
        PyObject* f = as_tuple(o, r->nfields);
        if (!f || !indices) return f;
        PyObject* i = THPVariable_Wrap(std::move(o[n - 1].t));
        if (!i) {
            Py_DECREF(f);
            return nullptr;
        }
        PyObject* both = PyTuple_New(2);
        PyTuple_SET_ITEM(both, 0, i);
        PyTuple_SET_ITEM(both, 1, f);
        return both;
    }
};

template <int (*kGather)(int64_t, const int64_t*, int64_t, void* const*, void*)>
PyObject* gather(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {  // gather(indices)
    HANDLE_TH_ERRORS
    ARGS(1)
    void* idx;
    int64_t n;
    if (!on_device(r, args[0], at::ScalarType::Long, &idx, &n)) Py_RETURN_NONE;
    Gathered g;
    if (n > 0) g.prepare(r, n, false);
    void* const stream = stream_of_current_device();
    CALL(kGather(r->handle, static_cast<int64_t*>(idx), n, g.fields, stream));
    return g.result(r);
    END_HANDLE_TH_ERRORS
}

template <int (*kSample)(int64_t, int64_t, int64_t*, void* const*, void*)>
PyObject* sample(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {  // sample(n, with_indices)
    HANDLE_TH_ERRORS
    ARGS(2)
    int64_t n;
    if (!integer(args[0], &n)) return nullptr;
    Gathered g;
    if (n > 0) g.prepare(r, n, args[1] == Py_True);
    void* const stream = stream_of_current_device();
    CALL(kSample(r->handle, n, static_cast<int64_t*>(g.indices), g.fields, stream));
    return g.result(r);
    END_HANDLE_TH_ERRORS
}

template <int (*kPut)(int64_t, const void* const*, int64_t, void*)>
PyObject* put(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {  // put(fields)
    HANDLE_TH_ERRORS
    ARGS(1)
    void* const stream = stream_of_current_device();
    Source src;
    if (!src.take(r, args[0])) Py_RETURN_NONE;
    CALL_WITH_ROWS(kPut(r->handle, src.ptr, src.nrows, stream));
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// ---- discounted return ---------------------------------------------------------------------------------------------

// A fresh contiguous float32 tensor of the given shape.
at::Tensor new_float(c10::IntArrayRef sizes, int device) {
    c10::OptionalDeviceGuard guard;
    if (c10::hip::current_device() != device) guard.reset_device(c10::Device(c10::DeviceType::CUDA, (c10::DeviceIndex)device));
    at::Tensor t = at::detail::make_tensor<c10::TensorImpl>(new_storage(c10::multiply_integers(sizes) * 4),
                                                            c10::DispatchKeySet(c10::DispatchKey::CUDA), caffe2::TypeMeta::Make<float>());
    t.unsafeGetTensorImpl()->set_sizes_contiguous(sizes);
    return t;
}

// The backward pass of a return that carries gradients: one launch, on the engine's own thread, without the interpreter.
struct ReturnBackward : torch::autograd::Node {
    torch::autograd::SavedVariable done;
    std::vector<int64_t> value_sizes;
    int64_t timesteps = 0, batch = 0, inner = 0;
    float gamma = 0.0f;
    std::string name() const override { return "DiscountedReturnBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        done.reset_data();
    }
    torch::autograd::variable_list apply(torch::autograd::variable_list&& grads) override {
        torch::autograd::variable_list out(2);
        if (!grads[0].defined()) return out;
        std::lock_guard<std::mutex> lock(mutex_);
        const at::Tensor g = grads[0].resolve_neg().contiguous();
        const int device = g.get_device();
        at::Tensor flags = done.unpack();  // (what saved-tensor hooks made of it)
        TORCH_CHECK(flags.get_device() == device && flags.scalar_type() == at::ScalarType::Bool && flags.numel() == timesteps * batch,
                    "the saved flags came back as another tensor");
        flags = flags.contiguous();
        out[0] = new_float(g.sizes(), device);
        if (task_should_compute_output(1)) out[1] = new_float(value_sizes, device);
        const int rc = mrb_discounted_return_grad(g.const_data_ptr<float>(), static_cast<const uint8_t*>(flags.const_data_ptr()),
                                                  out[0].mutable_data_ptr<float>(),
                                                  out[1].defined() ? out[1].mutable_data_ptr<float>() : nullptr, timesteps, batch,
                                                  inner, gamma, stream_of_current_device());
        TORCH_CHECK(rc == MRB_OK, "libmrb: ", mrb_last_error());
        if (!task_should_compute_output(0)) out[0] = at::Tensor();
        return out;
    }
};

// discounted_return(reward, done, last_state_value, gamma, differentiable, _lib.check, device index): contiguous tensors on
// that device, float32 and bool, of matching sizes
PyObject* discounted_return(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    float gamma;
    if (nargs != 7) {
        PyErr_Format(PyExc_TypeError, "expected 7 arguments, got %zd", nargs);
        return nullptr;
    }
    int64_t device;
    if (!real(args[3], &gamma) || !integer(args[6], &device)) return nullptr;
    for (int i = 0; i < 3; ++i)
        if (!THPVariable_Check(args[i])) Py_RETURN_NONE;
    const at::Tensor &reward = THPVariable_Unpack(args[0]), &done = THPVariable_Unpack(args[1]), &value = THPVariable_Unpack(args[2]);
    for (const at::Tensor* t : {&reward, &done, &value})
        if (!t->is_cuda() || t->layout() != c10::kStrided || !t->is_contiguous() || t->get_device() != device ||
            t->scalar_type() != (t == &done ? at::ScalarType::Bool : at::ScalarType::Float))
            Py_RETURN_NONE;
    if (reward.dim() == 0 || done.dim() == 0 || reward.numel() == 0 || done.numel() == 0 || reward.size(0) != done.size(0)) Py_RETURN_NONE;
    const int64_t timesteps = reward.size(0), batch = done.numel() / timesteps, inner = reward.numel() / done.numel();
    if (inner * done.numel() != reward.numel() || value.numel() != batch * inner) Py_RETURN_NONE;
    const bool differentiable =
        args[4] == Py_True && at::GradMode::is_enabled() && (reward.requires_grad() || value.requires_grad());
    if (args[4] == Py_True && (reward.requires_grad() || value.requires_grad()) &&
        (reward._fw_grad(0).defined() || value._fw_grad(0).defined())) {
        PyErr_SetString(PyExc_NotImplementedError, "DiscountedReturn has no forward-mode derivative");
        return nullptr;
    }
    c10::OptionalDeviceGuard guard;
    if (c10::hip::current_device() != device) guard.reset_device(reward.device());
    at::Tensor out = new_float(reward.sizes(), (int)device);
    void* const stream = stream_of_current_device();
    // (data_ptr: raises for tensors without memory)
    const float *x = static_cast<const float*>(reward.data_ptr()), *v = static_cast<const float*>(value.data_ptr());
    const uint8_t* d = static_cast<const uint8_t*>(done.data_ptr());
    float* const o = static_cast<float*>(out.mutable_data_ptr());
    int rc;
    Py_BEGIN_ALLOW_THREADS rc = mrb_discounted_return(x, d, v, o, timesteps, batch, inner, gamma, stream);
    Py_END_ALLOW_THREADS if (rc != MRB_OK) {
        Rows r;
        r.check = args[5];
        return failed(&r, rc);
    }
    if (differentiable) {
        std::shared_ptr<ReturnBackward> node(new ReturnBackward(), torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(reward, value));
        node->done = torch::autograd::SavedVariable(done, false);
        node->value_sizes = value.sizes().vec();
        node->timesteps = timesteps;
        node->batch = batch;
        node->inner = inner;
        node->gamma = gamma;
        torch::autograd::set_history(out, node);
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// ---- the type ----------------------------------------------------------------------------------------------------

// Rows(handle, shapes, dtypes, device index, _lib.check)
int rows_init(PyObject* self, PyObject* args, PyObject*) {
    Rows* const r = reinterpret_cast<Rows*>(self);
    long long handle;
    int device;
    PyObject *shapes, *types, *check;
    if (!PyArg_ParseTuple(args, "LO!O!iO", &handle, &PyTuple_Type, &shapes, &PyTuple_Type, &types, &device, &check)) return -1;
    const Py_ssize_t n = PyTuple_GET_SIZE(shapes);
    if (n < 1 || n > MRB_MAX_FIELDS || PyTuple_GET_SIZE(types) != n) {
        PyErr_SetString(PyExc_ValueError, "between 1 and 16 shapes, and a dtype for each");
        return -1;
    }
    for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject* const shape = PyTuple_GET_ITEM(shapes, i);
        PyObject* const type = PyTuple_GET_ITEM(types, i);
        if (!PyTuple_Check(shape) || PyTuple_GET_SIZE(shape) > kMaxDims || !THPDtype_Check(type)) {
            PyErr_SetString(PyExc_TypeError, "shapes are tuples of at most 62 numbers, dtypes torch dtypes");
            return -1;
        }
        Field& f = r->f[i];
        f.type = reinterpret_cast<THPDtype*>(type)->scalar_type;
        f.item = (int64_t)c10::elementSize(f.type);
        f.ndim = (int)PyTuple_GET_SIZE(shape);
        f.numel = 1;
        for (int k = 0; k < f.ndim; ++k) {
            if (!integer(PyTuple_GET_ITEM(shape, k), &f.shape[k])) return -1;
            f.numel *= f.shape[k];
        }
        f.bytes = f.numel * f.item;
        if (f.numel <= 0) {
            PyErr_SetString(PyExc_ValueError, "a field holds at least one value");
            return -1;
        }
    }
    r->nfields = (int)n;
    r->handle = handle;
    r->device = device;
    Py_INCREF(check);
    Py_XSETREF(r->check, check);
    return 0;
}

void rows_dealloc(PyObject* self) {
    Py_XDECREF(reinterpret_cast<Rows*>(self)->check);
    Py_TYPE(self)->tp_free(self);
}

#define METHOD(name, fn) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(fn)), METH_FASTCALL, nullptr}
PyMethodDef rows_methods[] = {
    METHOD("per_sample", per_sample),
    METHOD("per_sample_into", per_sample_into),
    METHOD("per_sample_many", per_sample_many),
    METHOD("per_sample_next", per_sample_next),
    METHOD("per_update", per_update),
    METHOD("per_push", per_push),
    METHOD("per_update_push", per_update_push),
    METHOD("per_step", per_step),
    METHOD("per_gather", gather<mrb_per_gather>),
    METHOD("urb_append", put<mrb_urb_append>),
    METHOD("urb_gather", gather<mrb_urb_gather>),
    METHOD("urb_sample", sample<mrb_urb_sample>),
    METHOD("res_push", put<mrb_res_push>),
    METHOD("res_sample", sample<mrb_res_sample>),
    {nullptr, nullptr, 0, nullptr},
};

PyTypeObject rows_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyMethodDef module_methods[] = {METHOD("discounted_return", discounted_return), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "mindrl_amd._native", nullptr, -1, module_methods};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) {
    rows_type.tp_name = "mindrl_amd._native.Rows";
    rows_type.tp_basicsize = sizeof(Rows);
    rows_type.tp_flags = Py_TPFLAGS_DEFAULT;
    rows_type.tp_new = PyType_GenericNew;
    rows_type.tp_init = rows_init;
    rows_type.tp_dealloc = rows_dealloc;
    rows_type.tp_methods = rows_methods;
    if (PyType_Ready(&rows_type) < 0) return nullptr;
    PyObject* const numpy = PyImport_ImportModule("numpy");
    if (!numpy) return nullptr;
    ndarray_type = reinterpret_cast<PyTypeObject*>(PyObject_GetAttrString(numpy, "ndarray"));
    Py_DECREF(numpy);
    if (!ndarray_type) return nullptr;
    PyObject* const m = PyModule_Create(&module_def);
    if (!m) return nullptr;
    Py_INCREF(&rows_type);
    if (PyModule_AddObject(m, "Rows", reinterpret_cast<PyObject*>(&rows_type)) < 0) {
        Py_DECREF(&rows_type);
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
