// The package's calls of the C ABI, as a CPython extension on torch's C++ tensors: read the tensors' shapes and pointers,
// allocate the result, find the stream and its workspace, launch.  A decode-sized launch is over on the GPU in 4 - 10 us;
// the same steps written in Python around ctypes took the host 11 - 13 us a call (4096 x 4096 at one row: 14.8 us from one
// call to the next where the kernel runs 4.3), so a program that launches kernel by kernel was bound by them, not by the
// GPU.
//
// Every function takes its arguments by position and returns new tensors, or None where an argument is not what the
// operator takes: the Python function of the same name then says what is wrong with it.  Error codes of the library are
// raised through the hook given to init().
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <vector>

#include "../../../include/gptq4.h"

namespace {

// The interpreter lock is given up around the library's calls, as ctypes does.
struct NoGil {
    PyThreadState *state = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(state); }
};

PyObject *g_workspace_hook = nullptr;  // (device index, bytes): makes the workspace of the current stream that large
PyObject *g_error_hook = nullptr;      // (code, name of the entry point): raises

// Workspaces as _lib.workspace() made them.  Looked up and changed with the interpreter lock held.
struct Workspace {
    int device;
    hipStream_t stream;
    void *data;
    size_t bytes;
};
std::vector<Workspace> g_workspaces;

const Workspace *known_workspace(int device, hipStream_t stream, size_t need) {
    for (const Workspace &w : g_workspaces)
        if (w.stream == stream && w.device == device) return w.bytes >= need ? &w : nullptr;
    return nullptr;
}

// false with a Python error set
bool workspace(int device, hipStream_t stream, size_t need, Workspace *out) {
    const Workspace *w = known_workspace(device, stream, need);
    if (w == nullptr) {
        PyObject *r = PyObject_CallFunction(g_workspace_hook, "in", device, (Py_ssize_t)need);
        if (r == nullptr) return false;
        Py_DECREF(r);
        w = known_workspace(device, stream, need);
        if (w == nullptr) {
            PyErr_SetString(PyExc_RuntimeError, "no workspace for the current stream");
            return false;
        }
    }
    *out = *w;
    return true;
}

PyObject *failed(int rc, const char *where) {
    PyObject *r = PyObject_CallFunction(g_error_hook, "is", rc, where);
    Py_XDECREF(r);
    if (r != nullptr) PyErr_Format(PyExc_RuntimeError, "%s failed: %d", where, rc);
    return nullptr;
}

// An argument that must be a tensor (null if it is none), or a tensor or None (`none` says which).
const at::Tensor *tensor(PyObject *o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

struct Args {
    PyObject *const *v;
    bool fine = true;
    const at::Tensor *need(int i) {
        const at::Tensor *t = tensor(v[i]);
        fine = fine && t != nullptr;
        return t;
    }
    const at::Tensor *may(int i) { return v[i] == Py_None ? nullptr : need(i); }
    long integer(int i) {
        const long x = PyLong_AsLong(v[i]);
        if (x == -1 && PyErr_Occurred()) {
            PyErr_Clear();
            fine = false;
        }
        return x;
    }
    double real(int i) {
        const double x = PyFloat_AsDouble(v[i]);
        if (x == -1.0 && PyErr_Occurred()) {
            PyErr_Clear();
            fine = false;
        }
        return x;
    }
};

bool is_rows(const at::Tensor *t) { return t->is_cuda() && t->scalar_type() == at::kHalf && t->dim() > 0 && t->is_contiguous(); }
// a weight tensor or an optional operand beside the activations on `device`
bool beside(const at::Tensor *t, at::Device device) { return t == nullptr || (t->device() == device && t->is_contiguous()); }
void *data(const at::Tensor *t) { return t == nullptr ? nullptr : t->data_ptr(); }
const int32_t *ints(const at::Tensor *t) { return static_cast<const int32_t *>(data(t)); }
const float *floats(const at::Tensor *t) { return static_cast<const float *>(data(t)); }

at::Tensor empty(at::IntArrayRef size, at::Device device, at::ScalarType type = at::kHalf) {
    return at::Tensor(at::detail::empty_cuda(size, type, device, std::nullopt));
}

// `like`'s shape with another last dimension
at::Tensor empty_rows(const at::Tensor &like, int64_t last) {
    c10::SmallVector<int64_t, 6> size(like.sizes().begin(), like.sizes().end());
    size.back() = last;
    return empty(size, like.device());
}

hipStream_t stream_of(at::Device device) { return c10::hip::getCurrentHIPStream(device.index()).stream(); }

// x [..., K] against packed words [K/8, N]: what every projection asks of its arguments
bool projection_fits(const at::Tensor *x, const at::Tensor *words, long groupsize) {
    if (!is_rows(x) || words->dim() != 2) return false;
    const int64_t k = x->size(-1), n = words->size(1);
    return k == words->size(0) * 8 && k > 0 && k % 128 == 0 && n % 256 == 0 && groupsize % 128 == 0 && x->numel() / k < (1LL << 31);
}

// Bytes of workspace a streaming-order call needs: the zeroed head and room for the gathered rows of an act-order call (up to
// four rows mostly gathered in the kernel), and above 16 rows what the mid-M and tiled kernels ask for.
size_t stream_bytes(int op, long m, long k, long n, bool with_perm) {
    if (m > 16) return gptq4_workspace_bytes(op | (with_perm ? GPTQ4_OP_WITH_PERM : 0), (int)m, (int)k, (int)n);
    return GPTQ4_WS_HEAD_BYTES + (with_perm ? (size_t)2 * m * k : 0);
}

size_t plain_bytes(int op, long m, long k, long n, bool with_perm) {
    return gptq4_workspace_bytes(op | (with_perm ? GPTQ4_OP_WITH_PERM : 0), (int)m, (int)k, (int)n);
}

// The residual add and RMSNorm a projection does on its own input: (delta or None, norm weight, eps).
struct Norm {
    const at::Tensor *delta = nullptr, *weight = nullptr;
    float eps = 0.f;
    at::Tensor sum;
    bool fits(const at::Tensor *x) {
        if (weight == nullptr) return true;
        if (!is_rows(weight) || weight->dim() != 1 || weight->size(0) != x->size(-1)) return false;
        return delta == nullptr || (is_rows(delta) && delta->sizes() == x->sizes());
    }
    void *sum_for(const at::Tensor *x) {
        if (delta == nullptr) return nullptr;
        sum = empty(x->sizes(), x->device());
        return sum.data_ptr();
    }
    // the residual stream behind the add
    PyObject *stream(PyObject *x) {
        if (delta != nullptr) return THPVariable_Wrap(sum);
        Py_INCREF(x);
        return x;
    }
};

#define GPTQ4_TAKES(count)                                                                   \
    if (nargs != (count)) {                                                                  \
        PyErr_Format(PyExc_TypeError, "%d arguments are taken, %d given", count, (int)nargs); \
        return nullptr;                                                                      \
    }

// matmul(groupsize, x, qweight, scales, qzeros, bias, perm) -> y
PyObject *matmul(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    GPTQ4_TAKES(7)
    Args a{v};
    const long g = a.integer(0);
    const at::Tensor *x = a.need(1), *w = a.need(2), *s = a.need(3), *z = a.need(4), *bias = a.may(5), *perm = a.may(6);
    if (!a.fine || !projection_fits(x, w, g)) Py_RETURN_NONE;
    const at::Device dev = x->device();
    for (const at::Tensor *t : {w, s, z, bias, perm})
        if (!beside(t, dev)) Py_RETURN_NONE;
    const long k = x->size(-1), n = w->size(1), m = x->numel() / k;
    at::Tensor y = empty_rows(*x, n);
    if (m > 0) {
        const hipStream_t stream = stream_of(dev);
        Workspace ws;
        if (!workspace(dev.index(), stream, plain_bytes(GPTQ4_OP_MATMUL, m, k, n, perm != nullptr), &ws)) return nullptr;
        int rc;
        {
            NoGil unlocked;
            rc = gptq4_matmul(data(x), ints(w), ints(z), data(s), ints(perm), data(bias), y.data_ptr(), (int)m, (int)k, (int)n, (int)g,
                              ws.data, ws.bytes, stream);
        }
        if (rc) return failed(rc, "gptq4_matmul");
    }
    return THPVariable_Wrap(y);
    END_HANDLE_TH_ERRORS
}

// stream_matmul(groupsize, x, sweight, smeta, bias, perm) -> y
PyObject *stream_matmul(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    GPTQ4_TAKES(6)
    Args a{v};
    const long g = a.integer(0);
    const at::Tensor *x = a.need(1), *w = a.need(2), *meta = a.need(3), *bias = a.may(4), *perm = a.may(5);
    if (!a.fine || !projection_fits(x, w, g)) Py_RETURN_NONE;
    const at::Device dev = x->device();
    for (const at::Tensor *t : {w, meta, bias, perm})
        if (!beside(t, dev)) Py_RETURN_NONE;
    const long k = x->size(-1), n = w->size(1), m = x->numel() / k;
    at::Tensor y = empty_rows(*x, n);
    if (m > 0) {
        const hipStream_t stream = stream_of(dev);
        Workspace ws;
        if (!workspace(dev.index(), stream, stream_bytes(GPTQ4_OP_MATMUL, m, k, n, perm != nullptr), &ws)) return nullptr;
        int rc;
        {
            NoGil unlocked;
            rc = gptq4_stream_matmul(data(x), ints(w), ints(meta), ints(perm), data(bias), y.data_ptr(), (int)m, (int)k, (int)n, (int)g,
                                     ws.data, ws.bytes, stream);
        }
        if (rc) return failed(rc, "gptq4_stream_matmul");
    }
    return THPVariable_Wrap(y);
    END_HANDLE_TH_ERRORS
}

// mlp_gateup(groupsize, x, gate qweight, scales, qzeros, up qweight, scales, qzeros, perm, delta, norm weight, eps)
// -> h, or (x + delta, h) with a norm weight
PyObject *mlp_gateup(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    GPTQ4_TAKES(12)
    Args a{v};
    const long g = a.integer(0);
    const at::Tensor *x = a.need(1), *gw = a.need(2), *gs = a.need(3), *gz = a.need(4), *uw = a.need(5), *us = a.need(6), *uz = a.need(7);
    const at::Tensor *perm = a.may(8);
    Norm norm;
    norm.delta = a.may(9), norm.weight = a.may(10), norm.eps = (float)a.real(11);
    if (!a.fine || !projection_fits(x, gw, g) || !norm.fits(x)) Py_RETURN_NONE;
    if (gw->sizes() != uw->sizes() || gs->sizes() != us->sizes() || gz->sizes() != uz->sizes()) Py_RETURN_NONE;
    const at::Device dev = x->device();
    for (const at::Tensor *t : {gw, gs, gz, uw, us, uz, perm, norm.delta, norm.weight})
        if (!beside(t, dev)) Py_RETURN_NONE;
    const long k = x->size(-1), n = gw->size(1), m = x->numel() / k;
    at::Tensor h = empty_rows(*x, n);
    void *const sum = norm.sum_for(x);
    if (m > 0) {
        const hipStream_t stream = stream_of(dev);
        Workspace ws;
        if (!workspace(dev.index(), stream, plain_bytes(GPTQ4_OP_MLP_GATEUP, m, k, n, perm != nullptr && norm.weight == nullptr), &ws))
            return nullptr;
        int rc;
        {
            NoGil unlocked;
            rc = norm.weight != nullptr
                     ? gptq4_norm_mlp_gateup(data(x), data(norm.delta), data(norm.weight), norm.eps, sum, ints(gw), ints(gz), data(gs),
                                             ints(uw), ints(uz), data(us), ints(perm), h.data_ptr(), (int)m, (int)k, (int)n, (int)g,
                                             ws.data, ws.bytes, stream)
                     : gptq4_mlp_gateup(data(x), ints(gw), ints(gz), data(gs), ints(uw), ints(uz), data(us), ints(perm), h.data_ptr(),
                                        (int)m, (int)k, (int)n, (int)g, ws.data, ws.bytes, stream);
        }
        if (rc) return failed(rc, norm.weight != nullptr ? "gptq4_norm_mlp_gateup" : "gptq4_mlp_gateup");
    }
    if (norm.weight == nullptr) return THPVariable_Wrap(h);
    return Py_BuildValue("NN", norm.stream(v[1]), THPVariable_Wrap(h));
    END_HANDLE_TH_ERRORS
}

// stream_mlp_gateup(groupsize, x, gate sweight, smeta, up sweight, smeta, perm, delta, norm weight, eps)
// -> h, or (x + delta, h) with a norm weight
PyObject *stream_mlp_gateup(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    GPTQ4_TAKES(10)
    Args a{v};
    const long g = a.integer(0);
    const at::Tensor *x = a.need(1), *gw = a.need(2), *gm = a.need(3), *uw = a.need(4), *um = a.need(5), *perm = a.may(6);
    Norm norm;
    norm.delta = a.may(7), norm.weight = a.may(8), norm.eps = (float)a.real(9);
    if (!a.fine || !projection_fits(x, gw, g) || !norm.fits(x)) Py_RETURN_NONE;
    if (gw->sizes() != uw->sizes() || gm->sizes() != um->sizes()) Py_RETURN_NONE;
    const at::Device dev = x->device();
    for (const at::Tensor *t : {gw, gm, uw, um, perm, norm.delta, norm.weight})
        if (!beside(t, dev)) Py_RETURN_NONE;
    const long k = x->size(-1), n = gw->size(1), m = x->numel() / k;
    at::Tensor h = empty_rows(*x, n);
    void *const sum = norm.sum_for(x);
    if (m > 0) {
        const hipStream_t stream = stream_of(dev);
        Workspace ws;
        if (!workspace(dev.index(), stream, stream_bytes(GPTQ4_OP_MLP_GATEUP, m, k, n, perm != nullptr), &ws)) return nullptr;
        int rc;
        {
            NoGil unlocked;
            rc = gptq4_stream_mlp_gateup(data(x), data(norm.delta), data(norm.weight), norm.eps, sum, ints(gw), ints(gm), ints(uw), ints(um),
                                         ints(perm), h.data_ptr(), (int)m, (int)k, (int)n, (int)g, ws.data, ws.bytes, stream);
        }
        if (rc) return failed(rc, "gptq4_stream_mlp_gateup");
    }
    if (norm.weight == nullptr) return THPVariable_Wrap(h);
    return Py_BuildValue("NN", norm.stream(v[1]), THPVariable_Wrap(h));
    END_HANDLE_TH_ERRORS
}

// What both QKV functions take behind the weights: positions, cos, sin, heads, head_dim, perm, k buffer, v buffer (None:
// new tensors), row offset, delta, norm weight, eps.
struct Rotary {
    const at::Tensor *positions, *cos, *sin, *perm, *kbuf, *vbuf;
    long heads, dim, offset, capacity = 0;
    Norm norm;
    at::Tensor q, k, v;

    void take(Args &a, int i) {
        positions = a.need(i), cos = a.need(i + 1), sin = a.need(i + 2);
        heads = a.integer(i + 3), dim = a.integer(i + 4);
        perm = a.may(i + 5), kbuf = a.may(i + 6), vbuf = a.may(i + 7);
        offset = a.integer(i + 8);
        norm.delta = a.may(i + 9), norm.weight = a.may(i + 10), norm.eps = (float)a.real(i + 11);
    }
    bool fits(const at::Tensor *x, const at::Tensor *w) {
        if (x->dim() != 3 || w->size(1) != 3 * heads * dim || (kbuf == nullptr) != (vbuf == nullptr) || !norm.fits(x)) return false;
        const at::Device dev = x->device();
        for (const at::Tensor *t : {positions, cos, sin, perm, norm.delta, norm.weight})
            if (!beside(t, dev)) return false;
        const int64_t b = x->size(0), s = x->size(1);
        if (positions->scalar_type() != at::kInt || positions->dim() != 2 || positions->size(0) != b || positions->size(1) != s) return false;
        capacity = s;
        if (kbuf == nullptr) return offset == 0;
        if (kbuf->dim() != 4 || kbuf->sizes() != vbuf->sizes() || !beside(kbuf, dev) || !beside(vbuf, dev)) return false;
        capacity = kbuf->size(2);
        return kbuf->size(0) == b && kbuf->size(1) == heads && kbuf->size(3) == dim && offset >= GPTQ4_KV_AT_POSITION &&
               offset + s <= capacity;
    }
    void outputs(const at::Tensor *x) {
        const int64_t size[4] = {x->size(0), heads, x->size(1), dim};
        q = empty(size, x->device());
        if (kbuf == nullptr) k = empty(size, x->device()), v = empty(size, x->device());
    }
    void *kdata() { return kbuf == nullptr ? k.data_ptr() : data(kbuf); }
    void *vdata() { return vbuf == nullptr ? v.data_ptr() : data(vbuf); }
    PyObject *answer(PyObject *const *args, int i) {
        PyObject *kk = args[i + 6], *vv = args[i + 7];
        if (kbuf == nullptr) {
            kk = THPVariable_Wrap(k), vv = THPVariable_Wrap(v);
        } else {
            Py_INCREF(kk), Py_INCREF(vv);
        }
        if (norm.weight == nullptr) return Py_BuildValue("NNN", THPVariable_Wrap(q), kk, vv);
        return Py_BuildValue("NNNN", THPVariable_Wrap(q), kk, vv, norm.stream(args[1]));
    }
};

// qkv_rotary(groupsize, x, qweight, scales, qzeros, <Rotary>) -> (q, k, v) or, with a norm weight, (q, k, v, x + delta)
PyObject *qkv_rotary(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    GPTQ4_TAKES(17)
    Args a{v};
    const long g = a.integer(0);
    const at::Tensor *x = a.need(1), *w = a.need(2), *s = a.need(3), *z = a.need(4);
    Rotary r;
    r.take(a, 5);
    if (!a.fine || !projection_fits(x, w, g) || !r.fits(x, w)) Py_RETURN_NONE;
    const at::Device dev = x->device();
    for (const at::Tensor *t : {w, s, z})
        if (!beside(t, dev)) Py_RETURN_NONE;
    const long k = x->size(-1), n = w->size(1), b = x->size(0), len = x->size(1);
    r.outputs(x);
    void *const sum = r.norm.sum_for(x);
    if (b * len > 0) {
        const hipStream_t stream = stream_of(dev);
        Workspace ws;
        const bool normed = r.norm.weight != nullptr;
        if (!workspace(dev.index(), stream, plain_bytes(GPTQ4_OP_QKV_ROTARY, b * len, k, n, r.perm != nullptr && !normed), &ws)) return nullptr;
        int rc;
        {
            NoGil unlocked;
            rc = normed ? gptq4_norm_qkv_rotary(data(x), data(r.norm.delta), data(r.norm.weight), r.norm.eps, sum, ints(w), ints(z), data(s),
                                                ints(r.perm), ints(r.positions), floats(r.cos), floats(r.sin), (int)r.cos->size(0),
                                                r.q.data_ptr(), r.kdata(), r.vdata(), (int)b, (int)len, (int)r.heads, (int)r.dim, (int)k,
                                                (int)g, (int)r.capacity, (int)r.offset, ws.data, ws.bytes, stream)
                        : gptq4_qkv_rotary(data(x), ints(w), ints(z), data(s), ints(r.perm), ints(r.positions), floats(r.cos),
                                           floats(r.sin), (int)r.cos->size(0), r.q.data_ptr(), r.kdata(), r.vdata(), (int)b, (int)len,
                                           (int)r.heads, (int)r.dim, (int)k, (int)g, (int)r.capacity, (int)r.offset, ws.data, ws.bytes,
                                           stream);
        }
        if (rc) return failed(rc, normed ? "gptq4_norm_qkv_rotary" : "gptq4_qkv_rotary");
    }
    return r.answer(v, 5);
    END_HANDLE_TH_ERRORS
}

// stream_qkv_rotary(groupsize, x, sweight, smeta, <Rotary>): as qkv_rotary
PyObject *stream_qkv_rotary(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    GPTQ4_TAKES(16)
    Args a{v};
    const long g = a.integer(0);
    const at::Tensor *x = a.need(1), *w = a.need(2), *meta = a.need(3);
    Rotary r;
    r.take(a, 4);
    if (!a.fine || !projection_fits(x, w, g) || !r.fits(x, w)) Py_RETURN_NONE;
    const at::Device dev = x->device();
    for (const at::Tensor *t : {w, meta})
        if (!beside(t, dev)) Py_RETURN_NONE;
    const long k = x->size(-1), n = w->size(1), b = x->size(0), len = x->size(1);
    r.outputs(x);
    void *const sum = r.norm.sum_for(x);
    if (b * len > 0) {
        const hipStream_t stream = stream_of(dev);
        Workspace ws;
        if (!workspace(dev.index(), stream, stream_bytes(GPTQ4_OP_QKV_ROTARY, b * len, k, n, r.perm != nullptr), &ws)) return nullptr;
        int rc;
        {
            NoGil unlocked;
            rc = gptq4_stream_qkv_rotary(data(x), data(r.norm.delta), data(r.norm.weight), r.norm.eps, sum, ints(w), ints(meta),
                                         ints(r.perm), ints(r.positions), floats(r.cos), floats(r.sin), (int)r.cos->size(0), r.q.data_ptr(),
                                         r.kdata(), r.vdata(), (int)b, (int)len, (int)r.heads, (int)r.dim, (int)k, (int)g, (int)r.capacity,
                                         (int)r.offset, ws.data, ws.bytes, stream);
        }
        if (rc) return failed(rc, "gptq4_stream_qkv_rotary");
    }
    return r.answer(v, 4);
    END_HANDLE_TH_ERRORS
}

bool is_order(const at::Tensor *index, int64_t n, at::Device dev) {
    return index == nullptr || (beside(index, dev) && index->scalar_type() == at::kInt && index->dim() == 1 && index->size(0) == n);
}

// rms_norm(x, weight, eps, out_index) -> y
PyObject *rms_norm(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    GPTQ4_TAKES(4)
    Args a{v};
    const at::Tensor *x = a.need(0), *w = a.need(1), *index = a.may(3);
    const float eps = (float)a.real(2);
    if (!a.fine || !is_rows(x) || !is_rows(w)) Py_RETURN_NONE;
    const int64_t h = x->size(-1);
    if (w->dim() != 1 || w->size(0) != h || w->device() != x->device() || h == 0 || h % 8 != 0 || !is_order(index, h, x->device())) Py_RETURN_NONE;
    at::Tensor y = empty(x->sizes(), x->device());
    if (x->numel() > 0) {
        const hipStream_t stream = stream_of(x->device());
        int rc;
        {
            NoGil unlocked;
            rc = gptq4_rmsnorm(data(x), data(w), y.data_ptr(), ints(index), (int)(x->numel() / h), (int)h, eps, stream);
        }
        if (rc) return failed(rc, "gptq4_rmsnorm");
    }
    return THPVariable_Wrap(y);
    END_HANDLE_TH_ERRORS
}

// add_rms_norm(x, delta, weight, eps, out_index) -> (x + delta, y)
PyObject *add_rms_norm(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    GPTQ4_TAKES(5)
    Args a{v};
    const at::Tensor *x = a.need(0), *d = a.need(1), *w = a.need(2), *index = a.may(4);
    const float eps = (float)a.real(3);
    if (!a.fine || !is_rows(x) || !is_rows(d) || !is_rows(w)) Py_RETURN_NONE;
    const int64_t h = x->size(-1);
    if (w->dim() != 1 || w->size(0) != h || w->device() != x->device() || d->device() != x->device() || d->sizes() != x->sizes() || h == 0 ||
        h % 8 != 0 || !is_order(index, h, x->device()))
        Py_RETURN_NONE;
    at::Tensor s = empty(x->sizes(), x->device()), y = empty(x->sizes(), x->device());
    if (x->numel() > 0) {
        const hipStream_t stream = stream_of(x->device());
        int rc;
        {
            NoGil unlocked;
            rc = gptq4_add_rmsnorm(data(x), data(d), data(w), s.data_ptr(), y.data_ptr(), ints(index), (int)(x->numel() / h), (int)h, eps, stream);
        }
        if (rc) return failed(rc, "gptq4_add_rmsnorm");
    }
    return Py_BuildValue("NN", THPVariable_Wrap(s), THPVariable_Wrap(y));
    END_HANDLE_TH_ERRORS
}

// q [B, H, S, 128] and caches [B, H, capacity, 128] of one attention call
bool caches_fit(const at::Tensor *q, const at::Tensor *k, const at::Tensor *v) {
    if (!is_rows(q) || !is_rows(k) || !is_rows(v) || q->dim() != 4 || k->dim() != 4 || k->sizes() != v->sizes()) return false;
    return q->size(3) == 128 && k->size(3) == 128 && k->size(0) == q->size(0) && k->size(1) == q->size(1) && k->device() == q->device() &&
           v->device() == q->device();
}

// prefill_attention(q, k cache, v cache, past) -> [B, S, H * 128]
PyObject *prefill_attention(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    GPTQ4_TAKES(4)
    Args a{v};
    const at::Tensor *q = a.need(0), *kc = a.need(1), *vc = a.need(2);
    const long past = a.integer(3);
    if (!a.fine || !caches_fit(q, kc, vc)) Py_RETURN_NONE;
    const int64_t b = q->size(0), h = q->size(1), s = q->size(2), cap = kc->size(2);
    if (past < 0 || past + s > cap) Py_RETURN_NONE;
    const int64_t size[3] = {b, s, h * 128};
    at::Tensor out = empty(size, q->device());
    if (s > 0) {
        const hipStream_t stream = stream_of(q->device());
        int rc;
        {
            NoGil unlocked;
            rc = gptq4_prefill_attention(data(q), data(kc), data(vc), out.data_ptr(), (int)b, (int)h, (int)s, 128, (int)cap, (int)past,
                                         (float)(1.0 / std::sqrt(128.0)), stream);
        }
        if (rc) return failed(rc, "gptq4_prefill_attention");
    }
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// decode_attention(q, k cache, v cache, positions, out_index) -> [B, 1, H * 128]
PyObject *decode_attention(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    GPTQ4_TAKES(5)
    Args a{v};
    const at::Tensor *q = a.need(0), *kc = a.need(1), *vc = a.need(2), *pos = a.need(3), *index = a.may(4);
    if (!a.fine || !caches_fit(q, kc, vc) || q->size(2) != 1) Py_RETURN_NONE;
    const at::Device dev = q->device();
    const int64_t b = q->size(0), h = q->size(1), cap = kc->size(2);
    if (pos->scalar_type() != at::kInt || !beside(pos, dev) || pos->numel() != b || !is_order(index, h * 128, dev)) Py_RETURN_NONE;
    const int64_t size[3] = {b, 1, h * 128};
    at::Tensor out = empty(size, dev);
    const hipStream_t stream = stream_of(dev);
    Workspace ws;
    if (!workspace(dev.index(), stream, gptq4_workspace_bytes(GPTQ4_OP_DECODE_ATTENTION, (int)(b * h), (int)cap, 0), &ws)) return nullptr;
    int rc;
    {
        NoGil unlocked;
        rc = gptq4_decode_attention(data(q), data(kc), data(vc), ints(pos), out.data_ptr(), ints(index), (int)b, (int)h, 128, (int)cap,
                                    (float)(1.0 / std::sqrt(128.0)), ws.data, ws.bytes, stream);
    }
    if (rc) return failed(rc, "gptq4_decode_attention");
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// extend_attention(q, past k, past v, k, v, out_index) -> [B, 1, H * 128]; past k and v None: no past
PyObject *extend_attention(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    GPTQ4_TAKES(6)
    Args a{v};
    const at::Tensor *q = a.need(0), *pk = a.may(1), *pv = a.may(2), *kc = a.need(3), *vc = a.need(4), *index = a.may(5);
    if (!a.fine || !caches_fit(q, kc, vc) || q->size(2) != 1 || (pk == nullptr) != (pv == nullptr)) Py_RETURN_NONE;
    const at::Device dev = q->device();
    const int64_t b = q->size(0), h = q->size(1), past = pk == nullptr ? 0 : pk->dim() == 4 ? pk->size(2) : -1;
    if (past < 0 || (pk != nullptr && !caches_fit(q, pk, pv)) || kc->size(2) != past + 1 || !is_order(index, h * 128, dev)) Py_RETURN_NONE;
    const int64_t size[3] = {b, 1, h * 128};
    at::Tensor out = empty(size, dev);
    const hipStream_t stream = stream_of(dev);
    Workspace ws;
    if (!workspace(dev.index(), stream, gptq4_workspace_bytes(GPTQ4_OP_DECODE_ATTENTION, (int)(b * h), (int)past + 1, 0), &ws)) return nullptr;
    int rc;
    {
        NoGil unlocked;
        rc = gptq4_extend_attention(data(q), data(pk), data(pv), data(kc), data(vc), out.data_ptr(), ints(index), (int)b, (int)h, 128,
                                    (int)past, (float)(1.0 / std::sqrt(128.0)), ws.data, ws.bytes, stream);
    }
    if (rc) return failed(rc, "gptq4_extend_attention");
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

constexpr size_t HEAD_BYTES = GPTQ4_WS_HEAD_BYTES + (64 << 10);

// the fp16 lm_head weight [V, K] and an embedding of the same shape
bool is_table(const at::Tensor *w, int64_t k, at::Device dev) { return is_rows(w) && w->dim() == 2 && w->size(1) == k && w->device() == dev; }

// lm_head_argmax(x, weight) -> int64 tokens of x's shape without the last dimension
PyObject *lm_head_argmax(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    GPTQ4_TAKES(2)
    Args a{v};
    const at::Tensor *x = a.need(0), *w = a.need(1);
    if (!a.fine || !is_rows(x) || x->size(-1) == 0 || !is_table(w, x->size(-1), x->device())) Py_RETURN_NONE;
    const int64_t k = x->size(-1), b = x->numel() / k;
    at::Tensor out = empty(x->sizes().slice(0, x->dim() - 1), x->device(), at::kLong);
    const hipStream_t stream = stream_of(x->device());
    Workspace ws;
    if (!workspace(x->device().index(), stream, HEAD_BYTES, &ws)) return nullptr;
    int rc;
    {
        NoGil unlocked;
        rc = gptq4_lm_head_argmax(data(x), data(w), out.data_ptr<int64_t>(), (int)b, (int)k, (int)w->size(0), ws.data, ws.bytes, stream);
    }
    if (rc) return failed(rc, "gptq4_lm_head_argmax");
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// lm_head_logits(x, weight) -> fp16 logits, V in the place of x's last dimension
PyObject *lm_head_logits(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    GPTQ4_TAKES(2)
    Args a{v};
    const at::Tensor *x = a.need(0), *w = a.need(1);
    if (!a.fine || !is_rows(x) || x->size(-1) == 0 || !is_table(w, x->size(-1), x->device())) Py_RETURN_NONE;
    const int64_t k = x->size(-1), b = x->numel() / k;
    at::Tensor out = empty_rows(*x, w->size(0));
    const hipStream_t stream = stream_of(x->device());
    int rc;
    {
        NoGil unlocked;
        rc = gptq4_lm_head_logits(data(x), data(w), out.data_ptr(), (int)b, (int)k, (int)w->size(0), stream);
    }
    if (rc) return failed(rc, "gptq4_lm_head_logits");
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// greedy_step_end(x, delta, norm weight, eps, lm_head weight, tokens, positions, history, embedding, next hidden) -> True;
// embedding and next hidden None: not fetched
PyObject *greedy_step_end(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    GPTQ4_TAKES(10)
    Args a{v};
    const at::Tensor *x = a.need(0);
    Norm norm;
    norm.delta = a.may(1), norm.weight = a.may(2), norm.eps = (float)a.real(3);
    const at::Tensor *w = a.need(4), *tokens = a.need(5), *pos = a.need(6), *history = a.need(7), *embed = a.may(8), *next = a.may(9);
    if (!a.fine || !is_rows(x) || x->size(-1) == 0 || !norm.fits(x)) Py_RETURN_NONE;
    const at::Device dev = x->device();
    const int64_t k = x->size(-1), b = x->numel() / k;
    if (!is_table(w, k, dev) || (embed == nullptr) != (next == nullptr)) Py_RETURN_NONE;
    if (embed != nullptr && (!is_table(embed, k, dev) || embed->size(0) < w->size(0) || !is_rows(next) || next->numel() != b * k)) Py_RETURN_NONE;
    for (const at::Tensor *t : {tokens, pos, history, next, norm.delta, norm.weight})
        if (!beside(t, dev)) Py_RETURN_NONE;
    if (tokens->scalar_type() != at::kLong || tokens->numel() != b || pos->scalar_type() != at::kInt || pos->numel() != b ||
        history->scalar_type() != at::kLong || history->dim() != 2 || history->size(0) != b)
        Py_RETURN_NONE;
    const hipStream_t stream = stream_of(dev);
    Workspace ws;
    if (!workspace(dev.index(), stream, HEAD_BYTES, &ws)) return nullptr;
    int rc;
    {
        NoGil unlocked;
        rc = gptq4_greedy_step_end(data(x), data(norm.delta), data(norm.weight), norm.eps, data(w), (int)b, (int)k, (int)w->size(0),
                                   tokens->data_ptr<int64_t>(), pos->data_ptr<int32_t>(), history->data_ptr<int64_t>(), (int)history->size(1),
                                   data(embed), data(next), ws.data, ws.bytes, stream);
    }
    if (rc) return failed(rc, "gptq4_greedy_step_end");
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// stream_rows(selector, K, N, groupsize) -> gptq4_stream_rows()
PyObject *stream_rows(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    GPTQ4_TAKES(4)
    Args a{v};
    const long op = a.integer(0), k = a.integer(1), n = a.integer(2), g = a.integer(3);
    if (!a.fine || op != (int)op || k != (int)k || n != (int)n || g != (int)g) {
        PyErr_SetString(PyExc_TypeError, "stream_rows takes four integers of 32 bits");
        return nullptr;
    }
    return PyLong_FromLong(gptq4_stream_rows((int)op, (int)k, (int)n, (int)g));
    END_HANDLE_TH_ERRORS
}

// set_workspace(device index, stream handle, address, bytes): what _lib.workspace() made for that stream
PyObject *set_workspace(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    GPTQ4_TAKES(4)
    Workspace w;
    w.device = (int)PyLong_AsLong(v[0]);
    w.stream = reinterpret_cast<hipStream_t>(PyLong_AsVoidPtr(v[1]));
    w.data = PyLong_AsVoidPtr(v[2]);
    w.bytes = PyLong_AsSize_t(v[3]);
    if (PyErr_Occurred()) return nullptr;
    for (Workspace &have : g_workspaces)
        if (have.stream == w.stream && have.device == w.device) {
            have = w;
            Py_RETURN_NONE;
        }
    g_workspaces.push_back(w);
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

// init(workspace hook, error hook)
PyObject *init(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
    GPTQ4_TAKES(2)
    Py_INCREF(v[0]), Py_INCREF(v[1]);
    Py_XSETREF(g_workspace_hook, v[0]);
    Py_XSETREF(g_error_hook, v[1]);
    Py_RETURN_NONE;
}

#define GPTQ4_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {GPTQ4_METHOD(init),
                           GPTQ4_METHOD(set_workspace),
                           GPTQ4_METHOD(stream_rows),
                           GPTQ4_METHOD(matmul),
                           GPTQ4_METHOD(stream_matmul),
                           GPTQ4_METHOD(mlp_gateup),
                           GPTQ4_METHOD(stream_mlp_gateup),
                           GPTQ4_METHOD(qkv_rotary),
                           GPTQ4_METHOD(stream_qkv_rotary),
                           GPTQ4_METHOD(rms_norm),
                           GPTQ4_METHOD(add_rms_norm),
                           GPTQ4_METHOD(prefill_attention),
                           GPTQ4_METHOD(decode_attention),
                           GPTQ4_METHOD(extend_attention),
                           GPTQ4_METHOD(lm_head_argmax),
                           GPTQ4_METHOD(lm_head_logits),
                           GPTQ4_METHOD(greedy_step_end),
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_host", "The package's calls of libgptq4 on torch tensors.", -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&g_module); }
