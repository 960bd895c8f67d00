// The per-call host work of tennis_amd.capi in C++: argument checks, output allocation, the current stream and the C ABI
// call.  A small layer runs for 4 to 10 us on the GPU; marshalling its call through Python objects and ctypes took 11 to
// 18 us on the host, more than the kernel it launched.  Here a call takes 3 to 5 us, most of it the HIP launch.
//
// Every function takes the arguments of the capi function it stands behind and returns what that returns, or
// NotImplemented for anything but the plain case (device tensors that are contiguous and of the kernel's type, shapes
// that agree, a workspace that is large enough): capi's own code then converts, allocates or raises.  The entry points of
// libtsx_hip.so come as addresses from capi.lib() -- one library in the process, whichever build was loaded.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/TensorBase.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>
#include <memory>
#include <mutex>
#include <vector>

#include "tsx_hip.h"

namespace {

#define TSX_NATIVE_ENTRIES(X)                                                                                              \
    X(tsx_last_error) X(tsx_conv2d_out_size) X(tsx_quantize_f32_i8) X(tsx_conv2d_i8_nchw) X(tsx_quantize_conv2d_i8_nchw)     \
    X(tsx_conv2d_i8_staged_at) X(tsx_gemm_i8) X(tsx_conv2d_f32_nchw_ws) X(tsx_conv2d_f32_workspace_bytes) X(tsx_inner_prod_f32) X(tsx_add_bias_f32)              \
    X(tsx_relu_f32) X(tsx_leaky_relu_f32) X(tsx_add_f32) X(tsx_mul_f32) X(tsx_mish_f32) X(tsx_softplus_f32) X(tsx_tanh_f32) \
    X(tsx_batch_norm_f32) X(tsx_batch_scale_f32) X(tsx_fused_batch_norm_f32) X(tsx_depthwise_conv2d_f32)                    \
    X(tsx_pooling2d_out_size) X(tsx_pooling2d_f32) X(tsx_max_pooling2d_i8_staged) X(tsx_winograd_f63_workspace_bytes)       \
    X(tsx_winograd_f63_fast_workspace_bytes) X(tsx_winograd_f23_workspace_bytes) X(tsx_conv2d_winograd_f63_nchw)            \
    X(tsx_conv2d_winograd_f63_fast_nchw) X(tsx_conv2d_winograd_f23_nchw)

struct Library {
#define X(name) decltype(&::name) name;
    TSX_NATIVE_ENTRIES(X)
#undef X
} L;
PyObject *g_error = nullptr;          // capi.TsxError

struct Decline {};                    // not the plain case: NotImplemented
struct Raised {};                     // a Python error is set

void check(int rc) {
    if (rc == 0) return;
    PyErr_Format(g_error, "tsx error %d: %s", rc, L.tsx_last_error());
    throw Raised{};
}

// ---- arguments

const at::Tensor &tensor(PyObject *o, c10::ScalarType type) {
    if (!THPVariable_Check(o)) throw Decline{};
    const at::Tensor &t = THPVariable_Unpack(o);
    if (!t.is_cuda() || t.scalar_type() != type || !t.is_contiguous()) throw Decline{};
    return t;
}
const at::Tensor &f32(PyObject *o) { return tensor(o, c10::kFloat); }
const at::Tensor &i8(PyObject *o) { return tensor(o, c10::kChar); }
const float *f32_or_null(PyObject *o) { return o == Py_None ? nullptr : f32(o).const_data_ptr<float>(); }

long integer(PyObject *o) {
    const long v = PyLong_AsLong(o);
    if (v == -1 && PyErr_Occurred()) {
        PyErr_Clear();
        throw Decline{};
    }
    return v;
}
double number(PyObject *o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) {
        PyErr_Clear();
        throw Decline{};
    }
    return v;
}
bool truth(PyObject *o) {
    const int v = PyObject_IsTrue(o);
    if (v < 0) {
        PyErr_Clear();
        throw Decline{};
    }
    return v != 0;
}
template <int N>
void integers(PyObject *o, int32_t (&out)[N]) {
    if (!PyTuple_Check(o) || PyTuple_GET_SIZE(o) != N) throw Decline{};
    for (int i = 0; i < N; ++i) out[i] = int32_t(integer(PyTuple_GET_ITEM(o, i)));
}

struct Attr {                         // a new reference, released
    PyObject *o;
    Attr(PyObject *of, PyObject *name) : o(PyObject_GetAttr(of, name)) {
        if (!o) {
            PyErr_Clear();
            throw Decline{};
        }
    }
    ~Attr() { Py_DECREF(o); }
    Attr(const Attr &) = delete;
    Attr &operator=(const Attr &) = delete;
};
PyObject *n_buf, *n_hs, *n_ws, *n_cp, *n_pad_top, *n_pad_left, *n_upsample, *n_x_shape, *n_plan, *n_workspace, *n_keep;
int int_attr(PyObject *of, PyObject *name) { return int(integer(Attr(of, name).o)); }

// ---- results

at::TensorBase empty(at::IntArrayRef shape, c10::ScalarType type, const at::TensorBase &like) {
    return at::detail::empty_cuda(shape, type, like.device(), std::nullopt);
}
PyObject *wrap(at::TensorBase t) { return t.defined() ? THPVariable_Wrap(std::move(t)) : Py_NewRef(Py_None); }
template <class... T>
PyObject *results(T &...out) {        // a tuple of them
    PyObject *all = PyTuple_New(sizeof...(out));
    bool whole = all != nullptr;
    Py_ssize_t i = 0;
    const auto put = [&](at::TensorBase t) {
        PyObject *o = whole ? wrap(std::move(t)) : nullptr;
        whole = o != nullptr;
        if (o) PyTuple_SET_ITEM(all, i++, o);
    };
    (put(std::move(out)), ...);
    if (whole) return all;
    Py_XDECREF(all);
    throw Raised{};
}
void *stream() { return c10::hip::getCurrentHIPStream().stream(); }
template <class T>
T *data(at::TensorBase &t) { return t.defined() ? static_cast<T *>(t.mutable_data_ptr()) : nullptr; }

// ---- launches

// Outputs are allocated and kernels launched with the interpreter released: a launch waits where the stream's queue is full, an
// allocation may wait for the device, and other Python threads run meanwhile.  Everything that reads Python objects comes
// before; what a launch needs of them is held by the caller's arguments or by the function's own references.
struct WithoutGil {
    PyThreadState *state = PyEval_SaveThread();
    ~WithoutGil() { PyEval_RestoreThread(state); }
};
template <class F>
void launch(F &&enqueue) {
    int rc;
    {
        WithoutGil released;
        rc = enqueue();
    }
    check(rc);
}

// The kernels of one call write its workspace and read it back: two threads that share a layer and a stream must not enqueue
// theirs in between.  One of a fixed set of locks by address, held while a call's kernels are enqueued, never while the
// interpreter is waited for.
struct WorkspaceLock {
    std::lock_guard<std::mutex> held;
    explicit WorkspaceLock(const void *workspace) : held(of(workspace)) {}
    static std::mutex &of(const void *workspace) {
        static std::mutex locks[64];
        return locks[(reinterpret_cast<uintptr_t>(workspace) >> 9) % 64];       // allocations lie 512 bytes apart at least
    }
};

template <PyObject *(*F)(PyObject *const *, Py_ssize_t), int N>
PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != N) {
        PyErr_Format(PyExc_TypeError, "%d arguments expected, got %zd", N, n);
        return nullptr;
    }
    try {
        return F(args, n);
    } catch (const Decline &) {
        Py_RETURN_NOTIMPLEMENTED;
    } catch (const Raised &) {
        return nullptr;
    } catch (const std::exception &) {
        // as torch raises it from Python: an output that does not fit is a torch.OutOfMemoryError, which programs catch
        torch::translate_exception_to_python(std::current_exception());
        return nullptr;
    }
}

// ---- element by element

PyObject *unary(PyObject *const *a, Py_ssize_t) {      // what, x, slope
    const at::Tensor &x = f32(a[1]);
    const long what = integer(a[0]);
    const float slope = what == 1 ? float(number(a[2])) : 0.f;
    if (what < 0 || what > 4) throw Decline{};
    at::TensorBase out;
    launch([&] {
        out = empty(x.sizes(), c10::kFloat, x);
        const float *in = x.const_data_ptr<float>();
        float *o = data<float>(out);
        const int64_t n = x.numel();
        switch (what) {
            case 0: return L.tsx_relu_f32(in, n, o, stream());
            case 1: return L.tsx_leaky_relu_f32(in, n, slope, o, stream());
            case 2: return L.tsx_mish_f32(in, n, o, stream());
            case 3: return L.tsx_softplus_f32(in, n, o, stream());
            default: return L.tsx_tanh_f32(in, n, o, stream());
        }
    });
    return wrap(out);
}

PyObject *add(PyObject *const *a, Py_ssize_t) {        // a, b, act, slope, out
    const at::Tensor &x = f32(a[0]), &y = f32(a[1]);
    if (x.sizes() != y.sizes()) throw Decline{};
    const int32_t act = int32_t(integer(a[2]));
    const float slope = float(number(a[3]));
    at::TensorBase out;
    if (a[4] != Py_None) out = f32(a[4]);
    launch([&] {
        if (!out.defined()) out = empty(x.sizes(), c10::kFloat, x);
        return L.tsx_add_f32(x.const_data_ptr<float>(), y.const_data_ptr<float>(), x.numel(), act, slope, data<float>(out), stream());
    });
    return a[4] != Py_None ? Py_NewRef(a[4]) : wrap(out);
}

PyObject *mul(PyObject *const *a, Py_ssize_t) {
    const at::Tensor &x = f32(a[0]), &y = f32(a[1]);
    if (x.sizes() != y.sizes()) throw Decline{};
    at::TensorBase out;
    launch([&] {
        out = empty(x.sizes(), c10::kFloat, x);
        return L.tsx_mul_f32(x.const_data_ptr<float>(), y.const_data_ptr<float>(), x.numel(), data<float>(out), stream());
    });
    return wrap(out);
}

PyObject *quantize(PyObject *const *a, Py_ssize_t) {
    const at::Tensor &x = f32(a[0]), &s = f32(a[1]);
    at::TensorBase out;
    launch([&] {
        out = empty(x.sizes(), c10::kChar, x);
        return L.tsx_quantize_f32_i8(x.const_data_ptr<float>(), x.numel(), s.const_data_ptr<float>(), int32_t(s.numel()), data<int8_t>(out), stream());
    });
    return wrap(out);
}

struct Channels {                                      // x as [pre][channels][inner]
    int64_t pre = 1, inner = 1;
    int32_t channels;
    Channels(const at::Tensor &x, long dim) {
        if (dim < 0 || dim >= x.dim()) throw Decline{};
        for (long d = 0; d < dim; ++d) pre *= x.size(d);
        channels = int32_t(x.size(dim));
        for (long d = dim + 1; d < x.dim(); ++d) inner *= x.size(d);
    }
};

PyObject *add_bias(PyObject *const *a, Py_ssize_t) {   // x, bias, dim
    const at::Tensor &x = f32(a[0]);
    const Channels c(x, integer(a[2]));
    const float *bias = f32(a[1]).const_data_ptr<float>();
    at::TensorBase out;
    launch([&] {
        out = empty(x.sizes(), c10::kFloat, x);
        return L.tsx_add_bias_f32(x.const_data_ptr<float>(), c.pre, c.channels, c.inner, bias, data<float>(out), stream());
    });
    return wrap(out);
}

PyObject *batch_norm(PyObject *const *a, Py_ssize_t) { // x, mean, variance, scale, bias, epsilon, dim; absent pairs None
    const at::Tensor &x = f32(a[0]);
    const float *mean = f32_or_null(a[1]), *variance = f32_or_null(a[2]), *scale = f32_or_null(a[3]), *bias = f32_or_null(a[4]);
    const float epsilon = float(number(a[5]));
    const Channels c(x, integer(a[6]));
    at::TensorBase out;
    launch([&] {
        out = empty(x.sizes(), c10::kFloat, x);
        const float *in = x.const_data_ptr<float>();
        float *o = data<float>(out);
        if (mean && scale) return L.tsx_fused_batch_norm_f32(in, c.pre, c.channels, c.inner, mean, variance, scale, bias, epsilon, o, stream());
        if (mean) return L.tsx_batch_norm_f32(in, c.pre, c.channels, c.inner, mean, variance, epsilon, o, stream());
        return L.tsx_batch_scale_f32(in, c.pre, c.channels, c.inner, scale, bias, o, stream());
    });
    return wrap(out);
}

// ---- pooling

PyObject *pooling2d(PyObject *const *a, Py_ssize_t) {  // x, type, ksize, strides, pads, white
    const at::Tensor &x = f32(a[0]);
    if (x.dim() != 4) throw Decline{};
    int32_t k[2], s[2], p[4], ho, wo;
    integers(a[2], k);
    integers(a[3], s);
    integers(a[4], p);
    const int32_t h = int32_t(x.size(2)), w = int32_t(x.size(3));
    check(L.tsx_pooling2d_out_size(h, w, k[0], k[1], p[0], p[1], p[2], p[3], s[0], s[1], &ho, &wo));
    if (ho <= 0 || wo <= 0) throw Decline{};
    const int32_t type = int32_t(integer(a[1])), white = truth(a[5]) ? 1 : 0;
    at::TensorBase out;
    launch([&] {
        out = empty({x.size(0), x.size(1), ho, wo}, c10::kFloat, x);
        return L.tsx_pooling2d_f32(x.const_data_ptr<float>(), x.size(0) * x.size(1), h, w, type, p[0], p[2], k[0], k[1], s[0], s[1], white,
                                   data<float>(out), ho, wo, stream());
    });
    return wrap(out);
}

struct Shape4 {
    int32_t n, c, h, w;
    explicit Shape4(PyObject *of) {
        Attr shape(of, n_x_shape);
        int32_t v[4];
        integers(shape.o, v);
        n = v[0], c = v[1], h = v[2], w = v[3];
    }
};

tsx_staged_map staged_map(PyObject *o, const at::Tensor &buf) {
    const Shape4 s(o);
    return {buf.mutable_data_ptr(), s.n, int_attr(o, n_hs), int_attr(o, n_ws), int_attr(o, n_cp), int_attr(o, n_pad_top), int_attr(o, n_pad_left),
            s.h, s.w, s.c};
}

PyObject *max_pooling2d_staged(PyObject *const *a, Py_ssize_t) {      // src, dst, ksize, strides, pads
    int32_t k[2], s[2], p[4], ho, wo;
    integers(a[2], k);
    integers(a[3], s);
    integers(a[4], p);
    Attr from(a[0], n_buf), to(a[1], n_buf);
    const tsx_staged_map src = staged_map(a[0], i8(from.o)), dst = staged_map(a[1], i8(to.o));
    check(L.tsx_pooling2d_out_size(src.h, src.w, k[0], k[1], p[0], p[1], p[2], p[3], s[0], s[1], &ho, &wo));
    if (ho != dst.h || wo != dst.w) throw Decline{};
    launch([&] { return L.tsx_max_pooling2d_i8_staged(&src, &dst, k[0], k[1], p[0], p[2], s[0], s[1], stream()); });
    return Py_NewRef(a[1]);
}

// ---- fp32 convolutions and products

tsx_conv2d_geom geometry(const at::Tensor &x, const at::Tensor &w, PyObject *pads, PyObject *strides, PyObject *dilations) {
    if (x.dim() != 4 || w.dim() != 4 || w.size(1) != x.size(1)) throw Decline{};
    int32_t p[4], s[2] = {1, 1}, d[2] = {1, 1};
    integers(pads, p);
    if (strides) integers(strides, s);
    if (dilations) integers(dilations, d);
    return {int32_t(x.size(0)), int32_t(x.size(1)), int32_t(x.size(2)), int32_t(x.size(3)), int32_t(w.size(0)), int32_t(w.size(2)),
            int32_t(w.size(3)), p[0], p[1], p[2], p[3], s[0], s[1], d[0], d[1]};
}

struct OutSize {
    int32_t h, w;
    explicit OutSize(const tsx_conv2d_geom &g) {
        check(L.tsx_conv2d_out_size(&g, &h, &w));
        if (h <= 0 || w <= 0) throw Decline{};
    }
};

PyObject *conv2d_f32(PyObject *const *a, Py_ssize_t) {  // x, w, pads, strides, dilations, padding_value, bias, act, slope
    const at::Tensor &x = f32(a[0]), &w = f32(a[1]);
    const tsx_conv2d_geom g = geometry(x, w, a[2], a[3], a[4]);
    const float *bias = f32_or_null(a[6]);
    const float padding_value = float(number(a[5])), slope = float(number(a[8]));
    const int32_t act = int32_t(integer(a[7]));
    const OutSize o(g);
    at::TensorBase out;
    launch([&] {
        out = empty({g.n, g.cout, o.h, o.w}, c10::kFloat, x);
        const size_t bytes = L.tsx_conv2d_f32_workspace_bytes(&g, w.const_data_ptr<float>());
        at::TensorBase workspace;     // the allocator's again when the call is enqueued, for what follows on this stream
        if (bytes) workspace = empty({int64_t(bytes)}, c10::kByte, x);
        return L.tsx_conv2d_f32_nchw_ws(&g, x.const_data_ptr<float>(), w.const_data_ptr<float>(), padding_value, bias, act, slope, data<float>(out),
                                        data<uint8_t>(workspace), bytes, stream());
    });
    return wrap(out);
}

PyObject *depthwise_conv2d(PyObject *const *a, Py_ssize_t) {          // the same arguments, w [1][c][kh][kw]
    const at::Tensor &x = f32(a[0]), &w = f32(a[1]);
    tsx_conv2d_geom g = geometry(x, w, a[2], a[3], a[4]);
    g.cout = g.c;
    const float *bias = f32_or_null(a[6]);
    const float padding_value = float(number(a[5])), slope = float(number(a[8]));
    const int32_t act = int32_t(integer(a[7]));
    const OutSize o(g);
    at::TensorBase out;
    launch([&] {
        out = empty({g.n, g.cout, o.h, o.w}, c10::kFloat, x);
        return L.tsx_depthwise_conv2d_f32(&g, x.const_data_ptr<float>(), w.const_data_ptr<float>(), padding_value, bias, act, slope, data<float>(out),
                                          stream());
    });
    return wrap(out);
}

PyObject *inner_prod_f32(PyObject *const *a, Py_ssize_t) {            // lhs, rhs, transpose
    const at::Tensor &l = f32(a[0]), &r = f32(a[1]);
    if (l.dim() != 2 || r.dim() != 2) throw Decline{};
    const bool t = truth(a[2]);
    const int64_t k = l.size(1), n = r.size(t ? 0 : 1);
    if (r.size(t ? 1 : 0) != k) throw Decline{};
    at::TensorBase out;
    launch([&] {
        out = empty({l.size(0), n}, c10::kFloat, l);
        return L.tsx_inner_prod_f32(int32_t(l.size(0)), int32_t(n), int32_t(k), l.const_data_ptr<float>(), r.const_data_ptr<float>(), t ? 1 : 0,
                                    data<float>(out), stream());
    });
    return wrap(out);
}

PyObject *winograd(PyObject *const *a, Py_ssize_t) {   // mode (0 f23, 1 f63, 2 f63 fast), x, w, u, workspace, pads, padding_value, bias, act, slope
    const at::Tensor &x = f32(a[1]), &w = f32(a[2]), &u = f32(a[3]);
    const tsx_conv2d_geom g = geometry(x, w, a[5], nullptr, nullptr);
    if (a[4] == Py_None) throw Decline{};
    const at::Tensor &workspace = tensor(a[4], c10::kByte);
    const long mode = integer(a[0]);
    const size_t bytes = mode == 0 ? L.tsx_winograd_f23_workspace_bytes(&g) : mode == 1 ? L.tsx_winograd_f63_workspace_bytes(&g)
                                                                                        : L.tsx_winograd_f63_fast_workspace_bytes(&g);
    if (bytes == 0 || size_t(workspace.numel()) < bytes) throw Decline{};
    const float *bias = f32_or_null(a[7]);
    const float padding_value = float(number(a[6])), slope = float(number(a[9]));
    const int32_t act = int32_t(integer(a[8]));
    const OutSize o(g);
    const auto conv = mode == 0 ? L.tsx_conv2d_winograd_f23_nchw : mode == 1 ? L.tsx_conv2d_winograd_f63_nchw : L.tsx_conv2d_winograd_f63_fast_nchw;
    at::TensorBase out;
    launch([&] {
        out = empty({g.n, g.cout, o.h, o.w}, c10::kFloat, x);
        void *ws = workspace.mutable_data_ptr();
        const WorkspaceLock lock(ws);
        return conv(&g, x.const_data_ptr<float>(), u.const_data_ptr<float>(), padding_value, bias, act, slope, data<float>(out), ws, bytes, stream());
    });
    return wrap(out);
}

// ---- int8

// dq, row_scale, bias, act, slope, q_scales, residual, staged_out, residual_after_act as capi takes them
struct EpilogueArgs {
    PyObject *dq, *row_scale, *bias, *act, *slope, *q_scales, *residual, *staged_out, *residual_after_act;
};

struct HeldEpilogue : tsx_epilogue {
    at::Tensor staged;                // what staged_out_dev points into, whatever the attribute holds by the launch
    HeldEpilogue() : tsx_epilogue{} {}
};

HeldEpilogue epilogue(const EpilogueArgs &a) {
    HeldEpilogue e;
    e.dq_dev = f32(a.dq).const_data_ptr<float>();
    e.row_scale_dev = f32_or_null(a.row_scale);
    e.bias_dev = f32_or_null(a.bias);
    e.act = int32_t(integer(a.act));
    e.slope = float(number(a.slope));
    if (a.q_scales != Py_None) {
        const at::Tensor &q = f32(a.q_scales);
        e.q_scales_dev = q.const_data_ptr<float>();
        e.n_qscales = int32_t(q.numel());
    }
    e.residual_dev = f32_or_null(a.residual);
    e.residual_after_act = truth(a.residual_after_act) ? 1 : 0;
    if (a.staged_out != Py_None) {
        e.staged = i8(Attr(a.staged_out, n_buf).o);
        e.staged_out_dev = e.staged.mutable_data_ptr<int8_t>();
        e.staged_hs = int_attr(a.staged_out, n_hs);
        e.staged_ws = int_attr(a.staged_out, n_ws);
        e.staged_cp = int_attr(a.staged_out, n_cp);
        e.staged_pad_top = int_attr(a.staged_out, n_pad_top);
        e.staged_pad_left = int_attr(a.staged_out, n_pad_left);
        PyObject *up = PyObject_GetAttr(a.staged_out, n_upsample);
        if (up) {
            const long v = PyLong_AsLong(up);
            Py_DECREF(up);
            e.staged_upsample = int32_t(v);
        } else {
            e.staged_upsample = 1;
        }
        if (PyErr_Occurred()) PyErr_Clear();
    }
    return e;
}

PyObject *gemm_i8(PyObject *const *a, Py_ssize_t) {
    // packed, k, n, workspace, a, dq, row_scale, bias, act, slope, q_scales, want_f32, want_acc
    const at::Tensor &packed = tensor(a[0], c10::kByte), &lhs = i8(a[4]);
    const int32_t k = int32_t(integer(a[1])), n = int32_t(integer(a[2]));
    if (lhs.dim() != 2 || lhs.size(1) != k || lhs.size(0) < 1) throw Decline{};
    const int32_t m = int32_t(lhs.size(0));
    void *ws = nullptr;
    size_t ws_bytes = 0;
    if (k % 64 || reinterpret_cast<uintptr_t>(lhs.const_data_ptr()) % 16) {
        if (a[3] == Py_None) throw Decline{};
        const at::Tensor &workspace = tensor(a[3], c10::kByte);
        ws_bytes = size_t(m) * size_t((k + 63) / 64 * 64);
        if (size_t(workspace.numel()) < ws_bytes) throw Decline{};
        ws = workspace.mutable_data_ptr();
    }
    const bool with = a[5] != Py_None;
    HeldEpilogue e;
    if (with) e = epilogue({a[5], a[6], a[7], a[8], a[9], a[10], Py_None, Py_None, Py_False});
    const bool want_f32 = with && truth(a[11]), want_i8 = with && a[10] != Py_None, want_acc = truth(a[12]);
    at::TensorBase out_f32, out_i8, acc;
    launch([&] {
        if (want_f32) out_f32 = empty({m, n}, c10::kFloat, lhs);
        if (want_i8) out_i8 = empty({m, n}, c10::kChar, lhs);
        if (want_acc) acc = empty({m, n}, c10::kInt, lhs);
        const auto enqueue = [&] {
            return L.tsx_gemm_i8(m, n, k, lhs.const_data_ptr<int8_t>(), packed.const_data_ptr(), with ? &e : nullptr, data<float>(out_f32),
                                 data<int8_t>(out_i8), data<int32_t>(acc), ws, ws_bytes, stream());
        };
        if (!ws) return enqueue();
        const WorkspaceLock lock(ws);
        return enqueue();
    });
    return results(out_f32, out_i8, acc);
}

// What one Conv2dI8 has in hand for the input shapes it has seen last: geometry, packed weights, workspace and output size.
// A call holds the plan it uses: reading the attributes of its other arguments can run Python code, and with it other calls
// of the layer that replace the plans kept.
struct Plan {
    tsx_conv2d_geom geom;
    at::Tensor packed;
    size_t ws_bytes;
    int32_t ho, wo;
};
struct ConvState {
    PyObject_HEAD
    int32_t consts[11];               // cout, kh, kw, pads, strides, dilations
    int32_t cin;
    float padding_value;
    std::vector<std::shared_ptr<const Plan>> *plans;
    size_t turn;
};

PyObject *conv_state_new(PyTypeObject *type, PyObject *args, PyObject *) {
    PyObject *w;
    int p[4], s[2], d[2];
    float padding_value;
    if (!PyArg_ParseTuple(args, "O(iiii)(ii)(ii)f", &w, &p[0], &p[1], &p[2], &p[3], &s[0], &s[1], &d[0], &d[1], &padding_value)) return nullptr;
    if (!THPVariable_Check(w) || THPVariable_Unpack(w).dim() != 4) {
        PyErr_SetString(PyExc_TypeError, "conv weights: a tensor of four axes expected");
        return nullptr;
    }
    ConvState *self = reinterpret_cast<ConvState *>(type->tp_alloc(type, 0));
    if (!self) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(w);
    const int32_t c[11] = {int32_t(t.size(0)), int32_t(t.size(2)), int32_t(t.size(3)), p[0], p[1], p[2], p[3], s[0], s[1], d[0], d[1]};
    std::memcpy(self->consts, c, sizeof(c));
    self->cin = int32_t(t.size(1));
    self->padding_value = padding_value;
    self->plans = new std::vector<std::shared_ptr<const Plan>>();
    return reinterpret_cast<PyObject *>(self);
}
void conv_state_dealloc(PyObject *o) {
    delete reinterpret_cast<ConvState *>(o)->plans;
    Py_TYPE(o)->tp_free(o);
}

// layer._plan: packs the weights where that is due and grows layer._workspace to what the shape needs
PyObject *call_plan(PyObject *layer, int32_t n, int32_t c, int32_t h, int32_t w) {
    PyObject *shape = Py_BuildValue("(iiii)", n, c, h, w);
    PyObject *got = shape ? PyObject_CallMethodObjArgs(layer, n_plan, shape, nullptr) : nullptr;
    Py_XDECREF(shape);
    if (!got) throw Raised{};
    return got;
}

// The plan of `layer` (a capi.Conv2dI8) for an input shape
std::shared_ptr<const Plan> conv_plan(ConvState *st, PyObject *layer, int32_t n, int32_t c, int32_t h, int32_t w) {
    for (const auto &p : *st->plans)
        if (p->geom.n == n && p->geom.h == h && p->geom.w == w && p->geom.c == c) return p;
    if (c != st->cin) throw Decline{};
    PyObject *got = call_plan(layer, n, c, h, w);
    Plan p;
    const int32_t *k = st->consts;
    p.geom = {n, c, h, w, k[0], k[1], k[2], k[3], k[4], k[5], k[6], k[7], k[8], k[9], k[10]};
    PyObject *packed = PyTuple_GetItem(got, 1), *bytes = PyTuple_GetItem(got, 2);
    if (!packed || !bytes || !THPVariable_Check(packed)) {
        Py_DECREF(got);
        PyErr_Clear();
        throw Decline{};
    }
    p.packed = THPVariable_Unpack(packed);
    p.ws_bytes = PyLong_AsSize_t(bytes);
    Py_DECREF(got);
    check(L.tsx_conv2d_out_size(&p.geom, &p.ho, &p.wo));
    constexpr size_t MOST = 8;        // input shapes a layer keeps plans for
    auto made = std::make_shared<const Plan>(std::move(p));
    if (st->plans->size() < MOST) st->plans->push_back(made);
    else (*st->plans)[st->turn++ % MOST] = made;
    return made;
}

// The layer's one workspace, as large as the largest shape it has been called with; the call holds it while it enqueues
at::Tensor conv_workspace(PyObject *layer, const Plan &p) {
    for (int turn = 0; turn < 2; ++turn) {
        Attr held(layer, n_workspace);
        if (held.o != Py_None) {
            const at::Tensor &t = tensor(held.o, c10::kByte);
            if (size_t(t.numel()) >= p.ws_bytes) {
                // a graph that is being captured goes on writing it when a larger shape has replaced it
                if (c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None) {
                    PyObject *none = PyObject_CallMethodObjArgs(layer, n_keep, held.o, nullptr);
                    if (!none) throw Raised{};
                    Py_DECREF(none);
                }
                return t;
            }
        }
        if (turn == 0) Py_DECREF(call_plan(layer, p.geom.n, p.geom.c, p.geom.h, p.geom.w));
    }
    throw Decline{};
}

void check_residual(PyObject *residual, const Plan &p) {
    if (residual == Py_None) return;
    const at::Tensor &r = f32(residual);
    if (r.dim() != 4 || r.size(0) != p.geom.n || r.size(1) != p.geom.cout || r.size(2) != p.ho || r.size(3) != p.wo) throw Decline{};
}

PyObject *conv_i8(PyObject *const *a, Py_ssize_t) {
    // state, layer, x, dq, bias, act, slope, q_scales, x_scales, want_f32, want_acc, residual, staged_out, residual_after_act
    ConvState *st = reinterpret_cast<ConvState *>(a[0]);
    const bool fused = a[8] != Py_None;
    const at::Tensor &x = fused ? f32(a[2]) : i8(a[2]);
    if (x.dim() != 4) throw Decline{};
    const auto plan = conv_plan(st, a[1], int32_t(x.size(0)), int32_t(x.size(1)), int32_t(x.size(2)), int32_t(x.size(3)));
    const Plan &p = *plan;
    const bool with = a[3] != Py_None;
    HeldEpilogue e;
    if (with) {
        check_residual(a[11], p);
        e = epilogue({a[3], Py_None, a[4], a[5], a[6], a[7], a[11], a[12], a[13]});
    } else if (a[11] != Py_None) {
        throw Decline{};
    }
    const bool want_f32 = with && truth(a[9]), want_i8 = with && a[7] != Py_None && a[12] == Py_None, want_acc = truth(a[10]);
    const at::Tensor *xs = fused ? &f32(a[8]) : nullptr;
    const at::Tensor workspace = conv_workspace(a[1], p);
    at::TensorBase out_f32, out_i8, acc;
    launch([&] {
        const int64_t shape[4] = {p.geom.n, p.geom.cout, p.ho, p.wo};
        if (want_f32) out_f32 = empty(shape, c10::kFloat, x);
        if (want_i8) out_i8 = empty(shape, c10::kChar, x);
        if (want_acc) acc = empty(shape, c10::kInt, x);
        const tsx_epilogue *ep = with ? &e : nullptr;
        void *ws = workspace.mutable_data_ptr();
        const WorkspaceLock lock(ws);
        if (fused)
            return L.tsx_quantize_conv2d_i8_nchw(&p.geom, x.const_data_ptr<float>(), xs->const_data_ptr<float>(), int32_t(xs->numel()),
                                                 p.packed.const_data_ptr(), st->padding_value, ep, data<float>(out_f32), data<int8_t>(out_i8),
                                                 data<int32_t>(acc), ws, p.ws_bytes, stream());
        return L.tsx_conv2d_i8_nchw(&p.geom, x.const_data_ptr<int8_t>(), p.packed.const_data_ptr(), st->padding_value, ep, data<float>(out_f32),
                                    data<int8_t>(out_i8), data<int32_t>(acc), ws, p.ws_bytes, stream());
    });
    return results(out_f32, out_i8, acc);
}

PyObject *conv_i8_staged(PyObject *const *a, Py_ssize_t) {
    // state, layer, staged, dq, bias, act, slope, q_scales, want_f32, residual, staged_out, residual_after_act
    ConvState *st = reinterpret_cast<ConvState *>(a[0]);
    const Shape4 s(a[2]);
    const auto plan = conv_plan(st, a[1], s.n, s.c, s.h, s.w);
    const Plan &p = *plan;
    Attr buf(a[2], n_buf);
    const at::Tensor &in = i8(buf.o);
    check_residual(a[9], p);
    const HeldEpilogue e = epilogue({a[3], Py_None, a[4], a[5], a[6], a[7], a[9], a[10], a[11]});
    const int hs = int_attr(a[2], n_hs), ws = int_attr(a[2], n_ws);
    const bool want_f32 = truth(a[8]), want_i8 = a[7] != Py_None && a[10] == Py_None;
    at::TensorBase out_f32, out_i8;
    launch([&] {
        const int64_t shape[4] = {p.geom.n, p.geom.cout, p.ho, p.wo};
        if (want_f32) out_f32 = empty(shape, c10::kFloat, in);
        if (want_i8) out_i8 = empty(shape, c10::kChar, in);
        return L.tsx_conv2d_i8_staged_at(&p.geom, in.const_data_ptr(), hs, ws, p.packed.const_data_ptr(), &e, data<float>(out_f32), data<int8_t>(out_i8),
                                         nullptr, stream());
    });
    return results(out_f32, out_i8);
}

// ---- module

PyObject *bind(PyObject *, PyObject *args) {           // {entry point: address}, TsxError
    PyObject *entries, *error;
    if (!PyArg_ParseTuple(args, "O!O", &PyDict_Type, &entries, &error)) return nullptr;
#define X(name)                                                                                              \
    {                                                                                                        \
        PyObject *at = PyDict_GetItemString(entries, #name);                                                 \
        void *address = at ? PyLong_AsVoidPtr(at) : nullptr;                                                 \
        if (!address) {                                                                                      \
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_KeyError, #name);                                   \
            return nullptr;                                                                                  \
        }                                                                                                    \
        L.name = reinterpret_cast<decltype(&::name)>(address);                                               \
    }
    TSX_NATIVE_ENTRIES(X)
#undef X
    Py_INCREF(error);
    Py_XSETREF(g_error, error);
    Py_RETURN_NONE;
}

PyTypeObject conv_state_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

#define TSX_METHOD(name, count) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<name, count>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    TSX_METHOD(unary, 3), TSX_METHOD(add, 5), TSX_METHOD(mul, 2), TSX_METHOD(quantize, 2), TSX_METHOD(add_bias, 3), TSX_METHOD(batch_norm, 7),
    TSX_METHOD(pooling2d, 6), TSX_METHOD(max_pooling2d_staged, 5), TSX_METHOD(conv2d_f32, 9), TSX_METHOD(depthwise_conv2d, 9),
    TSX_METHOD(inner_prod_f32, 3), TSX_METHOD(winograd, 10), TSX_METHOD(gemm_i8, 13), TSX_METHOD(conv_i8, 14), TSX_METHOD(conv_i8_staged, 12),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_tsx_native", "The host work of tennis_amd.capi's calls.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__tsx_native() {
    struct { PyObject **at; const char *name; } names[] = {
        {&n_buf, "buf"}, {&n_hs, "hs"}, {&n_ws, "ws"}, {&n_cp, "cp"}, {&n_pad_top, "pad_top"}, {&n_pad_left, "pad_left"},
        {&n_upsample, "upsample"}, {&n_x_shape, "x_shape"}, {&n_plan, "_plan"}, {&n_workspace, "_workspace"}, {&n_keep, "_keep_for_graph"}};
    for (auto &n : names)
        if (!(*n.at = PyUnicode_InternFromString(n.name))) return nullptr;
    conv_state_type.tp_name = "_tsx_native.ConvState";
    conv_state_type.tp_basicsize = sizeof(ConvState);
    conv_state_type.tp_flags = Py_TPFLAGS_DEFAULT;
    conv_state_type.tp_new = conv_state_new;
    conv_state_type.tp_dealloc = conv_state_dealloc;
    if (PyType_Ready(&conv_state_type) < 0) return nullptr;
    PyObject *m = PyModule_Create(&module);
    if (!m) return nullptr;
    Py_INCREF(&conv_state_type);
    if (PyModule_AddObject(m, "ConvState", reinterpret_cast<PyObject *>(&conv_state_type)) < 0) return nullptr;
    return m;
}
