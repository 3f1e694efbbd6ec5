// Native fast path of torch_dwconv/_C.py: one CPython call per library call.
//
// What bounds the smallest workloads is the host: a call through ctypes took 13-24 us (a dozen Python checks, the
// allocation, 20 converted arguments) where the kernels of a batch-1 EfficientNet-B0 layer take 4-6 us.  Calls in a row on
// a 14x14 map, us, ctypes / here: dwconv2d 13.1 / 4.4, fused 18.4 / 4.5, backward 19.2 / 9.2, general backward 23.6 / 9.1.
// Each function here makes the checks, the allocations and the library call of its namesake in _C.py, for plain tensors on
// a GPU.  It returns None for anything else (wrong device, dtype or shape, tensor subclasses, tracing, function and dispatch
// modes, functorch wrappers): the Python function then goes its own way, with its own error messages.  Nothing is kept
// between calls.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/version.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <climits>
#include <stdexcept>
#include <string>

#include "dwconv_hip.h"

namespace {

using at::Tensor;

struct NotHere {};   // the call is one for the Python function
struct NoKernel {};  // (fused_backward) a call to serve here, but no kernel makes it: False

// The arguments of one call, taken from left to right.
class Args {
  public:
    Args(PyObject *const *args, Py_ssize_t n) : args_(args), left_(n) {}
    Tensor tensor()
    {
        PyObject *o = next();
        if (!THPVariable_CheckExact(o)) throw NotHere{};
        const Tensor &t = THPVariable_Unpack(o);
        const c10::DispatchKeySet odd({c10::DispatchKey::Python, c10::DispatchKey::ZeroTensor, c10::DispatchKey::Negative,
                                       c10::DispatchKey::Conjugate, c10::DispatchKey::Functionalize});
        if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.key_set().has_any(odd) || !t.has_storage()) throw NotHere{};
        return t;
    }
    c10::optional<Tensor> optional_tensor()
    {
        if (left_ > 0 && *args_ == Py_None) {
            next();
            return c10::nullopt;
        }
        return tensor();
    }
    int integer()
    {
        PyObject *o = next();
        if (!PyLong_Check(o)) throw NotHere{};
        const long v = PyLong_AsLong(o);
        if (v == -1 && PyErr_Occurred()) {
            PyErr_Clear();
            throw NotHere{};
        }
        if (v < INT_MIN || v > INT_MAX) throw NotHere{};
        return static_cast<int>(v);
    }
    void done() const
    {
        if (left_ != 0) throw NotHere{};
    }

  private:
    PyObject *next()
    {
        if (left_ <= 0) throw NotHere{};
        --left_;
        return *args_++;
    }
    PyObject *const *args_;
    Py_ssize_t left_;
};

enum Type { F32, F64, F16, BF16 };

Type type_of(const Tensor &t)
{
    switch (t.scalar_type()) {
        case at::kFloat: return F32;
        case at::kDouble: return F64;
        case at::kHalf: return F16;
        case at::kBFloat16: return BF16;
        default: throw NotHere{};
    }
}

void together(const Tensor &a, const Tensor &b)
{
    if (a.scalar_type() != b.scalar_type() || a.device() != b.device()) throw NotHere{};
}

bool channels_last(const Tensor &t)
{
    return t.dim() == 4 && t.is_contiguous(at::MemoryFormat::ChannelsLast) && !t.is_contiguous();
}

// Extents of a tensor as the library takes them.
int extent(const Tensor &t, int axis)
{
    const int64_t v = t.size(axis);
    if (v > INT_MAX) throw NotHere{};
    return static_cast<int>(v);
}

void input_and_kernel(const Tensor &input, const Tensor &kernel)
{
    if (input.dim() != 4 || kernel.dim() != 4 || kernel.size(0) != input.size(1) || kernel.size(1) != 1) throw NotHere{};
    together(input, kernel);
}

// An uninitialised result; at::empty_like where it takes the strides of an argument (those of axes of one element are free).
Tensor empty_like_format(const Tensor &t, at::IntArrayRef sizes, at::MemoryFormat format)
{
    return at::empty(sizes, t.options().requires_grad(false), format);
}

void *stream_of(const Tensor &t)
{
    return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

// The GIL is free from the parsed arguments to the results, as it is in torch's own functions and in ctypes: an allocation
// may wait for the device, a launch for room in a queue.
class NoGil {
  public:
    NoGil() : state_(PyEval_SaveThread()) {}
    ~NoGil() { PyEval_RestoreThread(state_); }
    NoGil(const NoGil &) = delete;
    NoGil &operator=(const NoGil &) = delete;

  private:
    PyThreadState *state_;
};

// What a function returns: one tensor, or several as a tuple (an undefined one is None).
using Results = c10::SmallVector<Tensor, 4>;

template <typename F>
void call(const Tensor &on, F &&f)
{
    const c10::DeviceGuard guard(on.device());
    const int rc = f(stream_of(on));
    if (rc != 0) throw std::runtime_error("libdwconv_hip error " + std::to_string(rc) + ": " + dwconv_last_error());
}

Tensor workspace(const Tensor &on, size_t bytes)
{
    return at::empty({static_cast<int64_t>(std::max<size_t>(bytes, 1))}, on.options().dtype(at::kByte).requires_grad(false));
}

template <typename T>
const T *in(const Tensor &t)
{
    return static_cast<const T *>(t.const_data_ptr());
}
template <typename T>
T *out(const Tensor &t)
{
    return static_cast<T *>(t.mutable_data_ptr());
}
using Half = unsigned short;  // 16-bit elements at the C boundary

// FN_f32 ... FN_bf16 by element type; NAME(T, fn) is the call.
#define DWCONV_BY_TYPE(TYPE, NAME, FN)                            \
    switch (TYPE) {                                               \
        case F32: NAME(float, FN##_f32) break;                    \
        case F64: NAME(double, FN##_f64) break;                   \
        case F16: NAME(Half, FN##_f16) break;                     \
        default: NAME(Half, FN##_bf16) break;                     \
    }

PyObject *wrap(const Tensor &t)
{
    if (t.defined()) return THPVariable_Wrap(t);
    Py_RETURN_NONE;
}

PyObject *wrap(const Results &results)
{
    if (results.size() == 1) return wrap(results[0]);
    PyObject *tuple = PyTuple_New(static_cast<Py_ssize_t>(results.size()));
    if (tuple == nullptr) return nullptr;
    for (size_t i = 0; i < results.size(); ++i) {
        PyObject *o = wrap(results[i]);
        if (o == nullptr) {
            Py_DECREF(tuple);
            return nullptr;
        }
        PyTuple_SET_ITEM(tuple, static_cast<Py_ssize_t>(i), o);
    }
    return tuple;
}

PyObject *wrap(bool b) { return PyBool_FromLong(b); }

// (input, kernel, up_h, up_w, down_h, down_w, pad_h0, pad_h1, pad_w0, pad_w1, forward)
Results conv(Args a)
{
    const Tensor input = a.tensor(), kernel = a.tensor();
    int v[8];
    for (int &e : v) e = a.integer();
    const int forward = a.integer() != 0;
    a.done();
    const NoGil nogil;
    input_and_kernel(input, kernel);
    const Type type = type_of(input);
    const Tensor x = input.contiguous(), k = kernel.contiguous();
    const int n = extent(x, 0), c = extent(x, 1), h = extent(x, 2), w = extent(x, 3), kh = extent(k, 2), kw = extent(k, 3);
    if (v[2] < 1 || v[3] < 1) throw NotHere{};
    const int oh = std::max(dwconv_out_size(h, v[0], v[2], v[4], v[5], kh), 0);
    const int ow = std::max(dwconv_out_size(w, v[1], v[3], v[6], v[7], kw), 0);
    const Tensor y = empty_like_format(x, {n, c, oh, ow}, at::MemoryFormat::Contiguous);
#define DWCONV_CALL(T, FN)                                                                                                  \
    call(x, [&](void *s) {                                                                                                  \
        return FN(in<T>(x), in<T>(k), out<T>(y), n, c, h, w, kh, kw, v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7], forward, s); \
    });
    DWCONV_BY_TYPE(type, DWCONV_CALL, dwconv2d)
#undef DWCONV_CALL
    return {y};
}

// (input, kernel, up_h, up_w, down_h, down_w, pad_h, pad_w, forward)
Results conv_small(Args a)
{
    const Tensor input = a.tensor(), kernel = a.tensor();
    int v[6];
    for (int &e : v) e = a.integer();
    const int forward = a.integer() != 0;
    a.done();
    const NoGil nogil;
    input_and_kernel(input, kernel);
    const Type type = type_of(input);
    const Tensor x = input.contiguous(), k = kernel.contiguous();
    const int n = extent(x, 0), c = extent(x, 1), h = extent(x, 2), w = extent(x, 3), kh = extent(k, 2), kw = extent(k, 3);
    const Tensor y = at::empty_like(x);
#define DWCONV_CALL(T, FN)                                                                                            \
    call(x, [&](void *s) {                                                                                            \
        return FN(in<T>(x), in<T>(k), out<T>(y), n, c, h, w, kh, kw, v[0], v[1], v[2], v[3], v[4], v[5], forward, s); \
    });
    DWCONV_BY_TYPE(type, DWCONV_CALL, dwconv2d_small)
#undef DWCONV_CALL
    return {y};
}

// (input, out_grad, kernel, stride_h, stride_w, pad_h, pad_w) -> (in_grad, kernel_grad)
Results backward(Args a)
{
    const Tensor input = a.tensor(), grad = a.tensor(), kernel = a.tensor();
    const int sh = a.integer(), sw = a.integer(), ph = a.integer(), pw = a.integer();
    a.done();
    const NoGil nogil;
    input_and_kernel(input, kernel);
    together(input, grad);
    if (grad.dim() != 4 || grad.size(0) != input.size(0) || grad.size(1) != input.size(1)) throw NotHere{};
    const Type type = type_of(input);
    if (type == F64) throw NotHere{};
    const Tensor x = input.contiguous(), gy = grad.contiguous(), k = kernel.contiguous();
    const int n = extent(x, 0), c = extent(x, 1), h = extent(x, 2), w = extent(x, 3), oh = extent(gy, 2), ow = extent(gy, 3);
    const int kh = extent(k, 2), kw = extent(k, 3);
    const Tensor gx = at::empty_like(x);
    const Tensor gw = at::empty_like(k);
    const size_t bytes = dwconv2d_backward_kernel_workspace_bytes(n, c, h, w, oh, ow, kh, kw, sh, sw, ph, pw,
                                                                  static_cast<int>(x.element_size()));
    const Tensor ws = workspace(x, bytes);
#define DWCONV_CALL(T, FN)                                                                                                      \
    call(x, [&](void *s) {                                                                                                      \
        return FN(in<T>(x), in<T>(gy), in<T>(k), out<T>(gx), out<T>(gw), ws.mutable_data_ptr(), bytes, n, c, h, w, oh, ow, kh, kw, \
                  sh, sw, ph, pw, s);                                                                                           \
    });
    switch (type) {
        case F32: DWCONV_CALL(float, dwconv2d_backward_f32) break;
        case F16: DWCONV_CALL(Half, dwconv2d_backward_f16) break;
        default: DWCONV_CALL(Half, dwconv2d_backward_bf16) break;
    }
#undef DWCONV_CALL
    return {gx, gw};
}

// (input, kernel, stride_h, stride_w, pad_h, pad_w), input channels-last or made so
Results conv_nhwc(Args a)
{
    const Tensor input = a.tensor(), kernel = a.tensor();
    const int sh = a.integer(), sw = a.integer(), ph = a.integer(), pw = a.integer();
    a.done();
    const NoGil nogil;
    input_and_kernel(input, kernel);
    const Type type = type_of(input);
    if (sh < 1 || sw < 1) throw NotHere{};
    const Tensor x = input.contiguous(at::MemoryFormat::ChannelsLast), k = kernel.contiguous();
    const int n = extent(x, 0), c = extent(x, 1), h = extent(x, 2), w = extent(x, 3), kh = extent(k, 2), kw = extent(k, 3);
    const int oh = std::max(dwconv_out_size(h, 1, sh, ph, ph, kh), 0), ow = std::max(dwconv_out_size(w, 1, sw, pw, pw, kw), 0);
    const Tensor y = empty_like_format(x, {n, c, oh, ow}, at::MemoryFormat::ChannelsLast);
#define DWCONV_CALL(T, FN) \
    call(x, [&](void *s) { return FN(in<T>(x), in<T>(k), out<T>(y), n, c, h, w, kh, kw, sh, sw, ph, pw, s); });
    DWCONV_BY_TYPE(type, DWCONV_CALL, dwconv2d_nhwc)
#undef DWCONV_CALL
    return {y};
}

// (input, out_grad, kernel, stride_h, stride_w, pad_h, pad_w, need_input_grad, need_kernel_grad)
Results backward_nhwc(Args a)
{
    const Tensor input = a.tensor(), grad = a.tensor(), kernel = a.tensor();
    const int sh = a.integer(), sw = a.integer(), ph = a.integer(), pw = a.integer();
    const bool need_x = a.integer() != 0, need_w = a.integer() != 0;
    a.done();
    const NoGil nogil;
    if (!need_x && !need_w) throw NotHere{};
    input_and_kernel(input, kernel);
    together(input, grad);
    if (grad.dim() != 4 || grad.size(0) != input.size(0) || grad.size(1) != input.size(1)) throw NotHere{};
    const Type type = type_of(input);
    const Tensor x = input.contiguous(at::MemoryFormat::ChannelsLast), gy = grad.contiguous(at::MemoryFormat::ChannelsLast);
    const Tensor k = kernel.contiguous();
    const int n = extent(x, 0), c = extent(x, 1), h = extent(x, 2), w = extent(x, 3), oh = extent(gy, 2), ow = extent(gy, 3);
    const int kh = extent(k, 2), kw = extent(k, 3);
    Tensor gx, gw;
    if (need_x) gx = empty_like_format(x, x.sizes(), at::MemoryFormat::ChannelsLast);
    if (need_w) gw = at::empty_like(k);
    const size_t bytes = dwconv2d_backward_nhwc_workspace_bytes(n, c, h, w, kh, kw, sh, sw, ph, pw, static_cast<int>(x.element_size()));
    const Tensor ws = workspace(x, bytes);
#define DWCONV_CALL(T, FN)                                                                                                  \
    call(x, [&](void *s) {                                                                                                  \
        return FN(in<T>(x), in<T>(gy), in<T>(k), need_x ? out<T>(gx) : nullptr, need_w ? out<T>(gw) : nullptr,              \
                  ws.mutable_data_ptr(), bytes, n, c, h, w, oh, ow, kh, kw, sh, sw, ph, pw, s);                             \
    });
    DWCONV_BY_TYPE(type, DWCONV_CALL, dwconv2d_backward_nhwc)
#undef DWCONV_CALL
    return {gx, gw};
}

// A per-channel vector as the library reads it: fp32 (fp64 beside fp64 tensors), dense, on the tensor's device.
c10::optional<Tensor> per_channel(const c10::optional<Tensor> &t, const Tensor &beside)
{
    if (!t) return t;
    if (t->numel() != beside.size(1)) throw NotHere{};
    const at::ScalarType type = beside.scalar_type() == at::kDouble ? at::kDouble : at::kFloat;
    if (t->dim() == 1 && t->scalar_type() == type && t->device() == beside.device() && t->is_contiguous()) return t;
    return t->detach().reshape(-1).to(beside.device(), type).contiguous();
}

// (input, kernel, scale | None, shift | None, activation, stride_h, stride_w, pad_h, pad_w)
Results fused(Args a)
{
    const Tensor input = a.tensor(), kernel = a.tensor();
    const c10::optional<Tensor> scale_ = a.optional_tensor(), shift_ = a.optional_tensor();
    const int act = a.integer(), sh = a.integer(), sw = a.integer(), ph = a.integer(), pw = a.integer();
    a.done();
    const NoGil nogil;
    input_and_kernel(input, kernel);
    const Type type = type_of(input);
    if (sh < 1 || sw < 1) throw NotHere{};
    const c10::optional<Tensor> scale = per_channel(scale_, input), shift = per_channel(shift_, input);
    const bool nhwc = channels_last(input);
    const at::MemoryFormat format = nhwc ? at::MemoryFormat::ChannelsLast : at::MemoryFormat::Contiguous;
    const Tensor x = input.contiguous(format), k = kernel.contiguous();
    const int n = extent(x, 0), c = extent(x, 1), h = extent(x, 2), w = extent(x, 3), kh = extent(k, 2), kw = extent(k, 3);
    const int oh = std::max(dwconv_out_size(h, 1, sh, ph, ph, kh), 0), ow = std::max(dwconv_out_size(w, 1, sw, pw, pw, kw), 0);
    const Tensor y = empty_like_format(x, {n, c, oh, ow}, format);
    const void *sc = scale ? scale->const_data_ptr() : nullptr, *sf = shift ? shift->const_data_ptr() : nullptr;
#define DWCONV_CALL(T, FN)                                                                                                \
    call(x, [&](void *s) {                                                                                                \
        using P = std::conditional_t<std::is_same<T, double>::value, double, float>;                                      \
        return FN(in<T>(x), in<T>(k), static_cast<const P *>(sc), static_cast<const P *>(sf), out<T>(y), n, c, h, w, kh,  \
                  kw, sh, sw, ph, pw, act, s);                                                                            \
    });
    if (nhwc) {
        DWCONV_BY_TYPE(type, DWCONV_CALL, dwconv2d_fused_nhwc)
    } else {
        DWCONV_BY_TYPE(type, DWCONV_CALL, dwconv2d_fused)
    }
#undef DWCONV_CALL
    return {y};
}

// (conv_out, out_grad, scale | None, shift | None, activation) -> (conv_out overwritten, scale_grad, shift_grad)
Results epilogue_backward(Args a)
{
    const Tensor conv_out = a.tensor(), grad = a.tensor();
    const c10::optional<Tensor> scale_ = a.optional_tensor(), shift_ = a.optional_tensor();
    const int act = a.integer();
    a.done();
    const NoGil nogil;
    together(conv_out, grad);
    if (conv_out.dim() != 4 || grad.sizes() != conv_out.sizes()) throw NotHere{};
    const Type type = type_of(conv_out);
    const bool nhwc = channels_last(conv_out);
    const at::MemoryFormat format = nhwc ? at::MemoryFormat::ChannelsLast : at::MemoryFormat::Contiguous;
    if (type == F64 || !conv_out.is_contiguous(format)) throw NotHere{};
    const c10::optional<Tensor> scale = per_channel(scale_, conv_out), shift = per_channel(shift_, conv_out);
    const Tensor gy = grad.contiguous(format);
    const int n = extent(conv_out, 0), c = extent(conv_out, 1), oh = extent(conv_out, 2), ow = extent(conv_out, 3);
    const Tensor grads = at::empty({c, 2}, conv_out.options().dtype(at::kFloat).requires_grad(false));
    const size_t bytes = dwconv2d_epilogue_backward_workspace_bytes(n, c, oh, ow, nhwc);
    const Tensor ws = workspace(conv_out, bytes);
    const float *sc = scale ? in<float>(*scale) : nullptr, *sf = shift ? in<float>(*shift) : nullptr;
#define DWCONV_CALL(T, FN)                                                                                            \
    call(conv_out, [&](void *s) {                                                                                     \
        return FN(in<T>(conv_out), in<T>(gy), sc, sf, out<T>(conv_out), out<float>(grads), ws.mutable_data_ptr(), bytes, n, c, \
                  oh, ow, act, nhwc, s);                                                                              \
    });
    switch (type) {
        case F32: DWCONV_CALL(float, dwconv2d_epilogue_backward_f32) break;
        case F16: DWCONV_CALL(Half, dwconv2d_epilogue_backward_f16) break;
        default: DWCONV_CALL(Half, dwconv2d_epilogue_backward_bf16) break;
    }
#undef DWCONV_CALL
    return {conv_out, grads.select(1, 0), grads.select(1, 1)};
}

// (input, out_grad, kernel, scale | None, shift | None, activation, stride_h, stride_w, pad_h, pad_w)
//   -> (in_grad, kernel_grad, scale_grad, shift_grad), or False where no kernel makes them in one sweep
Results fused_backward(Args a)
{
    const Tensor input = a.tensor(), grad = a.tensor(), kernel = a.tensor();
    const c10::optional<Tensor> scale_ = a.optional_tensor(), shift_ = a.optional_tensor();
    const int act = a.integer(), sh = a.integer(), sw = a.integer(), ph = a.integer(), pw = a.integer();
    a.done();
    const NoGil nogil;
    input_and_kernel(input, kernel);
    together(input, grad);
    if (grad.dim() != 4 || grad.size(0) != input.size(0) || grad.size(1) != input.size(1)) throw NotHere{};
    const Type type = type_of(input);
    if (type == F64 || channels_last(input)) throw NoKernel{};
    const int n = extent(input, 0), c = extent(input, 1), h = extent(input, 2), w = extent(input, 3), oh = extent(grad, 2), ow = extent(grad, 3);
    const int kh = extent(kernel, 2), kw = extent(kernel, 3);
    const size_t bytes = dwconv2d_fused_backward_workspace_bytes(n, c, h, w, oh, ow, kh, kw, sh, sw, ph, pw,
                                                                 static_cast<int>(input.element_size()));
    if (bytes == 0) throw NoKernel{};
    const c10::optional<Tensor> scale = per_channel(scale_, input), shift = per_channel(shift_, input);
    const Tensor x = input.contiguous(), gy = grad.contiguous(), k = kernel.contiguous();
    const Tensor gx = at::empty_like(x);
    const Tensor gw = at::empty_like(k);
    const Tensor grads = at::empty({c, 2}, x.options().dtype(at::kFloat).requires_grad(false));
    const Tensor ws = workspace(x, bytes);
    const float *sc = scale ? in<float>(*scale) : nullptr, *sf = shift ? in<float>(*shift) : nullptr;
#define DWCONV_CALL(T, FN)                                                                                                     \
    call(x, [&](void *s) {                                                                                                     \
        const int rc = FN(in<T>(x), in<T>(gy), in<T>(k), sc, sf, out<T>(gx), out<T>(gw), out<float>(grads),                    \
                          ws.mutable_data_ptr(), bytes, n, c, h, w, oh, ow, kh, kw, sh, sw, ph, pw, act, s);                   \
        if (rc == DWCONV_ERR_UNSUPPORTED) throw NoKernel{};                                                                     \
        return rc;                                                                                                             \
    });
    switch (type) {
        case F32: DWCONV_CALL(float, dwconv2d_fused_backward_f32) break;
        case F16: DWCONV_CALL(Half, dwconv2d_fused_backward_f16) break;
        default: DWCONV_CALL(Half, dwconv2d_fused_backward_bf16) break;
    }
#undef DWCONV_CALL
    return {gx, gw, grads.select(1, 0), grads.select(1, 1)};
}

// Input and a kernel of shape (C * M, 1, KH, KW); returns M.
int multiplier(const Tensor &input, const Tensor &kernel)
{
    if (input.dim() != 4 || kernel.dim() != 4 || kernel.size(1) != 1 || input.size(1) == 0 || kernel.size(0) == 0 ||
        kernel.size(0) % input.size(1) != 0)
        throw NotHere{};
    together(input, kernel);
    return static_cast<int>(kernel.size(0) / input.size(1));
}
int dilated_out(int in, int k, int stride, int pad, int dil)
{
    const long room = in + 2l * pad - static_cast<long>(dil) * (k - 1) - 1;
    return room < 0 ? 0 : static_cast<int>(room / stride + 1);
}

// (input, kernel, stride_h, stride_w, pad_h, pad_w, dil_h, dil_w)
Results general(Args a)
{
    const Tensor input = a.tensor(), kernel = a.tensor();
    int v[6];
    for (int &e : v) e = a.integer();
    a.done();
    const NoGil nogil;
    const int m = multiplier(input, kernel);
    const Type type = type_of(input);
    if (v[0] < 1 || v[1] < 1) throw NotHere{};
    const Tensor x = input.contiguous(), k = kernel.contiguous();
    const int n = extent(x, 0), c = extent(x, 1), h = extent(x, 2), w = extent(x, 3), kh = extent(k, 2), kw = extent(k, 3);
    const Tensor y = empty_like_format(x, {n, static_cast<int64_t>(c) * m, dilated_out(h, kh, v[0], v[2], v[4]),
                                           dilated_out(w, kw, v[1], v[3], v[5])}, at::MemoryFormat::Contiguous);
#define DWCONV_CALL(T, FN)                                                                                            \
    call(x, [&](void *s) {                                                                                            \
        return FN(in<T>(x), in<T>(k), out<T>(y), n, c, h, w, m, kh, kw, v[0], v[1], v[2], v[3], v[4], v[5], s);       \
    });
    DWCONV_BY_TYPE(type, DWCONV_CALL, dwconv2d_general)
#undef DWCONV_CALL
    return {y};
}

// (input, out_grad, kernel, stride_h, stride_w, pad_h, pad_w, dil_h, dil_w) -> (in_grad, kernel_grad)
Results general_backward(Args a)
{
    const Tensor input = a.tensor(), grad = a.tensor(), kernel = a.tensor();
    int v[6];
    for (int &e : v) e = a.integer();
    a.done();
    const NoGil nogil;
    const int m = multiplier(input, kernel);
    together(input, grad);
    if (grad.dim() != 4 || grad.size(0) != input.size(0) || grad.size(1) != input.size(1) * m) throw NotHere{};
    const Type type = type_of(input);
    const Tensor x = input.contiguous(), gy = grad.contiguous(), k = kernel.contiguous();
    const int n = extent(x, 0), c = extent(x, 1), h = extent(x, 2), w = extent(x, 3), oh = extent(gy, 2), ow = extent(gy, 3);
    const int kh = extent(k, 2), kw = extent(k, 3);
    const Tensor gx = at::empty_like(x);
    const Tensor gw = at::empty_like(k);
    const size_t bytes = dwconv2d_general_backward_workspace_bytes(n, c, h, w, m, kh, kw, v[0], v[1], v[2], v[3], v[4], v[5],
                                                                   static_cast<int>(x.element_size()));
    const Tensor ws = workspace(x, bytes);
#define DWCONV_CALL(T, FN)                                                                                            \
    call(x, [&](void *s) {                                                                                            \
        return FN(in<T>(x), in<T>(gy), in<T>(k), out<T>(gx), out<T>(gw), ws.mutable_data_ptr(), bytes, n, c, h, w, oh, ow, m, \
                  kh, kw, v[0], v[1], v[2], v[3], v[4], v[5], s);                                                     \
    });
    DWCONV_BY_TYPE(type, DWCONV_CALL, dwconv2d_general_backward)
#undef DWCONV_CALL
    return {gx, gw};
}

// (tensor): channels-last and not also dense NCHW
bool is_channels_last(Args a)
{
    const Tensor t = a.tensor();
    a.done();
    return channels_last(t);
}

// (input, kernel, up_h, up_w, down_h, down_w, pad_h, pad_w)
bool use_small(Args a)
{
    const Tensor input = a.tensor(), kernel = a.tensor();
    int v[6];
    for (int &e : v) e = a.integer();
    a.done();
    if (input.dim() != 4 || kernel.dim() != 4) throw NotHere{};
    return dwconv_use_dwconv2d_small(extent(input, 2), extent(input, 3), extent(kernel, 2), extent(kernel, 3), v[0], v[1], v[2],
                                     v[3], v[4], v[5]) != 0;
}

// Modes under which tensor functions are not simply run: the Python functions, which call them one by one, serve then.
bool observed()
{
    return c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled() ||
           torch::jit::tracer::isTracing() ||
           c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) ||
           c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Functionalize);
}

template <auto F>
PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    try {
        if (!observed()) return wrap(F(Args(args, n)));
    } catch (const NotHere &) {
    } catch (const NoKernel &) {
        Py_RETURN_FALSE;
    }
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

#define DWCONV_METHOD(NAME) {#NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<NAME>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {DWCONV_METHOD(conv),          DWCONV_METHOD(conv_small), DWCONV_METHOD(backward),
                         DWCONV_METHOD(conv_nhwc),     DWCONV_METHOD(backward_nhwc), DWCONV_METHOD(fused),
                         DWCONV_METHOD(epilogue_backward), DWCONV_METHOD(fused_backward), DWCONV_METHOD(general),
                         DWCONV_METHOD(general_backward), DWCONV_METHOD(is_channels_last), DWCONV_METHOD(use_small), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_binding", "Native calls behind torch_dwconv._C.", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__binding(void)
{
    PyObject *m = PyModule_Create(&module);
    // torch's C++ interface holds for one release: _C.py uses the module under that one only
    if (m != nullptr && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) != 0) Py_CLEAR(m);
    return m;
}
