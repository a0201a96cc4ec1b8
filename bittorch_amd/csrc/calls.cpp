// Host side of the calls whose kernels take a few microseconds: what the functions of _C.py do for an ordinary call (plain GPU
// tensors as the library reads them, on the current device), in one native call.  In Python the checks, the allocations, the
// workspace query and some twenty argument conversions were most of such a call's time: one fp16 row through 4096 x 4096 took
// 13.6 us a call around a kernel of 4.6.
//
// Every function returns None for a call that is not ordinary: another dtype, device, stride or alignment, a subclass, a mode, a
// transform or a trace being active, or an argument that the Python function refuses.  _C.py then goes on as if it had not asked,
// with its copies, its conversions and its messages.  Nothing is kept from one call for the next.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <string>
#include <type_traits>

#include "../../include/bittorch_hip.h"

namespace {

// The library as _lib.py has loaded it: bind() gives the addresses.
#define BT_FUNCTIONS(X)                                                                                                       \
    X(bt_last_error) X(bt_tiled_weights_bytes) X(bt_tiled_forward_workspace_bytes) X(bt_packed_forward_workspace_bytes)        \
    X(bt_packed_forward_fused_workspace_bytes) X(bt_tensor_core_workspace_bytes) X(bt_linear_grad_weight_workspace_bytes)      \
    X(bt_linear_grad_weight_16_workspace_bytes) X(bt_ternary_linear_tiled_forward) X(bt_ternary_linear_packed_forward)         \
    X(bt_ternary_linear_tensor_core_forward) X(bt_quantize_pack) X(bt_ternary_linear_grad_input) X(bt_linear_grad_weight)      \
    X(bt_linear_grad_weight_16) X(bt_unpack_dequant) X(bt_swiglu) X(bt_rmsnorm) X(bt_ternary_gemm_i8_tiled) \
    X(bt_ternary_swiglu_i8_tiled) X(bt_act_quant_i8_layout)
struct Library {
#define X(name) decltype(&::name) name = nullptr;
    BT_FUNCTIONS(X)
#undef X
} lib;
bool bound = false;

int tag(at::ScalarType t) {
    return t == at::kFloat ? BT_F32 : t == at::kHalf ? BT_F16 : t == at::kBFloat16 ? BT_BF16 : -1;
}

// No mode, transform or trace that would see, or stand in for, the tensor operations of the Python function.
bool undisturbed() {
    using c10::DispatchKey;
    return bound && at::impl::PythonTorchFunctionTLS::stack_len() == 0 && !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
           !c10::impl::tls_is_dispatch_key_included(DispatchKey::FuncTorchDynamicLayerFrontMode) &&
           !c10::impl::tls_is_dispatch_key_included(DispatchKey::Tracer) &&
           !c10::impl::tls_is_dispatch_key_included(DispatchKey::Functionalize) &&
           !c10::impl::tls_is_dispatch_key_included(DispatchKey::PythonDispatcher);
}

// A tensor of this very class with values of its own on the current device, or null; plain: in contiguous memory.
const at::Tensor* on_device(PyObject* o, int device) {
    using c10::DispatchKey;
    static const c10::DispatchKeySet special({DispatchKey::Python, DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchGradWrapper,
                                              DispatchKey::Batched, DispatchKey::Functionalize, DispatchKey::Conjugate,
                                              DispatchKey::Negative, DispatchKey::ZeroTensor});
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(special) && t.get_device() == device && t.numel() > 0
               ? &t : nullptr;
}
const at::Tensor* plain(PyObject* o, int device) {
    const at::Tensor* t = on_device(o, device);
    return t && t->is_contiguous() ? t : nullptr;
}
bool aligned(const at::Tensor& t, uintptr_t to) { return reinterpret_cast<uintptr_t>(t.const_data_ptr()) % to == 0; }

// A scale or bias vector of n entries (or one), fp32 or 16-bit.
const at::Tensor* vec(PyObject* o, int64_t n, bool one_entry, int device) {
    const at::Tensor* t = plain(o, device);
    return t && t->dim() == 1 && (t->size(0) == n || (one_entry && t->size(0) == 1)) && tag(t->scalar_type()) >= 0 ? t : nullptr;
}

at::Tensor output(at::IntArrayRef shape, at::ScalarType dtype, const at::Tensor& like) {
    return at::empty(shape, at::TensorOptions().dtype(dtype).device(like.device()));
}
struct Scratch {  // of one call
    at::Tensor t;
    Scratch(size_t bytes, const at::Tensor& like) {
        if (bytes) t = output({(int64_t)bytes}, at::kByte, like);
    }
    void* ptr() const { return t.defined() ? t.data_ptr() : nullptr; }
    size_t size() const { return t.defined() ? (size_t)t.numel() : 0; }
};
void* stream_of(int device) { return c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream(); }

struct Unlocked {  // the interpreter, until the end of the block however it is left
    PyThreadState* const state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
};
// The library's call without the interpreter lock, as through ctypes.  Its arguments are values: what they are read from (tensors, whose
// accessors may throw and which other threads may point elsewhere) is asked under the lock.
template <typename... P>
void call(int (*f)(P...), std::common_type_t<P>... args) {
    int rc;
    {
        const Unlocked unlocked;
        rc = f(args...);
    }
    if (rc != 0) {
        const char* text = lib.bt_last_error();
        TORCH_CHECK_WITH(Error, false, text && text[0] ? std::string(text) : "libbittorch_hip call failed (" + std::to_string(rc) + ")");
    }
}

bool as_int(PyObject* o, int64_t* v) {
    if (!PyLong_CheckExact(o)) return false;
    *v = PyLong_AsLongLong(o);
    if (*v == -1 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    return true;
}
bool as_float(PyObject* o, double* v) {
    if (PyFloat_CheckExact(o)) *v = PyFloat_AS_DOUBLE(o);
    else {
        int64_t i;
        if (!as_int(o, &i)) return false;
        *v = (double)i;
    }
    return true;
}
bool as_bool(PyObject* o, bool* v) {
    *v = o == Py_True;
    return o == Py_True || o == Py_False;
}

// The current device, if the first argument is a GPU tensor and nothing stands in between.
bool here(PyObject* o, int* device) {
    if (!undisturbed() || !THPVariable_CheckExact(o) || !THPVariable_Unpack(o).is_cuda()) return false;
    *device = (int)c10::hip::current_device();
    return true;
}
// X as the first argument: rows of values of a float type.
const at::Tensor* rows_of(PyObject* o, int* device) {
    if (!here(o, device)) return nullptr;
    const at::Tensor* x = plain(o, *device);
    return x && x->dim() >= 1 && tag(x->scalar_type()) >= 0 ? x : nullptr;
}
// A residual of the output's shape and dtype.
const at::Tensor* residual_of(PyObject* o, const at::Tensor& x, int64_t n, int device) {
    const at::Tensor* r = plain(o, device);
    if (!r || r->scalar_type() != x.scalar_type() || r->dim() != x.dim() || r->size(-1) != n || !aligned(*r, 16)) return nullptr;
    for (int64_t d = 0; d + 1 < x.dim(); d++)
        if (r->size(d) != x.size(d)) return nullptr;
    return r;
}
at::DimVector with_last(const at::Tensor& x, int64_t n) {
    at::DimVector shape(x.sizes());
    shape.back() = n;
    return shape;
}
#define ORDINARY(cond) \
    if (!(cond)) Py_RETURN_NONE

// tiled_forward(X, W_tiled, scale, bias, in_features, out_features, residual, norm, swiglu_up, swiglu_pairs, natural_from_pairs)
PyObject* tiled_forward(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    int device;
    int64_t K, N;
    bool pairs, natural;
    ORDINARY(n_args == 11);
    const at::Tensor* x = rows_of(a[0], &device);
    ORDINARY(x && as_int(a[4], &K) && as_int(a[5], &N) && as_bool(a[9], &pairs) && as_bool(a[10], &natural));
    ORDINARY(K > 0 && N > 0 && x->size(-1) == K && !(pairs && natural) && (!(pairs || natural) || N % 32 == 0));
    const at::Tensor *w = plain(a[1], device), *scale = vec(a[2], N, true, device);
    ORDINARY(w && scale && w->scalar_type() == at::kByte && w->dim() == 1 && (size_t)w->numel() == lib.bt_tiled_weights_bytes(N, K));
    const at::Tensor *bias = nullptr, *res = nullptr, *pro = nullptr;
    if (a[3] != Py_None) ORDINARY((bias = vec(a[3], N, false, device)));
    if (a[6] != Py_None) ORDINARY(!pairs && (res = residual_of(a[6], *x, N, device)));
    int op = 0;
    double eps = 0.0;
    if (a[7] != Py_None) {
        ORDINARY(a[8] == Py_None && PyTuple_CheckExact(a[7]) && PyTuple_GET_SIZE(a[7]) == 2 && as_float(PyTuple_GET_ITEM(a[7], 1), &eps));
        PyObject* weight = PyTuple_GET_ITEM(a[7], 0);
        op = 1;
        if (weight != Py_None) {
            pro = plain(weight, device);
            ORDINARY(pro && pro->dim() == 1 && pro->size(0) == K && pro->scalar_type() == x->scalar_type());
        }
    } else if (a[8] != Py_None) {
        pro = plain(a[8], device);
        ORDINARY(!pairs && pro && pro->sizes() == x->sizes() && pro->scalar_type() == x->scalar_type());
        op = 2;
    }
    const int dt = tag(x->scalar_type()), epi = pairs ? 1 : natural ? 2 : 0;
    const int64_t B = x->numel() / K, Ny = pairs ? N / 2 : N;
    at::Tensor y = output(with_last(*x, Ny), x->scalar_type(), *x);
    const Scratch ws(op == 0 && !pairs ? lib.bt_tiled_forward_workspace_bytes(B, N, K, dt) : lib.bt_packed_forward_fused_workspace_bytes(B, N, K, dt), *x);
    void* st = stream_of(device);
    call(lib.bt_ternary_linear_tiled_forward, x->const_data_ptr(), K, dt, op, pro ? pro->const_data_ptr() : nullptr,
        op == 2 ? K : 0, (float)eps, (const uint8_t*)w->const_data_ptr(), scale->const_data_ptr(), tag(scale->scalar_type()),
        scale->numel(), bias ? bias->const_data_ptr() : nullptr, bias ? tag(bias->scalar_type()) : 0,
        res ? res->const_data_ptr() : nullptr, epi, y.data_ptr(), B, N, K, ws.ptr(), ws.size(), st);
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// W_T [ceil(K / 4), N]
const at::Tensor* packed_weights(PyObject* o, int64_t K, int device) {
    const at::Tensor* w = plain(o, device);
    return w && w->scalar_type() == at::kByte && w->dim() == 2 && w->size(0) == (K + 3) / 4 ? w : nullptr;
}

// packed_forward(X, W_T, scale, bias, in_features)
PyObject* packed_forward(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    int device;
    int64_t K;
    ORDINARY(n_args == 5);
    const at::Tensor* x = rows_of(a[0], &device);
    ORDINARY(x && as_int(a[4], &K) && K > 0 && x->size(-1) == K);
    const at::Tensor* w = packed_weights(a[1], K, device);
    ORDINARY(w);
    const int64_t N = w->size(1), B = x->numel() / K;
    const at::Tensor *scale = vec(a[2], N, true, device), *bias = nullptr;
    ORDINARY(scale);
    if (a[3] != Py_None) ORDINARY((bias = vec(a[3], N, false, device)));
    const int dt = tag(x->scalar_type());
    at::Tensor y = output(with_last(*x, N), x->scalar_type(), *x);
    const Scratch ws(lib.bt_packed_forward_workspace_bytes(B, N, K, dt), *x);
    void* st = stream_of(device);
    call(lib.bt_ternary_linear_packed_forward, x->const_data_ptr(), dt, (const uint8_t*)w->const_data_ptr(),
        scale->const_data_ptr(), tag(scale->scalar_type()), scale->numel(), bias ? bias->const_data_ptr() : nullptr,
        bias ? tag(bias->scalar_type()) : 0, y.data_ptr(), B, N, K, ws.ptr(), ws.size(), st);
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// tensor_core_forward(X, W_T, scale, bias, in_features): version 2
PyObject* tensor_core_forward(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    int device;
    int64_t K;
    ORDINARY(n_args == 5);
    const at::Tensor* x = rows_of(a[0], &device);
    ORDINARY(x && x->dim() == 2 && as_int(a[4], &K) && K > 0 && x->size(1) == K);
    const at::Tensor* w = packed_weights(a[1], K, device);
    ORDINARY(w);
    const int64_t N = w->size(1), B = x->size(0);
    const at::Tensor *scale = vec(a[2], N, true, device), *bias = nullptr;
    ORDINARY(scale);
    if (a[3] != Py_None) ORDINARY((bias = vec(a[3], N, false, device)));
    at::Tensor y = output({B, N}, x->scalar_type(), *x);
    const Scratch ws(lib.bt_tensor_core_workspace_bytes(B, N, K), *x);
    void* st = stream_of(device);
    call(lib.bt_ternary_linear_tensor_core_forward, x->const_data_ptr(), tag(x->scalar_type()), (const uint8_t*)w->const_data_ptr(),
        scale->const_data_ptr(), tag(scale->scalar_type()), scale->numel(), bias ? bias->const_data_ptr() : nullptr,
        bias ? tag(bias->scalar_type()) : 0, y.data_ptr(), B, N, K, ws.ptr(), ws.size(), st);
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// quantize_pack(weight, threshold_factor, per_channel, as_half) -> (packed, scale, None)
PyObject* quantize_pack(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    int device;
    double threshold;
    bool per_channel, as_half;
    ORDINARY(n_args == 4);
    const at::Tensor* w = rows_of(a[0], &device);
    ORDINARY(w && w->dim() == 2 && as_float(a[1], &threshold) && as_bool(a[2], &per_channel) && as_bool(a[3], &as_half));
    ORDINARY(!as_half || w->scalar_type() == at::kFloat);
    const int64_t N = w->size(0), K = w->size(1);
    at::Tensor packed = output({(K + 3) / 4, N}, at::kByte, *w), scale = output({per_channel ? N : 1}, at::kFloat, *w);
    void* st = stream_of(device);
    constexpr int kF32AsF16 = 4;
    call(lib.bt_quantize_pack, w->const_data_ptr(), as_half ? kF32AsF16 : tag(w->scalar_type()), N, K, threshold,
        per_channel ? 1 : 0, (uint8_t*)packed.data_ptr(), (float*)scale.data_ptr(), nullptr, st);
    const at::ScalarType dtype = as_half ? at::kHalf : w->scalar_type();
    if (dtype != at::kFloat) scale = scale.to(dtype);
    if (!per_channel) scale = scale.squeeze(0);
    PyObject* out = PyTuple_New(3);
    if (!out) return nullptr;
    PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(std::move(packed)));
    PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(std::move(scale)));
    Py_INCREF(Py_None);
    PyTuple_SET_ITEM(out, 2, Py_None);
    return out;
    END_HANDLE_TH_ERRORS
}

// grad_input(dY, W_T, scale, in_features): fp32
PyObject* grad_input(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    int device;
    int64_t K;
    ORDINARY(n_args == 4);
    const at::Tensor* dy = rows_of(a[0], &device);
    ORDINARY(dy && dy->dim() == 2 && dy->scalar_type() == at::kFloat && as_int(a[3], &K) && K > 0);
    const at::Tensor *w = packed_weights(a[1], K, device), *scale = plain(a[2], device);
    const int64_t M = dy->size(0), N = dy->size(1);
    ORDINARY(w && w->size(1) == N && scale && scale->scalar_type() == at::kFloat && (scale->numel() == N || scale->numel() == 1));
    at::Tensor out = output({M, K}, at::kFloat, *dy);
    void* st = stream_of(device);
    call(lib.bt_ternary_linear_grad_input, (const float*)dy->const_data_ptr(), (const uint8_t*)w->const_data_ptr(),
        (const float*)scale->const_data_ptr(), scale->numel(), (float*)out.data_ptr(), M, N, K, st);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// grad_weight(dY, X, scale, want_bias) -> (dW, dBias or None): fp32
PyObject* grad_weight(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    int device;
    bool want_bias;
    ORDINARY(n_args == 4);
    const at::Tensor* dy = rows_of(a[0], &device);
    ORDINARY(dy && dy->dim() == 2 && dy->scalar_type() == at::kFloat && as_bool(a[3], &want_bias));
    const at::Tensor *x = plain(a[1], device), *scale = plain(a[2], device);
    ORDINARY(x && x->dim() == 2 && x->scalar_type() == at::kFloat && x->size(0) == dy->size(0) && scale && scale->scalar_type() == at::kFloat);
    const int64_t M = dy->size(0), N = dy->size(1), K = x->size(1);
    ORDINARY(scale->numel() == N || scale->numel() == 1);
    at::Tensor dw = output({N, K}, at::kFloat, *dy), db;
    if (want_bias) db = output({N}, at::kFloat, *dy);
    const Scratch ws(lib.bt_linear_grad_weight_workspace_bytes(M, N, K), *dy);
    void* st = stream_of(device);
    call(lib.bt_linear_grad_weight, (const float*)dy->const_data_ptr(), (const float*)x->const_data_ptr(),
        (const float*)scale->const_data_ptr(), scale->numel(), (float*)dw.data_ptr(), want_bias ? (float*)db.data_ptr() : nullptr,
        M, N, K, ws.ptr(), ws.size(), st);
    PyObject* out = PyTuple_New(2);
    if (!out) return nullptr;
    PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(std::move(dw)));
    if (want_bias) {
        PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(std::move(db)));
    } else {
        Py_INCREF(Py_None);
        PyTuple_SET_ITEM(out, 1, Py_None);
    }
    return out;
    END_HANDLE_TH_ERRORS
}

// int8 rows quantized by row_op, times a tiled copy:
// gemm_i8_tiled(Q [B, K], s_x, W_tiled, scale, bias, in_features, out_features, like (its dtype), residual [B, N], q_operand_order)
PyObject* gemm_i8_tiled(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    int device;
    int64_t K, N;
    bool oo;
    ORDINARY(n_args == 10 && here(a[0], &device) && as_int(a[5], &K) && as_int(a[6], &N) && as_bool(a[9], &oo) && K > 0 && N > 0);
    const at::Tensor *q = plain(a[0], device), *sx = plain(a[1], device), *w = plain(a[2], device), *scale = vec(a[3], N, true, device);
    ORDINARY(q && q->scalar_type() == at::kChar && q->dim() == 2 && q->size(1) == K && sx && sx->scalar_type() == at::kFloat &&
             sx->numel() == q->size(0) && scale);
    ORDINARY(w && w->scalar_type() == at::kByte && w->dim() == 1 && (size_t)w->numel() == lib.bt_tiled_weights_bytes(N, K));
    ORDINARY(THPDtype_Check(a[7]));
    const at::ScalarType dtype = reinterpret_cast<THPDtype*>(a[7])->scalar_type;
    ORDINARY(tag(dtype) >= 0);
    const int64_t B = q->size(0);
    const at::Tensor *bias = nullptr, *res = nullptr;
    if (a[4] != Py_None) ORDINARY((bias = vec(a[4], N, false, device)));
    if (a[8] != Py_None) {
        res = plain(a[8], device);
        ORDINARY(res && res->scalar_type() == dtype && res->dim() == 2 && res->size(0) == B && res->size(1) == N && aligned(*res, 16));
    }
    at::Tensor y = output({B, N}, dtype, *q);
    void* st = stream_of(device);
    call(lib.bt_ternary_gemm_i8_tiled, (const int8_t*)q->const_data_ptr(), oo ? 1 : 0, (const float*)sx->const_data_ptr(),
        (const uint8_t*)w->const_data_ptr(), scale->const_data_ptr(), tag(scale->scalar_type()), scale->numel(),
        bias ? bias->const_data_ptr() : nullptr, bias ? tag(bias->scalar_type()) : 0, res ? res->const_data_ptr() : nullptr,
        y.data_ptr(), tag(dtype), nullptr, B, N, K, st);
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// swiglu_i8_tiled(Q [B, K] in operand order, s_x, W_tiled, scale, bias, in_features, out_features, dtype) -> [B, N / 2]
PyObject* swiglu_i8_tiled(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    int device;
    int64_t K, N;
    ORDINARY(n_args == 8 && here(a[0], &device) && as_int(a[5], &K) && as_int(a[6], &N) && K > 0 && N > 0 && N % 32 == 0);
    const at::Tensor *q = plain(a[0], device), *sx = plain(a[1], device), *w = plain(a[2], device), *scale = vec(a[3], N, true, device);
    ORDINARY(q && q->scalar_type() == at::kChar && q->dim() == 2 && q->size(1) == K && sx && sx->scalar_type() == at::kFloat &&
             sx->numel() == q->size(0) && scale);
    ORDINARY(w && w->scalar_type() == at::kByte && w->dim() == 1 && (size_t)w->numel() == lib.bt_tiled_weights_bytes(N, K));
    ORDINARY(THPDtype_Check(a[7]));
    const at::ScalarType dtype = reinterpret_cast<THPDtype*>(a[7])->scalar_type;
    ORDINARY(dtype == at::kHalf || dtype == at::kBFloat16);
    const int64_t B = q->size(0);
    const at::Tensor* bias = nullptr;
    if (a[4] != Py_None) ORDINARY((bias = vec(a[4], N, false, device)));
    at::Tensor h = output({B, N / 2}, dtype, *q);
    void* st = stream_of(device);
    call(lib.bt_ternary_swiglu_i8_tiled, (const int8_t*)q->const_data_ptr(), (const float*)sx->const_data_ptr(),
        (const uint8_t*)w->const_data_ptr(), scale->const_data_ptr(), tag(scale->scalar_type()), scale->numel(),
        bias ? bias->const_data_ptr() : nullptr, bias ? tag(bias->scalar_type()) : 0, h.data_ptr(), tag(dtype), B, N, K, st);
    return THPVariable_Wrap(std::move(h));
    END_HANDLE_TH_ERRORS
}

// grad_weight_16(dY, X, scale, out_dtype)
PyObject* grad_weight_16(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    int device;
    ORDINARY(n_args == 4);
    const at::Tensor* dy = rows_of(a[0], &device);
    ORDINARY(dy && dy->dim() == 2 && dy->scalar_type() != at::kFloat && THPDtype_Check(a[3]));
    const at::ScalarType dtype = reinterpret_cast<THPDtype*>(a[3])->scalar_type;
    const at::Tensor *x = plain(a[1], device), *scale = plain(a[2], device);
    ORDINARY(x && x->dim() == 2 && x->scalar_type() == dy->scalar_type() && x->size(0) == dy->size(0) && scale && tag(scale->scalar_type()) >= 0);
    const int64_t M = dy->size(0), N = dy->size(1), K = x->size(1);
    ORDINARY((dtype == dy->scalar_type() || dtype == at::kFloat) && (scale->numel() == N || scale->numel() == 1));
    at::Tensor out = output({N, K}, dtype, *dy);
    const Scratch ws(lib.bt_linear_grad_weight_16_workspace_bytes(M, N, K), *dy);
    void* st = stream_of(device);
    call(lib.bt_linear_grad_weight_16, dy->const_data_ptr(), x->const_data_ptr(), tag(dy->scalar_type()), scale->const_data_ptr(),
        tag(scale->scalar_type()), scale->numel(), out.data_ptr(), tag(dtype), M, N, K, ws.ptr(), ws.size(), st);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// A matrix whose rows lie any distance apart, their elements side by side.
const at::Tensor* strided_rows(PyObject* o, int device) {
    const at::Tensor* t = on_device(o, device);
    return t && t->dim() == 2 && t->stride(1) == 1 && t->stride(0) >= t->size(1) ? t : nullptr;
}
PyObject* int8_rows(at::Tensor q, at::Tensor s) {
    PyObject* out = PyTuple_New(2);
    if (!out) return nullptr;
    PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(std::move(q)));
    PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(std::move(s)));
    return out;
}

// act_quant_int8(x [B, K], operand_order) -> (Q, s_x)
PyObject* act_quant_int8(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    int device;
    bool oo;
    ORDINARY(n_args == 2);
    const at::Tensor* x = rows_of(a[0], &device);
    ORDINARY(x && x->dim() == 2 && as_bool(a[1], &oo));
    const int64_t B = x->size(0), K = x->size(1);
    at::Tensor q = output({B, K}, at::kChar, *x), s = output({B}, at::kFloat, *x);
    void* st = stream_of(device);
    call(lib.bt_act_quant_i8_layout, x->const_data_ptr(), tag(x->scalar_type()), B, K, (int8_t*)q.data_ptr(), (float*)s.data_ptr(),
        oo ? 1 : 0, st);
    return int8_rows(std::move(q), std::move(s));
    END_HANDLE_TH_ERRORS
}

// rmsnorm_int8(x [B, K], weight, eps, operand_order) -> (Q, s_x)
PyObject* rmsnorm_int8(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    int device;
    double eps;
    bool oo;
    ORDINARY(n_args == 4);
    const at::Tensor* x = rows_of(a[0], &device);
    ORDINARY(x && x->dim() == 2 && as_float(a[2], &eps) && as_bool(a[3], &oo));
    const int64_t B = x->size(0), K = x->size(1);
    const at::Tensor* w = nullptr;
    if (a[1] != Py_None) {
        w = plain(a[1], device);
        ORDINARY(w && w->dim() == 1 && w->size(0) == K && w->scalar_type() == x->scalar_type());
    }
    at::Tensor q = output({B, K}, at::kChar, *x), s = output({B}, at::kFloat, *x);
    void* st = stream_of(device);
    call(lib.bt_rmsnorm, x->const_data_ptr(), K, w ? w->const_data_ptr() : nullptr, (float)eps, tag(x->scalar_type()), B, K,
        nullptr, (int8_t*)q.data_ptr(), (float*)s.data_ptr(), oo ? 1 : 0, st);
    return int8_rows(std::move(q), std::move(s));
    END_HANDLE_TH_ERRORS
}

// swiglu_int8(gate [B, K], up [B, K], operand_order) -> (Q, s_x)
PyObject* swiglu_int8(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    int device;
    bool oo;
    ORDINARY(n_args == 3 && here(a[0], &device) && as_bool(a[2], &oo));
    const at::Tensor *g = strided_rows(a[0], device), *u = strided_rows(a[1], device);
    ORDINARY(g && u && tag(g->scalar_type()) >= 0 && u->scalar_type() == g->scalar_type() && u->sizes() == g->sizes());
    const int64_t B = g->size(0), K = g->size(1);
    at::Tensor q = output({B, K}, at::kChar, *g), s = output({B}, at::kFloat, *g);
    void* st = stream_of(device);
    call(lib.bt_swiglu, g->const_data_ptr(), g->stride(0), u->const_data_ptr(), u->stride(0), tag(g->scalar_type()), B, K, nullptr,
        (int8_t*)q.data_ptr(), (float*)s.data_ptr(), oo ? 1 : 0, st);
    return int8_rows(std::move(q), std::move(s));
    END_HANDLE_TH_ERRORS
}

// unpack_dequant(W_T, in_features, scale, out_dtype): dense [N, K] of a float type
PyObject* unpack_dequant(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    int device;
    int64_t K;
    ORDINARY(n_args == 4 && here(a[0], &device) && as_int(a[1], &K) && K > 0 && THPDtype_Check(a[3]));
    const at::ScalarType dtype = reinterpret_cast<THPDtype*>(a[3])->scalar_type;
    const at::Tensor *w = packed_weights(a[0], K, device), *scale = plain(a[2], device);
    ORDINARY(tag(dtype) >= 0 && w && scale && tag(scale->scalar_type()) >= 0 && (scale->numel() == w->size(1) || scale->numel() == 1));
    const at::Tensor scale_f = scale->scalar_type() == at::kFloat ? *scale : scale->detach().to(at::kFloat);
    at::Tensor out = output({w->size(1), K}, dtype, *w);
    void* st = stream_of(device);
    call(lib.bt_unpack_dequant, (const uint8_t*)w->const_data_ptr(), (const float*)scale_f.const_data_ptr(), scale_f.numel(),
        out.data_ptr(), tag(dtype), w->size(1), K, st);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// generic_kernel_asked(): whether BITTORCH_KERNEL=generic, read now
PyObject* generic_kernel_asked(PyObject*, PyObject* const*, Py_ssize_t) {
    const char* env = std::getenv("BITTORCH_KERNEL");
    return PyBool_FromLong(env && !std::strcmp(env, "generic"));
}

// stamp(): what this file was compiled against.  Its accessors are inlined from torch's headers and its calls typed by
// bittorch_hip.h, so _lib.py binds it to that build of torch and that ABI alone.
#define BT_TEXT(x) #x
#define BT_TEXT_OF(x) BT_TEXT(x)
PyObject* stamp(PyObject*, PyObject* const*, Py_ssize_t) { return PyUnicode_FromString("abi " BT_TEXT_OF(BT_ABI_VERSION) ", " BT_CALLS_BUILD); }

// bind({name: address}): the library's functions
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    if (n_args != 1 || !PyDict_Check(a[0])) {
        PyErr_SetString(PyExc_TypeError, "bind takes a dict of addresses");
        return nullptr;
    }
#define X(name)                                                                   \
    {                                                                             \
        PyObject* at = PyDict_GetItemString(a[0], #name);                         \
        void* p = at ? PyLong_AsVoidPtr(at) : nullptr;                            \
        if (!p) {                                                                 \
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_KeyError, #name);        \
            return nullptr;                                                       \
        }                                                                         \
        lib.name = reinterpret_cast<decltype(lib.name)>(p);                       \
    }
    BT_FUNCTIONS(X)
#undef X
    bound = true;
    Py_RETURN_NONE;
}
PyObject* names(PyObject*, PyObject* const*, Py_ssize_t) {
    static const char* const all[] = {
#define X(name) #name,
        BT_FUNCTIONS(X)
#undef X
    };
    PyObject* out = PyList_New(0);
    for (const char* n : all) {
        PyObject* s = PyUnicode_FromString(n);
        if (!out || !s || PyList_Append(out, s) != 0) return nullptr;
        Py_DECREF(s);
    }
    return out;
}

#define METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {METHOD(bind), METHOD(names), METHOD(stamp), METHOD(tiled_forward), METHOD(packed_forward), METHOD(tensor_core_forward),
                         METHOD(quantize_pack), METHOD(grad_input), METHOD(grad_weight),
                         METHOD(grad_weight_16), METHOD(unpack_dequant), METHOD(rmsnorm_int8), METHOD(swiglu_int8), METHOD(gemm_i8_tiled), METHOD(swiglu_i8_tiled), METHOD(act_quant_int8),
                         METHOD(generic_kernel_asked), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", "Native host side of small calls (csrc/calls.cpp)", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls() { return PyModule_Create(&module); }
