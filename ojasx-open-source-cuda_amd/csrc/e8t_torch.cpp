// e8t_torch.cpp -- the eager calls of ojasx_amd on plain GPU tensors, without the Python-level
// op dispatch (a CPython extension over the C ABI and torch's C++ tensors).
//
// A call of a torch.library custom op from Python costs 15-20 us of host time before its
// kernel is enqueued (op dispatch through Python kernels, argument checks, allocation, the
// ctypes call), more than most decode and small-batch kernels run.  These functions make
// the same checks, allocations and library calls in C++.  Each returns None, having done
// nothing, for every call that is not plain eager work on tensors it knows: the caller then
// takes the registered op, which handles (or refuses) it as before.  Plain means: exact
// Tensor or Parameter objects on one ROCm device; no autograd to record (grad mode off, or
// nothing requires grad); no tangents; and no dispatch or function mode, functorch
// transform or tracer active.
//
// Measured, us per call among others: one bf16 token through a 4096 x 4096 layer 26.2 -> 6.2
// (host time 5.9, kernel 5.2), 77 rows in 2 bits through 3072 x 4100 32.0 -> 21.2, a training
// step of 16 fp32 tokens with an adapter 239 -> 106.

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/record_function.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <string>

#include "../../include/ojasx_e8t.h"

namespace {

using at::Tensor;

// Tensors and thread states that only the dispatcher treats correctly.
const c10::DispatchKeySet kSpecialTensor({
    c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::Conjugate,
    c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor, c10::DispatchKey::Functionalize,
    c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
    c10::DispatchKey::BatchedNestedTensor, c10::DispatchKey::Batched,
});
const c10::DispatchKeySet kSpecialState({
    c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::PythonDispatcher,
    c10::DispatchKey::PreDispatch, c10::DispatchKey::Functionalize, c10::DispatchKey::Tracer,
    c10::DispatchKey::FuncTorchDynamicLayerFrontMode, c10::DispatchKey::FuncTorchDynamicLayerBackMode,
    c10::DispatchKey::FuncTorchVmapMode, c10::DispatchKey::VmapMode,
});

bool plain_state() {
    return c10::impl::TorchDispatchModeTLS::stack_len() == 0 &&
           at::impl::PythonTorchFunctionTLS::stack_len() == 0 &&
           !c10::impl::tls_local_dispatch_key_set().included_.has_any(kSpecialState);
}

bool plain(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return false;
    const Tensor& t = THPVariable_Unpack(o);
    return t.defined() && t.layout() == at::kStrided && t.is_cuda() &&
           !t.key_set().has_any(kSpecialTensor) && !t._fw_grad(0).defined();
}

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return OJX_F32;
        case at::kHalf: return OJX_F16;
        case at::kBFloat16: return OJX_BF16;
        default: return -1;
    }
}

// Code bytes of `padded` weights; the unit a group size must be a multiple of.
int64_t code_bytes(int fmt, int64_t padded) {
    return fmt == OJX_FMT_TERNARY ? padded * 3 / 16 : fmt == OJX_FMT_E8 ? padded / 4 : padded / 8;
}
int64_t gs_unit(int fmt) { return fmt == OJX_FMT_TERNARY ? 16 : fmt == OJX_FMT_E8 ? 4 : 8; }
int64_t padded_to(int64_t n, int64_t gs) { return n + (gs - n % gs) % gs; }

// A layer's buffers as the ops accept them without a copy.
bool layer_ok(const Tensor& packed, const Tensor& scales, int fmt, int64_t N, int64_t K,
              int64_t gs) {
    if (fmt < 0 || fmt > 2 || gs <= 0 || gs % gs_unit(fmt) != 0 || N < 1 || K < 1) return false;
    const int64_t padded = padded_to(N * K, gs);
    return packed.scalar_type() == at::kByte && scales.scalar_type() == at::kHalf &&
           packed.is_contiguous() && scales.is_contiguous() &&
           packed.numel() >= code_bytes(fmt, padded) && scales.numel() >= padded / gs;
}

// The interpreter lock is given up while memory is allocated and kernels are launched, as the
// registered ops do: both can wait (a full queue, a new segment), and other threads go on.
class Unlocked {
  public:
    Unlocked() : state_(PyEval_SaveThread()) {}
    ~Unlocked() { lock(); }
    void lock() {
        if (state_) PyEval_RestoreThread(state_);
        state_ = nullptr;
    }

  private:
    PyThreadState* state_;
};

void* data(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

void* current_stream(const c10::Device& d) {
    return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(d.index()).stream();
}

void check(int status, const char* what) {
    if (status != OJX_OK)
        throw std::runtime_error(std::string("ojasx_e8t ") + what + " failed (status " +
                                 std::to_string(status) + "): " + ojx_e8t_last_error());
}

Tensor workspace(size_t bytes, const Tensor& like) {
    return bytes ? at::empty({(int64_t)bytes}, like.options().dtype(at::kByte)) : Tensor();
}

struct Args {
    PyObject* const* a;
    Py_ssize_t n;
    int64_t i64(int i) const {
        const int64_t v = PyLong_AsLongLong(a[i]);
        if (v == -1 && PyErr_Occurred()) throw python_error();
        return v;
    }
    double f64(int i) const {
        const double v = PyFloat_AsDouble(a[i]);
        if (v == -1.0 && PyErr_Occurred()) throw python_error();
        return v;
    }
    bool flag(int i) const { return a[i] == Py_True; }
    const Tensor& t(int i) const { return THPVariable_Unpack(a[i]); }
};

void expect(Py_ssize_t n, Py_ssize_t want, const char* what) {
    if (n != want)
        throw std::runtime_error(std::string(what) + " takes " + std::to_string(want) +
                                 " arguments (got " + std::to_string(n) + ")");
}

typedef int (*FwdFn)(const void*, const uint8_t*, const uint16_t*, const void*, void*, int64_t,
                     int64_t, int64_t, int64_t, int, void*, size_t, void*);
typedef int (*LoraFn)(const void*, const uint8_t*, const uint16_t*, const void*, const void*,
                      const void*, int64_t, float, float*, void*, int64_t, int64_t, int64_t,
                      int64_t, int, void*, size_t, void*);
typedef int (*BwdFn)(const void*, const uint8_t*, const uint16_t*, void*, int64_t, int64_t, int64_t,
                     int64_t, int, void*, size_t, void*);
const FwdFn kFwd[] = {ojx_e8t_gemm_fwd, ojx_e8_gemm_fwd, ojx_e8r_gemm_fwd};
const LoraFn kFwdLora[] = {ojx_e8t_gemm_fwd_lora, ojx_e8_gemm_fwd_lora, ojx_e8r_gemm_fwd_lora};
const BwdFn kBwd[] = {ojx_e8t_gemm_bwd_dx, ojx_e8_gemm_bwd_dx, ojx_e8r_gemm_bwd_dx};

bool records(const Tensor& t) { return t.defined() && t.requires_grad(); }

std::vector<int64_t> with_last(const Tensor& x, int64_t last) {
    std::vector<int64_t> s(x.sizes().begin(), x.sizes().end());
    s.back() = last;
    return s;
}

// linear(x, packed, scales, bias | None, N, K, gs, fmt): y, the forward of one layer
PyObject* linear(PyObject*, PyObject* const* argv, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    expect(n, 8, "linear");
    const Args a{argv, n};
    if (!plain_state() || !plain(argv[0]) || !plain(argv[1]) || !plain(argv[2]) ||
        (argv[3] != Py_None && !plain(argv[3])))
        Py_RETURN_NONE;
    const Tensor &x = a.t(0), &packed = a.t(1), &scales = a.t(2);
    const Tensor bias = argv[3] == Py_None ? Tensor() : a.t(3);
    const int64_t N = a.i64(4), K = a.i64(5), gs = a.i64(6);
    const int fmt = (int)a.i64(7), dt = dtype_code(x.scalar_type());
    if (dt < 0 || x.dim() < 1 || x.size(-1) != K || !layer_ok(packed, scales, fmt, N, K, gs) ||
        packed.device() != x.device() || scales.device() != x.device())
        Py_RETURN_NONE;
    if (bias.defined() && (bias.numel() != N || bias.scalar_type() != x.scalar_type() ||
                           !bias.is_contiguous() || bias.device() != x.device()))
        Py_RETURN_NONE;
    if (c10::GradMode::is_enabled() && (records(x) || records(bias))) Py_RETURN_NONE;
    RECORD_FUNCTION("ojasx_e8t::linear", std::vector<c10::IValue>());
    Unlocked unlocked;
    const c10::DeviceGuard on_device(x.device());
    const Tensor xc = x.contiguous();
    const int64_t M = xc.numel() / K;
    Tensor y = at::empty(with_last(x, N), x.options());
    size_t bytes = 0;
    check(ojx_gemm_workspace_bytes(fmt, 0, M, N, K, gs, dt, &bytes), "gemm_workspace_bytes");
    const Tensor ws = workspace(bytes, x);
    check(kFwd[fmt](data(xc), (const uint8_t*)data(packed), (const uint16_t*)data(scales),
                    data(bias), data(y), M, N, K, gs, dt, data(ws), bytes,
                    current_stream(x.device())),
          "gemm_fwd");
    unlocked.lock();
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// linear_bwd(gy, packed, scales, N, K, gs, fmt): gx
PyObject* linear_bwd(PyObject*, PyObject* const* argv, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    expect(n, 7, "linear_bwd");
    const Args a{argv, n};
    if (!plain_state() || !plain(argv[0]) || !plain(argv[1]) || !plain(argv[2])) Py_RETURN_NONE;
    const Tensor &gy = a.t(0), &packed = a.t(1), &scales = a.t(2);
    const int64_t N = a.i64(3), K = a.i64(4), gs = a.i64(5);
    const int fmt = (int)a.i64(6), dt = dtype_code(gy.scalar_type());
    if (dt < 0 || gy.dim() < 1 || gy.size(-1) != N || !layer_ok(packed, scales, fmt, N, K, gs) ||
        packed.device() != gy.device() || scales.device() != gy.device() ||
        (c10::GradMode::is_enabled() && records(gy)))
        Py_RETURN_NONE;
    RECORD_FUNCTION("ojasx_e8t::linear_bwd", std::vector<c10::IValue>());
    Unlocked unlocked;
    const c10::DeviceGuard on_device(gy.device());
    const Tensor gc = gy.contiguous();
    const int64_t M = gc.numel() / N;
    Tensor gx = at::empty(with_last(gy, K), gy.options());
    size_t bytes = 0;
    check(ojx_gemm_workspace_bytes(fmt, 1, M, N, K, gs, dt, &bytes), "gemm_workspace_bytes");
    const Tensor ws = workspace(bytes, gy);
    check(kBwd[fmt](data(gc), (const uint8_t*)data(packed), (const uint16_t*)data(scales), data(gx),
                    M, N, K, gs, dt, data(ws), bytes, current_stream(gy.device())),
          "gemm_bwd_dx");
    unlocked.lock();
    return THPVariable_Wrap(std::move(gx));
    END_HANDLE_TH_ERRORS
}

// The adapter's factors as the kernels read them.
bool factors_ok(const Tensor& x, const Tensor& la, const Tensor& lb, int64_t N, int64_t K) {
    return la.dim() == 2 && lb.dim() == 2 && la.size(0) == K && lb.size(1) == N &&
           la.size(1) == lb.size(0) && la.size(1) >= 1 && la.size(1) <= 64 &&
           la.scalar_type() == x.scalar_type() && lb.scalar_type() == x.scalar_type() &&
           la.is_contiguous() && lb.is_contiguous() && la.device() == x.device() &&
           lb.device() == x.device();
}

// linear_lora(x, packed, scales, bias | None, lora_a, lora_b, scaling, fmt, N, K, gs): y
PyObject* linear_lora(PyObject*, PyObject* const* argv, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    expect(n, 11, "linear_lora");
    const Args a{argv, n};
    if (!plain_state() || !plain(argv[0]) || !plain(argv[1]) || !plain(argv[2]) ||
        (argv[3] != Py_None && !plain(argv[3])) || !plain(argv[4]) || !plain(argv[5]))
        Py_RETURN_NONE;
    const Tensor &x = a.t(0), &packed = a.t(1), &scales = a.t(2), &la = a.t(4), &lb = a.t(5);
    const Tensor bias = argv[3] == Py_None ? Tensor() : a.t(3);
    const float scaling = (float)a.f64(6);
    const int fmt = (int)a.i64(7), dt = dtype_code(x.scalar_type());
    const int64_t N = a.i64(8), K = a.i64(9), gs = a.i64(10);
    if (dt < 0 || x.dim() < 1 || x.size(-1) != K || !layer_ok(packed, scales, fmt, N, K, gs) ||
        packed.device() != x.device() || scales.device() != x.device() ||
        !factors_ok(x, la, lb, N, K))
        Py_RETURN_NONE;
    if (bias.defined() && (bias.numel() != N || bias.scalar_type() != x.scalar_type() ||
                           !bias.is_contiguous() || bias.device() != x.device()))
        Py_RETURN_NONE;
    if (c10::GradMode::is_enabled() && (records(x) || records(bias) || records(la) || records(lb)))
        Py_RETURN_NONE;
    RECORD_FUNCTION("ojasx_e8t::linear_lora", std::vector<c10::IValue>());
    Unlocked unlocked;
    const c10::DeviceGuard on_device(x.device());
    const Tensor xc = x.contiguous();
    const int64_t M = xc.numel() / K, r = la.size(1);
    Tensor y = at::empty(with_last(x, N), x.options());
    const Tensor u = at::empty({M, r}, x.options().dtype(at::kFloat));
    size_t bytes = 0;
    check(ojx_gemm_workspace_bytes(fmt, 0, M, N, K, gs, dt, &bytes), "gemm_workspace_bytes");
    const Tensor ws = workspace(bytes, x);
    check(kFwdLora[fmt](data(xc), (const uint8_t*)data(packed), (const uint16_t*)data(scales),
                        data(bias), data(la), data(lb), r, scaling, (float*)data(u), data(y), M, N,
                        K, gs, dt, data(ws), bytes, current_stream(x.device())),
          "gemm_fwd_lora");
    unlocked.lock();
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// linear_lora_bwd(x, gy, packed, scales, lora_a, lora_b, scaling, fmt, N, K, gs, need_x, need_a,
// need_b): (gx | None, ga | None, gb | None)
PyObject* linear_lora_bwd(PyObject*, PyObject* const* argv, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    expect(n, 14, "linear_lora_bwd");
    const Args a{argv, n};
    if (!plain_state()) Py_RETURN_NONE;
    for (int i = 0; i < 6; ++i)
        if (!plain(argv[i])) Py_RETURN_NONE;
    const Tensor &x = a.t(0), &gy = a.t(1), &packed = a.t(2), &scales = a.t(3), &la = a.t(4),
                 &lb = a.t(5);
    const float scaling = (float)a.f64(6);
    const int fmt = (int)a.i64(7), dt = dtype_code(x.scalar_type());
    const int64_t N = a.i64(8), K = a.i64(9), gs = a.i64(10);
    const bool need_x = a.flag(11), need_a = a.flag(12), need_b = a.flag(13);
    if (dt < 0 || gy.scalar_type() != x.scalar_type() || x.dim() < 1 || x.size(-1) != K ||
        gy.dim() < 1 || gy.size(-1) != N || !layer_ok(packed, scales, fmt, N, K, gs) ||
        packed.device() != x.device() || scales.device() != x.device() ||
        gy.device() != x.device() || !factors_ok(x, la, lb, N, K) || x.numel() == 0 ||
        x.numel() / K != gy.numel() / N || c10::GradMode::is_enabled())
        Py_RETURN_NONE;
    RECORD_FUNCTION("ojasx_e8t::linear_lora_bwd", std::vector<c10::IValue>());
    Unlocked unlocked;
    const c10::DeviceGuard on_device(x.device());
    const Tensor xc = x.contiguous(), gc = gy.contiguous();
    const int64_t M = xc.numel() / K, r = la.size(1);
    Tensor gx = need_x ? at::empty(x.sizes(), gy.options()) : Tensor();
    Tensor ga = need_a ? at::empty({K, r}, gy.options()) : Tensor();
    Tensor gb = need_b ? at::empty({r, N}, gy.options()) : Tensor();
    const Tensor uv = at::empty({2, M, r}, x.options().dtype(at::kFloat));
    size_t bytes = 0;
    check(ojx_gemm_bwd_lora_workspace_bytes(fmt, M, N, K, gs, r, need_x, need_a, need_b, dt, &bytes),
          "gemm_bwd_lora_workspace_bytes");
    const Tensor ws = workspace(bytes, x);
    check(ojx_gemm_bwd_lora(fmt, data(xc), data(gc), (const uint8_t*)data(packed),
                            (const uint16_t*)data(scales), data(la), data(lb), r, scaling,
                            (float*)data(uv), data(gx), data(ga), data(gb), M, N, K, gs, dt,
                            data(ws), bytes, current_stream(x.device())),
          "gemm_bwd_lora");
    unlocked.lock();
    PyObject* out = PyTuple_New(3);
    if (!out) throw python_error();
    Tensor* ts[] = {&gx, &ga, &gb};
    for (int i = 0; i < 3; ++i) {
        if (ts[i]->defined()) {
            PyTuple_SET_ITEM(out, i, THPVariable_Wrap(std::move(*ts[i])));
        } else {
            Py_INCREF(Py_None);
            PyTuple_SET_ITEM(out, i, Py_None);
        }
    }
    return out;
    END_HANDLE_TH_ERRORS
}

typedef int (*EncodeFn)(const void*, int, int64_t, int64_t, uint8_t*, uint16_t*, void*);
typedef int (*DecodeFn)(const uint8_t*, const uint16_t*, int64_t, int64_t, int, void*, void*);
const EncodeFn kEncode[] = {ojx_e8t_encode, ojx_e8_encode, ojx_e8r_encode};
const DecodeFn kDecode[] = {ojx_e8t_decode, ojx_e8_decode, ojx_e8r_decode};
int64_t pack_unit(int fmt) { return fmt == OJX_FMT_TERNARY ? 16 : 8; }

// encode(w, gs, fmt): (packed, scales)
PyObject* encode(PyObject*, PyObject* const* argv, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    expect(n, 3, "encode");
    const Args a{argv, n};
    if (!plain_state() || !plain(argv[0])) Py_RETURN_NONE;
    const Tensor& w = a.t(0);
    const int64_t gs = a.i64(1);
    const int fmt = (int)a.i64(2), dt = dtype_code(w.scalar_type());
    if (dt < 0 || fmt < 0 || fmt > 2 || gs <= 0 || gs % pack_unit(fmt) != 0 ||
        (c10::GradMode::is_enabled() && records(w)))
        Py_RETURN_NONE;
    RECORD_FUNCTION("ojasx_e8t::encode", std::vector<c10::IValue>());
    Unlocked unlocked;
    const c10::DeviceGuard on_device(w.device());
    const Tensor wc = w.contiguous();
    const int64_t padded = padded_to(wc.numel(), gs);
    Tensor packed = at::empty({code_bytes(fmt, padded)}, w.options().dtype(at::kByte));
    Tensor scales = at::empty({padded / gs}, w.options().dtype(at::kHalf));
    check(kEncode[fmt](data(wc), dt, wc.numel(), gs, (uint8_t*)data(packed),
                       (uint16_t*)data(scales), current_stream(w.device())),
          "encode");
    unlocked.lock();
    PyObject* out = PyTuple_New(2);
    if (!out) throw python_error();
    PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(std::move(packed)));
    PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(std::move(scales)));
    return out;
    END_HANDLE_TH_ERRORS
}

// decode(packed, scales, numel, gs, dtype, fmt): flat weights, dtype a code of the C ABI
PyObject* decode(PyObject*, PyObject* const* argv, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    expect(n, 6, "decode");
    const Args a{argv, n};
    if (!plain_state() || !plain(argv[0]) || !plain(argv[1])) Py_RETURN_NONE;
    const Tensor &packed = a.t(0), &scales = a.t(1);
    const int64_t numel = a.i64(2), gs = a.i64(3);
    const int dt = (int)a.i64(4), fmt = (int)a.i64(5);
    if (dt < 0 || dt > 2 || fmt < 0 || fmt > 2 || gs <= 0 || gs % pack_unit(fmt) != 0 ||
        numel < 0 || packed.scalar_type() != at::kByte || scales.scalar_type() != at::kHalf ||
        !packed.is_contiguous() || !scales.is_contiguous() ||
        packed.device() != scales.device() ||
        packed.numel() < code_bytes(fmt, padded_to(numel, gs)) ||
        scales.numel() < padded_to(numel, gs) / gs ||
        (c10::GradMode::is_enabled() && records(scales)))
        Py_RETURN_NONE;
    RECORD_FUNCTION("ojasx_e8t::decode", std::vector<c10::IValue>());
    Unlocked unlocked;
    const c10::DeviceGuard on_device(packed.device());
    const at::ScalarType types[] = {at::kFloat, at::kHalf, at::kBFloat16};
    Tensor out = at::empty({numel}, packed.options().dtype(types[dt]));
    check(kDecode[fmt]((const uint8_t*)data(packed), (const uint16_t*)data(scales), numel, gs, dt,
                       data(out), current_stream(packed.device())),
          "decode");
    unlocked.lock();
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// plain(tensor, ...): whether a Function over these tensors is plain eager work (grad aside)
PyObject* is_plain(PyObject*, PyObject* const* argv, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (!plain_state()) Py_RETURN_FALSE;
    for (Py_ssize_t i = 0; i < n; ++i)
        if (argv[i] != Py_None && !plain(argv[i])) Py_RETURN_FALSE;
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {
    {"linear", (PyCFunction)(void*)linear, METH_FASTCALL, nullptr},
    {"linear_bwd", (PyCFunction)(void*)linear_bwd, METH_FASTCALL, nullptr},
    {"linear_lora", (PyCFunction)(void*)linear_lora, METH_FASTCALL, nullptr},
    {"linear_lora_bwd", (PyCFunction)(void*)linear_lora_bwd, METH_FASTCALL, nullptr},
    {"encode", (PyCFunction)(void*)encode, METH_FASTCALL, nullptr},
    {"decode", (PyCFunction)(void*)decode, METH_FASTCALL, nullptr},
    {"is_plain", (PyCFunction)(void*)is_plain, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_ojasx_eager", nullptr, -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__ojasx_eager(void) { return PyModule_Create(&kModule); }
