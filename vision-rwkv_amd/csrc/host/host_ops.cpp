// RUN_CUDA, RUN_CUDA_RWKV6 and a block's native call without the interpreter: argument checks, allocations and autograd nodes in C++
// around the entry points of libvrwkv_hip.so (include/vrwkv_hip.h).
//
// What it saves is host time beside short kernels: through autograd.Function and ctypes a forward costs the host 14 us and a backward
// 60, since the engine's thread takes the interpreter's lock, allocates and marshals there.  Python classes -> here, us per call, results
// bit for bit the same:
//   Bi-WKV forward, 1 x 196 x 192 fp32 (kernel 5.6)             14.6 -> 6.3
//   Bi-WKV training, 64 x 196 x 768 bf16 (kernels 56)           119.6 -> 76.1        2 x 4150 x 768 fp32 (kernels 120)   128 -> 120
//   wkv6 training, 8 x 577 x 384 fp32 (kernels 115)             159 -> 116
//   twelve native blocks, 1 x 196 x 192 bf16 (kernels 397)      602 -> 507
//
// The operators take the plain case: exact tensors and parameters, contiguous, on the current GPU, of the types that the kernels read as
// they lie, outside every transform, mode and trace.  To everything else they answer None, and the Python classes in ops.py go on as
// before: converting, refusing, tracing.
#include <cstddef>
#include <string_view>
#include <unordered_map>
#include <torch/extension.h>
#include <torch/version.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include "../../../include/vrwkv_hip.h"

namespace {
using torch::autograd::AutogradContext;
using torch::autograd::tensor_list;
using torch::autograd::Variable;

int code(at::ScalarType t) { return t == at::kFloat ? VRWKV_F32 : t == at::kBFloat16 ? VRWKV_BF16 : t == at::kHalf ? VRWKV_F16 : -1; }

void* stream_of(const at::Tensor& t) { return (void*)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.get_device()).stream(); }

using Guard = c10::hip::HIPGuardMasqueradingAsCUDA;

// Tracing, functorch levels, dispatch and function modes are to see the operators' Python classes.
bool transformed() {
    return torch::jit::tracer::isTracing() || c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) || c10::impl::TorchDispatchModeTLS::any_modes_set() ||
           at::impl::PythonTorchFunctionTLS::stack_len() > 0;
}

// An exact Tensor or Parameter with memory of its own, dense, contiguous, on a GPU.
bool plain(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return false;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage() || !t.is_contiguous() || t.is_conj() || t.is_neg()) return false;
    const auto keys = t.key_set();
    return !keys.has(c10::DispatchKey::FuncTorchBatched) && !keys.has(c10::DispatchKey::Batched) && !keys.has(c10::DispatchKey::Python) &&
           !keys.has(c10::DispatchKey::FuncTorchGradWrapper) && !keys.has(c10::DispatchKey::Functionalize) && code(t.scalar_type()) >= 0;
}

// The entry points take dimensions as int, the Bi-WKV backward 65535 sequences.
bool fits(const at::Tensor& t) { return t.size(0) <= 65535 && t.size(1) <= INT_MAX && t.size(2) <= INT_MAX; }

// Forward-mode tangents are refused by the Python classes.
bool tangent(const at::Tensor& t) { return t._fw_grad(0).defined(); }

// A tensor that a hook on saved tensors, or the engine, hands to a backward.
at::Tensor dense(const at::Tensor& t, const at::Tensor& like) {
    TORCH_CHECK(t.defined() && t.has_storage() && t.is_cuda() && t.device() == like.device() && code(t.scalar_type()) >= 0,
                "the saved tensors and the gradient must be CUDA tensors on one device");
    return t.contiguous();
}

at::Tensor bytes(size_t n, const at::Tensor& like) { return at::empty({(int64_t)n}, like.options().dtype(at::kByte).requires_grad(false)); }

// ---- Bi-WKV --------------------------------------------------------------------------------------------------------------
// y, or an undefined tensor where the entry point refuses the call
at::Tensor wkv_forward(const at::Tensor& w, const at::Tensor& u, const at::Tensor& k, const at::Tensor& v, float factor) {
    const int B = (int)k.size(0), T = (int)k.size(1), C = (int)k.size(2), dt = code(k.scalar_type());
    Guard guard(k.device());
    at::Tensor y = at::empty_like(k), ws;
    const size_t n = vrwkv_biwkv_fwd_workspace_bytes(B, T, C, dt);
    if (n) ws = bytes(n, k);
    const int rc = vrwkv_biwkv_fwd_as(w.data_ptr(), u.data_ptr(), code(w.scalar_type()), factor, k.data_ptr(), v.data_ptr(), y.data_ptr(), B, T, C, dt,
                                      n ? ws.data_ptr() : nullptr, n, stream_of(k));
    return rc == VRWKV_OK ? y : at::Tensor();
}

struct Wkv : torch::autograd::Function<Wkv> {
    static Variable forward(AutogradContext* ctx, const Variable& w, const Variable& u, const Variable& k, const Variable& v, double factor, const at::Tensor* y) {
        ctx->save_for_backward({w, u, k, v});
        ctx->saved_data["factor"] = factor;
        return *y;
    }
    static tensor_list backward(AutogradContext* ctx, tensor_list grads) {
        at::NoGradGuard no_grad;
        const auto saved = ctx->get_saved_variables();
        const at::Tensor k = dense(saved[2], saved[2]), v = dense(saved[3], k), w = dense(saved[0], k), u = dense(saved[1], k);
        const at::Tensor gy = dense(grads[0].to(k.scalar_type()), k);
        TORCH_CHECK(k.dim() == 3 && v.sizes() == k.sizes() && gy.sizes() == k.sizes() && w.numel() == k.size(2) && u.numel() == k.size(2) &&
                        v.scalar_type() == k.scalar_type() && u.scalar_type() == w.scalar_type(),
                    "k, v and gy must all be (B,T,C)");
        const int B = (int)k.size(0), T = (int)k.size(1), C = (int)k.size(2), dt = code(k.scalar_type());
        Guard guard(k.device());
        at::Tensor gw = at::empty_like(w), gu = at::empty_like(u), gk = at::empty_like(k), gv = at::empty_like(v);
        const size_t n = vrwkv_biwkv_bwd_workspace_bytes(B, T, C, dt);
        at::Tensor ws = bytes(n, k);
        const int rc = vrwkv_biwkv_bwd_as(w.data_ptr(), u.data_ptr(), code(w.scalar_type()), (float)ctx->saved_data["factor"].toDouble(), k.data_ptr(),
                                          v.data_ptr(), gy.data_ptr(), gw.data_ptr(), gu.data_ptr(), gk.data_ptr(), gv.data_ptr(), B, T, C, dt,
                                          ws.data_ptr(), n, stream_of(k));
        TORCH_CHECK(rc == VRWKV_OK, "vrwkv status ", rc, ": ", vrwkv_last_error());
        return {gw, gu, gk, gv, Variable(), Variable()};
    }
};

// RUN_CUDA(w * factor, u * factor, k, v), the product in the parameters' type; None where the Python class has to decide.
py::object wkv(py::handle w_, py::handle u_, py::handle k_, py::handle v_, double factor) {
    if (transformed() || !plain(w_.ptr()) || !plain(u_.ptr()) || !plain(k_.ptr()) || !plain(v_.ptr())) return py::none();
    const at::Tensor &w = THPVariable_Unpack(w_.ptr()), &u = THPVariable_Unpack(u_.ptr()), &k = THPVariable_Unpack(k_.ptr()), &v = THPVariable_Unpack(v_.ptr());
    const auto dt = k.scalar_type();
    if (k.dim() != 3 || k.numel() == 0 || v.sizes() != k.sizes() || v.scalar_type() != dt || w.scalar_type() != dt || u.scalar_type() != dt ||
        w.numel() != k.size(2) || u.numel() != k.size(2) || w.device() != k.device() || u.device() != k.device() || v.device() != k.device() ||
        k.get_device() != c10::hip::current_device() || !fits(k) || tangent(w) || tangent(u) || tangent(k) || tangent(v))
        return py::none();
    at::Tensor y;
    {
        py::gil_scoped_release release;
        y = wkv_forward(w, u, k, v, (float)factor);
        if (y.defined() && at::GradMode::is_enabled() && (w.requires_grad() || u.requires_grad() || k.requires_grad() || v.requires_grad()))
            y = Wkv::apply(w, u, k, v, factor, &y);
    }
    if (!y.defined()) return py::none();
    return py::reinterpret_steal<py::object>(THPVariable_Wrap(y));
}

// ---- wkv6 ----------------------------------------------------------------------------------------------------------------
at::Tensor wkv6_forward(const at::Tensor& r, const at::Tensor& k, const at::Tensor& v, const at::Tensor& w, const at::Tensor& u, int H, bool whole) {
    const int B = (int)r.size(0), T = (int)r.size(1), C = (int)r.size(2);
    Guard guard(r.device());
    at::Tensor y = at::empty_like(r, r.options().dtype(at::kFloat)), ws;
    if (whole) {
        const int rc = vrwkv_wkv6_fwd_whole(r.data_ptr(), k.data_ptr(), v.data_ptr(), w.data_ptr(), (const float*)u.data_ptr(), (float*)y.data_ptr(),
                                            B, T, C, H, code(r.scalar_type()), code(w.scalar_type()), 0, stream_of(r));
        return rc == VRWKV_OK ? y : at::Tensor();
    }
    const size_t n = vrwkv_wkv6_fwd_workspace_bytes(B, T, C, H);
    if (n) ws = bytes(n, r);
    const int rc = vrwkv_wkv6_fwd(r.data_ptr(), k.data_ptr(), v.data_ptr(), w.data_ptr(), (const float*)u.data_ptr(), (float*)y.data_ptr(), B, T, C, H,
                                  code(r.scalar_type()), code(w.scalar_type()), 0, n ? ws.data_ptr() : nullptr, n, stream_of(r));
    return rc == VRWKV_OK ? y : at::Tensor();
}

struct Wkv6 : torch::autograd::Function<Wkv6> {
    static Variable forward(AutogradContext* ctx, const Variable& r, const Variable& k, const Variable& v, const Variable& w, const Variable& u, int64_t H, const at::Tensor* y) {
        ctx->save_for_backward({r, k, v, w, u});
        ctx->saved_data["H"] = H;
        return *y;
    }
    static tensor_list backward(AutogradContext* ctx, tensor_list grads) {
        at::NoGradGuard no_grad;
        const auto saved = ctx->get_saved_variables();
        const at::Tensor r = dense(saved[0], saved[0]), k = dense(saved[1], r), v = dense(saved[2], r), w = dense(saved[3], r), u = dense(saved[4], r);
        if (!grads[0].is_contiguous()) {                                                       // an AssertionError, as the Python class raises
            py::gil_scoped_acquire gil;
            PyErr_SetNone(PyExc_AssertionError);
            python_error e;
            e.persist();
            throw std::move(e);
        }
        const at::Tensor gy = dense(grads[0].to(at::kFloat), r);
        const int B = (int)r.size(0), T = (int)r.size(1), C = (int)r.size(2), H = (int)ctx->saved_data["H"].toInt();
        TORCH_CHECK(k.sizes() == r.sizes() && v.sizes() == r.sizes() && w.sizes() == r.sizes() && gy.sizes() == r.sizes() && u.numel() == C &&
                        k.scalar_type() == r.scalar_type() && v.scalar_type() == r.scalar_type() && u.scalar_type() == at::kFloat,
                    "r, k, v, w, gy must all be (B,T,C)");
        Guard guard(r.device());
        at::Tensor gr = at::empty_like(r), gk = at::empty_like(k), gv = at::empty_like(v), gw = at::empty_like(w);
        at::Tensor gu = at::empty({H, C / H}, u.options().requires_grad(false));
        const int dt = code(r.scalar_type()), wt = code(w.scalar_type());
        const size_t n = vrwkv_wkv6_bwd_like_workspace_bytes(B, T, C, H, dt, wt);
        at::Tensor ws = bytes(n, r);
        const int rc = vrwkv_wkv6_bwd_like(r.data_ptr(), k.data_ptr(), v.data_ptr(), w.data_ptr(), (const float*)u.data_ptr(), (const float*)gy.data_ptr(), gr.data_ptr(),
                                           gk.data_ptr(), gv.data_ptr(), gw.data_ptr(), (float*)gu.data_ptr(), B, T, C, H, dt, wt, 0, ws.data_ptr(), n, stream_of(r));
        TORCH_CHECK(rc == VRWKV_OK, "vrwkv status ", rc, ": ", vrwkv_last_error());
        return {gr, gk, gv, gw, gu, Variable(), Variable()};
    }
};

// RUN_CUDA_RWKV6; whole: what WKV_6.stays_whole says of the call, which holds where autograd records.
py::object wkv6(int64_t B, int64_t T, int64_t C, int64_t H, py::handle r_, py::handle k_, py::handle v_, py::handle w_, py::handle u_, bool whole) {
    if (transformed() || !plain(r_.ptr()) || !plain(k_.ptr()) || !plain(v_.ptr()) || !plain(w_.ptr()) || !plain(u_.ptr())) return py::none();
    const at::Tensor &r = THPVariable_Unpack(r_.ptr()), &k = THPVariable_Unpack(k_.ptr()), &v = THPVariable_Unpack(v_.ptr()), &w = THPVariable_Unpack(w_.ptr()),
                     &u = THPVariable_Unpack(u_.ptr());
    const auto dt = r.scalar_type();
    if (H <= 0 || C != 64 * H || r.dim() != 3 || r.size(0) != B || r.size(1) != T || r.size(2) != C || r.numel() == 0 || k.sizes() != r.sizes() ||
        v.sizes() != r.sizes() || w.sizes() != r.sizes() || k.scalar_type() != dt || v.scalar_type() != dt || (w.scalar_type() != dt && w.scalar_type() != at::kFloat) ||
        u.scalar_type() != at::kFloat || u.dim() != 2 || u.size(0) != H || u.size(1) != 64 || k.device() != r.device() || v.device() != r.device() ||
        w.device() != r.device() || u.device() != r.device() || !fits(r) || tangent(r) || tangent(k) || tangent(v) || tangent(w) || tangent(u))
        return py::none();
    at::Tensor y;
    {
        py::gil_scoped_release release;
        const bool record = at::GradMode::is_enabled() && (r.requires_grad() || k.requires_grad() || v.requires_grad() || w.requires_grad() || u.requires_grad());
        y = wkv6_forward(r, k, v, w, u, (int)H, whole && record);
        if (y.defined() && record) y = Wkv6::apply(r, k, v, w, u, H, &y);
    }
    if (!y.defined()) return py::none();
    return py::reinterpret_steal<py::object>(THPVariable_Wrap(y));
}
// ---- blocks --------------------------------------------------------------------------------------------------------------
#define POINTER(n) {#n, offsetof(vrwkv_block_args, n)}
const std::unordered_map<std::string_view, size_t> block_pointers = {
    POINTER(ln1_w), POINTER(ln1_b), POINTER(ln2_w), POINTER(ln2_b), POINTER(gamma1), POINTER(gamma2), POINTER(att_mix), POINTER(ffn_mix), POINTER(w),
    POINTER(u), POINTER(key), POINTER(value), POINTER(receptance), POINTER(output), POINTER(att_kn_w), POINTER(att_kn_b), POINTER(ffn_key),
    POINTER(ffn_receptance), POINTER(ffn_value), POINTER(ffn_kn_w), POINTER(ffn_kn_b), POINTER(gate), POINTER(maa), POINTER(maa_w1), POINTER(maa_w2),
    POINTER(decay), POINTER(decay_w1), POINTER(decay_w2), POINTER(gn_w), POINTER(gn_b)};
const std::unordered_map<std::string_view, size_t> block_ints = {POINTER(hidden), POINTER(heads), POINTER(Hp), POINTER(Wp), POINTER(shift_pixel),
                                                                 POINTER(quarter), POINTER(post_norm)};
const std::unordered_map<std::string_view, size_t> block_floats = {POINTER(ln1_eps), POINTER(ln2_eps), POINTER(att_kn_eps), POINTER(ffn_kn_eps), POINTER(gn_eps)};
#undef POINTER
#define POINTER(n) {#n, offsetof(vrwkv_block6_params, n)}
const std::unordered_map<std::string_view, size_t> block6_pointers = {
    POINTER(maa_w1), POINTER(maa_w2), POINTER(decay_w1), POINTER(decay_w2), POINTER(maa_x), {"maa_w", offsetof(vrwkv_block6_params, maa)},
    {"maa_k", offsetof(vrwkv_block6_params, maa) + sizeof(void*)}, {"maa_v", offsetof(vrwkv_block6_params, maa) + 2 * sizeof(void*)},
    {"maa_r", offsetof(vrwkv_block6_params, maa) + 3 * sizeof(void*)}, {"maa_g", offsetof(vrwkv_block6_params, maa) + 4 * sizeof(void*)},
    POINTER(ffn_mix_k), POINTER(ffn_mix_r), POINTER(u), POINTER(att_kn_w), POINTER(att_kn_b)};
#undef POINTER

std::string_view text(PyObject* key) {
    Py_ssize_t n = 0;
    const char* s = PyUnicode_AsUTF8AndSize(key, &n);
    if (!s) throw py::error_already_set();
    return {s, (size_t)n};
}

const at::Tensor& tensor(PyObject* o) {
    TORCH_CHECK_TYPE(THPVariable_Check(o), "the block's weights must be tensors");
    return THPVariable_Unpack(o);
}

// block_weights_fit of ops.py
bool weights_fit(py::handle x_, py::iterable weights) {
    const at::Tensor& x = tensor(x_.ptr());
    for (py::handle p : weights) {
        if ((PyObject*)Py_TYPE(p.ptr()) != ParameterClass) return false;
        const at::Tensor& t = THPVariable_Unpack(p.ptr());
        if (t.scalar_type() != x.scalar_type() || t.get_device() != x.get_device() || !t.is_contiguous()) return false;
    }
    return true;
}

// block_forward of ops.py: the result, None where a pointer is not 16-byte aligned, or the status of a call that was refused
py::object block_forward(py::handle x_, py::dict tensors, py::object params, py::dict scalars) {
    const at::Tensor& x = tensor(x_.ptr());
    TORCH_CHECK(x.dim() == 3 && x.is_cuda() && code(x.scalar_type()) >= 0, "x must be a (B,T,C) CUDA tensor of float32 / bfloat16 / float16");
    vrwkv_block_args a = {};
    char* at_args = (char*)&a;
    uintptr_t bits = 0;
    PyObject *key, *value;
    for (Py_ssize_t i = 0; PyDict_Next(tensors.ptr(), &i, &key, &value);) {
        void* p = tensor(value).data_ptr();
        bits |= (uintptr_t)p;
        *(void**)(at_args + block_pointers.at(text(key))) = p;
    }
    for (Py_ssize_t i = 0; PyDict_Next(scalars.ptr(), &i, &key, &value);) {
        const auto name = text(key);
        if (auto f = block_floats.find(name); f != block_floats.end()) {
            *(float*)(at_args + f->second) = (float)PyFloat_AsDouble(value);
        } else {
            *(int*)(at_args + block_ints.at(name)) = (int)PyLong_AsLong(value);
        }
        if (PyErr_Occurred()) throw py::error_already_set();
    }
    vrwkv_block6_params six = {};
    if (!params.is_none()) {
        static const char* const vectors[] = {"maa_x", "maa_w", "maa_k", "maa_v", "maa_r", "maa_g", "ffn_mix_k", "ffn_mix_r", "u"};
        for (Py_ssize_t i = 0; PyDict_Next(params.ptr(), &i, &key, &value);) {
            const at::Tensor& t = tensor(value);
            const auto name = text(key);
            *(void**)((char*)&six + block6_pointers.at(name)) = t.data_ptr();
            if (t.scalar_type() == at::kFloat)
                for (int v = 0; v < 9; ++v)
                    if (name == vectors[v]) six.fp32_vectors |= 1 << v;
        }
    }
    Guard guard(x.device());
    at::Tensor out = at::empty_like(x);
    a.x = x.data_ptr(), a.out = out.data_ptr();
    if ((bits | (uintptr_t)a.x | (uintptr_t)a.out) & 15) return py::none();
    a.B = (int)x.size(0), a.T = (int)x.size(1), a.C = (int)x.size(2), a.dtype = code(x.scalar_type());
    a.workspace_bytes = vrwkv_block_fwd_workspace_bytes(a.B, a.T, a.C, a.hidden, a.heads, a.dtype);
    at::Tensor ws = bytes(a.workspace_bytes, x);
    a.workspace = ws.data_ptr();
    void* st = stream_of(x);
    int rc;
    {
        py::gil_scoped_release release;
        rc = params.is_none() ? vrwkv_block_fwd(&a, st) : vrwkv_block6_fwd(&a, &six, st);
    }
    if (rc != VRWKV_OK) return py::int_(rc);
    return py::reinterpret_steal<py::object>(THPVariable_Wrap(out));
}
}  // namespace

PYBIND11_MODULE(_host, m) {
    m.attr("torch_version") = TORCH_VERSION;               // what the module's calls into torch were compiled against
    m.def("weights_fit", &weights_fit);
    m.def("block_forward", &block_forward);
    m.def("wkv", &wkv);
    m.def("wkv6", &wkv6);
}
