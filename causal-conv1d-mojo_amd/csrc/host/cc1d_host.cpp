// cc1d_host.cpp -- the package's per-call host path in native code: argument
// checks, output allocation, the autograd node and the launch through the C
// ABI (include/cc1d.h), as a CPython extension module over libtorch.
//
// Why: the GPU work of a call takes 2 to 80 us at common sizes, and the same
// steps in Python took longer -- 13 us for a decode update, 25 for a forward,
// 85 to 200 for a training step, most of it in the backward, whose Python
// runs on the autograd engine's thread and waits for the interpreter lock
// there. Here a backward is a C++ node that needs no interpreter.
//
// Each entry takes the ordinary case only: plain strided GPU tensors, valid
// arguments, no tracing, mode, transform or forward-mode level in force.
// For anything else it returns NotImplemented and the caller's Python code
// runs, which raises the errors and goes through the torch.library ops that
// torch.compile, fake tensors, vmap, dispatch modes and the like see. The
// backward asks again when it runs and goes through the same op if need be.
// The interpreter lock is given up while a call allocates and launches: a
// launch waits when the stream's queue is full, and other threads run on.
// Nothing is kept from one call for the next.
#include <Python.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/record_function.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>

#include <optional>

#include "cc1d.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;
using torch::autograd::variable_list;

// entry points of the loaded library (set once by bind())
struct Api {
    decltype(&cc1d_strerror) strerror = nullptr;
    decltype(&cc1d_fwd) fwd = nullptr;
    decltype(&cc1d_bwd_workspace_floats) workspace = nullptr;
    decltype(&cc1d_bwd_typed) bwd = nullptr;
    decltype(&cc1d_update) update = nullptr;
    decltype(&cc1d_varlen_states) varlen = nullptr;
} api;

void check(int status) {
    TORCH_CHECK_WITH(Error, status == CC1D_OK, "causal_conv1d_amd native call failed: ", api.strerror(status),
                     " (status ", status, ")");
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// No dispatch or torch-function mode, transform or tracer in force on this
// thread: what the dispatcher would send straight to the backend.
bool plain_thread() {
    if (c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled()) return false;
    const auto tls = c10::impl::tls_local_dispatch_key_set();
    return (tls.included_ - c10::default_included_set - c10::autocast_dispatch_keyset).empty();
}

// A strided GPU tensor without a subclass, lazy bit, wrapper or tangent.
bool plain(const Tensor& t) {
    static const auto allowed = c10::DispatchKeySet(c10::DispatchKey::CUDA) |
                                c10::DispatchKeySet(c10::DispatchKey::AutogradCUDA) |
                                c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView) |
                                c10::DispatchKeySet(c10::DispatchKey::AutocastCUDA);
    return t.defined() && t.is_cuda() && t.layout() == at::kStrided &&
           (t.key_set().raw_repr() & ~allowed.raw_repr()) == 0 && !t._fw_grad(0).defined();
}

bool plain(PyObject* o) { return THPVariable_CheckExact(o) && plain(THPVariable_Unpack(o)); }
bool plain_or_none(PyObject* o) { return o == Py_None || plain(o); }
Tensor tensor_or_none(PyObject* o) { return o == Py_None ? Tensor() : THPVariable_Unpack(o); }

int dtype_code(const Tensor& t) {
    switch (t.scalar_type()) {
    case at::kHalf: return CC1D_DTYPE_FP16;
    case at::kBFloat16: return CC1D_DTYPE_BF16;
    case at::kFloat: return CC1D_DTYPE_FP32;
    default: return -1;
    }
}

// 0: no activation, 1: SiLU, -1: not one of the accepted values
int activation_code(PyObject* o) {
    if (o == Py_None) return 0;
    if (!PyUnicode_CheckExact(o)) return -1;
    return PyUnicode_CompareWithASCIIString(o, "silu") == 0 || PyUnicode_CompareWithASCIIString(o, "swish") == 0 ? 1 : -1;
}

bool same(const Tensor& t, const Tensor& like) {
    return t.scalar_type() == like.scalar_type() && t.device() == like.device();
}
bool shaped(const Tensor& t, at::IntArrayRef s) { return t.sizes() == s; }

const void* ptr(const Tensor& t) { return t.defined() ? t.const_data_ptr() : nullptr; }
void* out_ptr(const Tensor& t) { return t.defined() ? t.mutable_data_ptr() : nullptr; }

template <int N> void strides(int64_t (&dst)[N], const Tensor& t) {
    for (int i = 0; i < N; ++i) dst[i] = t.defined() ? t.stride(i) : 0;
}

// ---- forward / backward ------------------------------------------------

void launch_fwd(const Tensor& x, const Tensor& weight, const Tensor& bias, const Tensor& seq_idx, const Tensor& init,
                const Tensor& out, const Tensor& final_states, bool silu) {
    RECORD_FUNCTION("causal_conv1d_amd::_fwd_inplace", c10::ArrayRef<const c10::IValue>{});
    cc1d_fwd_params p{};
    p.x = ptr(x);
    p.weight = ptr(weight);
    p.bias = ptr(bias);
    p.seq_idx = static_cast<const int32_t*>(ptr(seq_idx));
    p.initial_states = ptr(init);
    p.out = out_ptr(out);
    p.final_states_out = out_ptr(final_states);
    p.batch = x.size(0);
    p.dim = x.size(1);
    p.seqlen = x.size(2);
    p.width = weight.size(1);
    strides(p.x_stride, x);
    strides(p.weight_stride, weight);
    p.bias_stride = bias.defined() ? bias.stride(0) : 0;
    strides(p.seq_idx_stride, seq_idx);
    strides(p.initial_states_stride, init);
    strides(p.out_stride, out);
    strides(p.final_states_stride, final_states);
    p.dtype = dtype_code(x);
    p.apply_silu = silu;
    check(api.fwd(&p, stream_of(x)));
}

void launch_bwd(const Tensor& x, const Tensor& weight, const Tensor& bias, const Tensor& dout, const Tensor& seq_idx,
                const Tensor& init, const Tensor& dfinal, const Tensor& dx, const Tensor& dweight, const Tensor& dbias,
                const Tensor& dinit, bool silu) {
    RECORD_FUNCTION("causal_conv1d_amd::_bwd_typed_inplace", c10::ArrayRef<const c10::IValue>{});
    cc1d_bwd_params p{};
    p.x = ptr(x);
    p.weight = ptr(weight);
    p.bias = ptr(bias);
    p.dout = ptr(dout);
    p.seq_idx = static_cast<const int32_t*>(ptr(seq_idx));
    p.initial_states = ptr(init);
    p.dfinal_states = ptr(dfinal);
    p.dx = out_ptr(dx);
    p.dinitial_states = out_ptr(dinit);
    p.batch = x.size(0);
    p.dim = x.size(1);
    p.seqlen = x.size(2);
    p.width = weight.size(1);
    strides(p.x_stride, x);
    strides(p.weight_stride, weight);
    p.bias_stride = bias.defined() ? bias.stride(0) : 0;
    strides(p.dout_stride, dout);
    strides(p.seq_idx_stride, seq_idx);
    strides(p.initial_states_stride, init);
    strides(p.dfinal_states_stride, dfinal);
    strides(p.dx_stride, dx);
    strides(p.dinitial_states_stride, dinit);
    p.dtype = dtype_code(x);
    p.apply_silu = silu;
    // per-call partial sums, from the allocator's pool of the current stream
    const int64_t n = api.workspace(&p);
    const Tensor ws = at::empty({n > 1 ? n : 1}, x.options().dtype(at::kFloat));
    cc1d_bwd_grads g{};
    g.dweight = out_ptr(dweight);
    g.dbias = out_ptr(dbias);
    strides(g.dweight_stride, dweight);
    g.dbias_stride = dbias.defined() ? dbias.stride(0) : 0;
    g.workspace = ws.data_ptr<float>();
    g.workspace_floats = ws.numel();
    check(api.bwd(&p, &g, stream_of(x)));
}

// dout in x's layout: a copy only where the time strides differ (or any, in a layout without unit time stride)
Tensor match_layout(const Tensor& t, const Tensor& like) {
    if (t.strides() == like.strides()) return t;
    if (like.stride(-1) == 1) return t.stride(-1) == 1 ? t : t.contiguous();
    return at::empty_like(like).copy_(t);
}

struct Conv1dFn : public torch::autograd::Function<Conv1dFn> {
    // backward() depends on its arguments and on what ctx saved alone
    static constexpr bool is_traceable = true;

    static variable_list forward(torch::autograd::AutogradContext* ctx, const Tensor& x, const Tensor& weight,
                                 const OptTensor& bias, const OptTensor& seq_idx, const OptTensor& init,
                                 bool silu, bool final_states) {
        const Tensor none;
        const Tensor out = at::empty_like(x);
        const Tensor fs = final_states ? at::empty({x.size(0), x.size(1), weight.size(1) - 1}, x.options()) : none;
        launch_fwd(x, weight, bias.value_or(none), seq_idx.value_or(none), init.value_or(none), out, fs, silu);
        ctx->save_for_backward({x, weight, bias.value_or(none), seq_idx.value_or(none), init.value_or(none)});
        ctx->saved_data["silu"] = silu;
        if (final_states) return {out, fs};
        return {out};
    }

    static variable_list backward(torch::autograd::AutogradContext* ctx, const variable_list& grads) {
        const auto saved = ctx->get_saved_variables();
        const Tensor &x = saved[0], &weight = saved[1], &bias = saved[2], &seq_idx = saved[3], &init = saved[4];
        const bool silu = ctx->saved_data["silu"].toBool();
        const c10::OptionalDeviceGuard device(x.device());
        Tensor dfinal = grads.size() > 1 ? grads[1] : Tensor();
        if (dfinal.defined() && dfinal.scalar_type() != x.scalar_type()) dfinal = dfinal.to(x.scalar_type());
        const Tensor dout = match_layout(grads[0], x);
        const Tensor dx = at::empty_like(x);
        // fp32 sums rounded once to the parameter dtype
        const Tensor dweight = at::empty(weight.sizes(), weight.options());
        const Tensor dbias = bias.defined() ? at::empty(bias.sizes(), bias.options()) : Tensor();
        const Tensor dinit = init.defined() ? at::empty_like(init) : Tensor();
        bool direct = plain_thread() && !at::GradMode::is_enabled();
        for (const Tensor& t : {x, weight, dout}) direct = direct && plain(t);
        for (const Tensor& t : {bias, seq_idx, init, dfinal}) direct = direct && (!t.defined() || plain(t));
        if (direct) {
            launch_bwd(x, weight, bias, dout, seq_idx, init, dfinal, dx, dweight, dbias, dinit, silu);
        } else {  // through the op: create_graph, modes, transforms, compiled autograd
            const auto op = c10::Dispatcher::singleton().findSchemaOrThrow("causal_conv1d_amd::_bwd_typed_inplace", "");
            auto opt = [](const Tensor& t) { return t.defined() ? c10::IValue(t) : c10::IValue(); };
            torch::jit::Stack stack{x, weight, opt(bias), dout, opt(seq_idx), opt(init), opt(dfinal), dx, dweight,
                                    opt(dbias), opt(dinit), silu};
            op.callBoxed(&stack);
        }
        return {dx, dweight, dbias, Tensor(), dinit, Tensor(), Tensor()};
    }
};

PyObject* not_implemented() { Py_RETURN_NOTIMPLEMENTED; }

// fn(x, weight, bias, seq_idx, initial_states, return_final_states, final_states_out, activation)
PyObject* py_fn(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(n == 8, "fn takes 8 arguments");
    const int act = activation_code(a[7]);
    if (act < 0 || !PyBool_Check(a[5]) || a[6] != Py_None || !plain(a[0]) || !plain(a[1]) || !plain_or_none(a[2]) ||
        !plain_or_none(a[3]) || !plain_or_none(a[4]) || !plain_thread())
        return not_implemented();
    const Tensor &x = THPVariable_Unpack(a[0]), &weight = THPVariable_Unpack(a[1]);
    const Tensor bias = tensor_or_none(a[2]), seq_idx = tensor_or_none(a[3]), init = tensor_or_none(a[4]);
    const bool final_states = a[5] == Py_True;
    const int dt = dtype_code(x);
    if (dt < 0 || x.dim() != 3 || weight.dim() != 2 || !same(weight, x) || x.numel() == 0) return not_implemented();
    const int64_t B = x.size(0), D = x.size(1), L = x.size(2), W = weight.size(1);
    if (W < 2 || W > (dt == CC1D_DTYPE_FP32 ? 5 : 9) || weight.size(0) != D) return not_implemented();
    if (bias.defined() && (!same(bias, x) || !shaped(bias, {D}))) return not_implemented();
    if (seq_idx.defined() &&
        (final_states || init.defined() || seq_idx.scalar_type() != at::kInt || seq_idx.device() != x.device() ||
         !shaped(seq_idx, {B, L}) || !seq_idx.is_contiguous()))
        return not_implemented();
    if (init.defined() && (!same(init, x) || !shaped(init, {B, D, W - 1}))) return not_implemented();

    std::optional<pybind11::gil_scoped_release> unlocked(std::in_place);
    const c10::OptionalDeviceGuard device(x.device());
    auto wants = [](const Tensor& t) { return t.defined() && t.requires_grad(); };
    Tensor out, fs;
    if (at::GradMode::is_enabled() && (wants(x) || wants(weight) || wants(bias) || wants(init))) {
        auto opt = [](const Tensor& t) { return t.defined() ? OptTensor(t) : OptTensor(); };
        const auto r = Conv1dFn::apply(x, weight, opt(bias), opt(seq_idx), opt(init), act == 1, final_states);
        out = r[0];
        if (final_states) fs = r[1];
    } else {
        out = at::empty_like(x);
        if (final_states) fs = at::empty({B, D, W - 1}, x.options());
        launch_fwd(x, weight, bias, seq_idx, init, out, fs, act == 1);
    }
    unlocked.reset();
    if (!final_states) return THPVariable_Wrap(std::move(out));
    PyObject* t = PyTuple_New(2);
    if (t == nullptr) throw python_error();
    PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(std::move(out)));
    PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(std::move(fs)));
    return t;
    END_HANDLE_TH_ERRORS
}

// update(x, conv_state, weight, bias, activation, cache_seqlens, conv_state_indices)
PyObject* py_update(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(n == 7, "update takes 7 arguments");
    const int act = activation_code(a[4]);
    if (act < 0 || !plain(a[0]) || !plain(a[1]) || !plain(a[2]) || !plain_or_none(a[3]) || !plain_or_none(a[5]) ||
        !plain_or_none(a[6]) || !plain_thread())
        return not_implemented();
    const Tensor &x = THPVariable_Unpack(a[0]), &state = THPVariable_Unpack(a[1]), &weight = THPVariable_Unpack(a[2]);
    const Tensor bias = tensor_or_none(a[3]), heads = tensor_or_none(a[5]), idx = tensor_or_none(a[6]);
    if (dtype_code(x) < 0 || (x.dim() != 2 && x.dim() != 3) || state.dim() != 3 || weight.dim() != 2 ||
        !same(weight, x) || !same(state, x) || x.numel() == 0)
        return not_implemented();
    const int64_t B = x.size(0), D = x.size(1), W = weight.size(1), S = state.size(2);
    if (W < 2 || W > 9 || weight.size(0) != D || S < W - 1) return not_implemented();
    if (bias.defined() && (!same(bias, x) || !shaped(bias, {D}))) return not_implemented();
    if (state.size(1) != D || (!idx.defined() && state.size(0) != B)) return not_implemented();
    for (const Tensor* t : {&heads, &idx})
        if (t->defined() && (t->scalar_type() != at::kInt || t->device() != x.device() || !shaped(*t, {B}) ||
                             !t->is_contiguous()))
            return not_implemented();

    std::optional<pybind11::gil_scoped_release> unlocked(std::in_place);
    const c10::OptionalDeviceGuard device(x.device());
    Tensor out;
    {
        const at::NoGradGuard no_grad;  // (an allocation and a launch: nothing to differentiate)
        out = at::empty_like(x);
    }
    cc1d_update_params p{};
    p.x = ptr(x);
    p.weight = ptr(weight);
    p.bias = ptr(bias);
    p.conv_state = out_ptr(state);
    p.conv_state_indices = static_cast<const int32_t*>(ptr(idx));
    p.cache_seqlens = static_cast<const int32_t*>(ptr(heads));
    p.out = out_ptr(out);
    p.batch = B;
    p.dim = D;
    p.seqlen = x.dim() == 3 ? x.size(2) : 1;
    p.width = W;
    p.state_len = S;
    p.state_rows = state.size(0);
    for (int i = 0; i < 3; ++i) {
        p.x_stride[i] = i < x.dim() ? x.stride(i) : 1;
        p.out_stride[i] = i < x.dim() ? out.stride(i) : 1;
    }
    strides(p.weight_stride, weight);
    p.bias_stride = bias.defined() ? bias.stride(0) : 0;
    strides(p.conv_state_stride, state);
    p.dtype = dtype_code(x);
    p.apply_silu = act;
    check(api.update(&p, stream_of(x)));
    unlocked.reset();
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// varlen_states(x, cu_seqlens, state_len)
PyObject* py_varlen_states(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(n == 3, "varlen_states takes 3 arguments");
    if (!plain(a[0]) || !plain(a[1]) || !PyLong_CheckExact(a[2]) || !plain_thread()) return not_implemented();
    const Tensor &x = THPVariable_Unpack(a[0]), &cu = THPVariable_Unpack(a[1]);
    int over = 0;
    const long long S = PyLong_AsLongLongAndOverflow(a[2], &over);
    const int64_t es = x.element_size();
    if (over != 0 || S < 0 || x.dim() != 2 || cu.dim() != 1 || cu.size(0) < 1 || cu.scalar_type() != at::kInt ||
        cu.device() != x.device() || !cu.is_contiguous() || (es != 1 && es != 2 && es != 4 && es != 8 && es != 16))
        return not_implemented();
    std::optional<pybind11::gil_scoped_release> unlocked(std::in_place);
    const c10::OptionalDeviceGuard device(x.device());
    Tensor states = at::empty({cu.size(0) - 1, S, x.size(1)}, x.options()).transpose(1, 2);
    cc1d_varlen_params p{};
    p.x = ptr(x);
    p.cu_seqlens = static_cast<const int32_t*>(ptr(cu));
    p.states = out_ptr(states);
    p.total_tokens = x.size(0);
    p.dim = x.size(1);
    p.batch = cu.size(0) - 1;
    p.state_len = S;
    strides(p.x_stride, x);
    strides(p.states_stride, states);
    p.dtype = 0;
    p.elem_bytes = (int32_t)es;  // a bit-for-bit copy of any element type
    check(api.varlen(&p, stream_of(x)));
    unlocked.reset();
    return THPVariable_Wrap(std::move(states));
    END_HANDLE_TH_ERRORS
}

// bind(addresses of strerror, fwd, bwd_workspace_floats, bwd_typed, update, varlen_states)
PyObject* py_bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(n == 6, "bind takes 6 addresses");
    void* f[6];
    for (int i = 0; i < 6; ++i) {
        f[i] = PyLong_AsVoidPtr(a[i]);
        if (PyErr_Occurred()) throw python_error();
        TORCH_CHECK(f[i] != nullptr, "a null address");
    }
    api.strerror = reinterpret_cast<decltype(api.strerror)>(f[0]);
    api.fwd = reinterpret_cast<decltype(api.fwd)>(f[1]);
    api.workspace = reinterpret_cast<decltype(api.workspace)>(f[2]);
    api.bwd = reinterpret_cast<decltype(api.bwd)>(f[3]);
    api.update = reinterpret_cast<decltype(api.update)>(f[4]);
    api.varlen = reinterpret_cast<decltype(api.varlen)>(f[5]);
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

#define CC1D_FAST(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL
PyMethodDef methods[] = {
    {"bind", CC1D_FAST(py_bind), "the library's entry points"},
    {"fn", CC1D_FAST(py_fn), "causal_conv1d_fn's ordinary case, or NotImplemented"},
    {"update", CC1D_FAST(py_update), "causal_conv1d_update's ordinary case, or NotImplemented"},
    {"varlen_states", CC1D_FAST(py_varlen_states), "causal_conv1d_varlen_states' ordinary case, or NotImplemented"},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "cc1d_host", "native host path of causal_conv1d_amd", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_cc1d_host(void) { return PyModule_Create(&module); }
