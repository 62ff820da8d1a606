// Native host path of the GPU ops: argument checks, output allocation, autograd nodes and the launches of
// libebr_attn.so (include/ebr_*.h) in C++, for calls on plain GPU tensors.
//
// The Python layer (ebr_amd/fused_attn/ops.py, rope_split.py, block.py, descent.py, linear.py) defines the ops, their
// fakes and their autograd Functions, and stays the path of every call this file does not take: tensor subclasses and
// fake tensors, torch.func transforms, dispatch and function modes, tracing, forward-mode duals, saved-tensor hooks,
// tensors off the GPU, and every argument the Python layer would refuse or pad. Each entry point below returns None for
// those, and the caller goes on in Python. A node asks again when it runs: a backward under a transform (batched
// gradients), a mode, a tracer or hooks, or with cotangents of another kind, takes the Python formulas of its gradient
// (python_grads).
//
// Why it exists: a graded attention step (three launches) spent 453 us on the host in Python (autograd Functions,
// custom-op dispatch, ctypes marshalling, GIL hand-overs to the engine's threads) against 45 us of kernel time for one
// board and 310 us for the 768-board batch. The same nodes without Python take 140 us, of which two empty trips through
// torch's autograd engine are 66.
//
// Nothing is kept between calls: outputs and scratch come from torch's allocator on the current stream, launches go to
// the current stream of the tensors' device, and the nodes hold saved tensors through torch's SavedVariable only.
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/SavedTensorHooks.h>
#include <ATen/record_function.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/engine.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>

#include <optional>

#include "ebr_attn.h"
#include "ebr_block.h"
#include "ebr_descent.h"
#include "ebr_rope.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;
namespace py = pybind11;

// ---------------------------------------------------------------------------------------------------------------------
// Which calls are taken
// ---------------------------------------------------------------------------------------------------------------------

// No mode, transform, tracer or saved-tensor hook that has to see the ops or their saved tensors.
bool plain_context() {
    return !at::impl::torch_function_mode_enabled() && !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
           !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
           !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Functionalize) &&
           !torch::jit::tracer::isTracing() && !at::SavedTensorDefaultHooks::get_hooks().has_value();
}

// An ordinary dense GPU tensor.
bool plain_tensor(const Tensor& t) {
    static const c10::DispatchKeySet allowed({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA,
                                              c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutocastCUDA});
    return t.defined() && t.is_cuda() && (t.key_set().raw_repr() & ~allowed.raw_repr()) == 0 && !t.is_inference() &&
           !t._fw_grad(/*level=*/0).defined();
}

// The tensor behind a Python argument if it is one of those, else an undefined one.
Tensor plain(const py::handle& h) {
    if (!THPVariable_CheckExact(h.ptr())) return {};
    const Tensor& t = THPVariable_Unpack(h.ptr());
    return plain_tensor(t) ? t : Tensor();
}

// Whether a node's backward runs here: its saved tensors were plain when it was made, its cotangents and the context have
// to be now.
bool native(const variable_list& grads) {
    for (const Tensor& t : grads)
        if (t.defined() && !plain_tensor(t)) return false;
    return plain_context();
}

// A node's gradients by its Python formula (ebr_amd._host.GRADS), which runs the ops through the dispatcher.
template <class... Args> variable_list python_grads(const char* name, size_t n, const Args&... args) {
    const py::gil_scoped_acquire gil;
    try {
        const py::tuple r = py::module_::import("ebr_amd._host").attr("GRADS")[name](args...);
        TORCH_CHECK(r.size() <= n, name, ": ", r.size(), " gradients for ", n, " inputs");
        variable_list out(n);
        for (size_t i = 0; i < r.size(); ++i)
            if (!r[i].is_none()) out[i] = r[i].cast<Tensor>();
        return out;
    } catch (py::error_already_set& e) {
        e.restore();
        python_error err;
        err.persist();
        throw err;
    }
}

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return EBR_DTYPE_F32;
        case at::kBFloat16: return EBR_DTYPE_BF16;
        case at::kHalf: return EBR_DTYPE_F16;
        case at::kDouble: return EBR_DTYPE_F64;
        default: return -1;
    }
}

bool same_kind(const Tensor& a, const Tensor& b) {
    return a.scalar_type() == b.scalar_type() && a.device() == b.device();
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

void check(int rc, const char* what) {
    if (rc == 0) return;
    TORCH_CHECK_TYPE(rc != EBR_ERR_DTYPE, what, ": ", ebr_attn_error_string(rc), " (code ", rc, ")");
    TORCH_CHECK_VALUE(rc != EBR_ERR_SHAPE, what, ": ", ebr_attn_error_string(rc), " (code ", rc, ")");
    TORCH_CHECK(false, what, ": ", ebr_attn_error_string(rc), " (code ", rc, ")");
}

// Outputs of a backward that is not differentiable again, for a derivative that is recorded: as torch's
// once_differentiable, an error when a later backward reaches them.
variable_list last(variable_list outs) {
    variable_list in;
    std::vector<size_t> at_;
    for (size_t i = 0; i < outs.size(); ++i)
        if (outs[i].defined()) {
            in.push_back(outs[i].detach().set_requires_grad(true));
            at_.push_back(i);
        }
    const auto err = std::make_shared<torch::autograd::DelayedError>(
        "trying to differentiate twice a function that was marked with @once_differentiable", (int64_t)in.size());
    const variable_list out = err->apply(std::move(in));
    for (size_t i = 0; i < at_.size(); ++i) outs[at_[i]] = out[i];
    return outs;
}

// An operand that a call may lack, as an autograd node takes it.
std::optional<Tensor> maybe(const Tensor& t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; }

bool recorded(std::initializer_list<Tensor> ts) {
    if (!at::GradMode::is_enabled()) return false;
    for (const Tensor& t : ts)
        if (t.defined() && t.requires_grad()) return true;
    return false;
}

// ---------------------------------------------------------------------------------------------------------------------
// Attention
// ---------------------------------------------------------------------------------------------------------------------

struct Str3 {
    int64_t s[3];
    explicit Str3(const Tensor& t) : s{t.stride(0), t.stride(1), t.stride(2)} {}
};

// Any B/H/L strides whose row starts are 16-byte aligned, with unit D stride; else a contiguous copy.
Tensor rows(const Tensor& t) {
    const int64_t es = t.element_size();
    bool ok = t.stride(3) == 1 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
    for (int i = 0; i < 3; ++i) ok = ok && t.stride(i) >= 0 && (t.stride(i) * es) % 16 == 0;
    return ok ? t : t.contiguous();
}

Tensor contig(const Tensor& t) {
    return t.is_contiguous() && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0
               ? t
               : t.clone(at::MemoryFormat::Contiguous);
}

struct Dims {
    int B, H, L, D;
    explicit Dims(const Tensor& q)
        : B((int)q.size(0)), H((int)q.size(1)), L((int)q.size(2)), D((int)q.size(3)) {}
};

Tensor scratch(int op, const Tensor& q) {
    const Dims d(q);
    const int64_t n = ebr_attn_scratch_bytes(op, d.B, d.H, d.L, d.D);
    return n > 0 ? at::empty({(n + 3) / 4}, q.options().dtype(at::kFloat)) : Tensor();
}

float* fptr(const Tensor& t) { return t.defined() ? static_cast<float*>(t.data_ptr()) : nullptr; }

variable_list attn_fwd(const Tensor& q_, const Tensor& k_, const Tensor& v_, double scale) {
    RECORD_FUNCTION("ebr_fused::attn_fwd", std::vector<c10::IValue>());
    const c10::DeviceGuard on(q_.device());
    const Tensor q = rows(q_), k = rows(k_), v = rows(v_);
    const Dims d(q);
    const Tensor o = at::empty(q.sizes(), q.options());
    const Tensor lse = at::empty({d.B, d.H, d.L}, q.options().dtype(at::kFloat));
    check(ebr_attn_fwd(dtype_code(q.scalar_type()), d.B, d.H, d.L, d.D, (float)scale, q.data_ptr(), Str3(q).s,
                       k.data_ptr(), Str3(k).s, v.data_ptr(), Str3(v).s, o.data_ptr(), lse.data_ptr(), stream_of(q)),
          "ebr_attn_fwd");
    return {o, lse};
}

variable_list attn_bwd(const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& o_, const Tensor& lse_,
                       const Tensor& do_, double scale) {
    RECORD_FUNCTION("ebr_fused::attn_bwd", std::vector<c10::IValue>());
    const c10::DeviceGuard on(q_.device());
    const Tensor q = rows(q_), k = rows(k_), v = rows(v_), dO = rows(do_.to(q_.scalar_type()));
    const Tensor o = contig(o_), lse = contig(lse_);
    const Dims d(q);
    variable_list out(3);
    for (Tensor& t : out) t = at::empty(q.sizes(), q.options());
    const Tensor s = scratch(EBR_OP_BWD, q);
    check(ebr_attn_bwd(dtype_code(q.scalar_type()), d.B, d.H, d.L, d.D, (float)scale, q.data_ptr(), Str3(q).s,
                       k.data_ptr(), Str3(k).s, v.data_ptr(), Str3(v).s, o.data_ptr(), lse.data_ptr(), dO.data_ptr(),
                       Str3(dO).s, out[0].data_ptr(), out[1].data_ptr(), out[2].data_ptr(), fptr(s), stream_of(q)),
          "ebr_attn_bwd");
    return out;
}

variable_list attn_bwd_bwd(const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& o_,
                           const Tensor& lse_, const Tensor& do_, const Tensor& gq_, const Tensor& gk_,
                           const Tensor& gv_, double scale) {
    RECORD_FUNCTION("ebr_fused::attn_bwd_bwd", std::vector<c10::IValue>());
    const c10::DeviceGuard on(q_.device());
    const auto st = q_.scalar_type();
    const Tensor q = rows(q_), k = rows(k_), v = rows(v_), dO = rows(do_.to(st));
    const Tensor gq = rows(gq_.to(st)), gk = rows(gk_.to(st)), gv = rows(gv_.to(st));
    const Tensor o = contig(o_), lse = contig(lse_);
    const Dims d(q);
    variable_list out(4);
    for (Tensor& t : out) t = at::empty(q.sizes(), q.options());
    const Tensor s = scratch(EBR_OP_BWD_BWD, q);
    check(ebr_attn_bwd_bwd(dtype_code(st), d.B, d.H, d.L, d.D, (float)scale, q.data_ptr(), Str3(q).s, k.data_ptr(),
                           Str3(k).s, v.data_ptr(), Str3(v).s, o.data_ptr(), lse.data_ptr(), dO.data_ptr(),
                           Str3(dO).s, gq.data_ptr(), Str3(gq).s, gk.data_ptr(), Str3(gk).s, gv.data_ptr(),
                           Str3(gv).s, out[0].data_ptr(), out[1].data_ptr(), out[2].data_ptr(), out[3].data_ptr(),
                           fptr(s), stream_of(q)),
          "ebr_attn_bwd_bwd");
    return out;
}

struct AttnBwdBwd : Function<AttnBwdBwd> {
    static variable_list forward(AutogradContext*, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o,
                                 const Tensor& lse, const Tensor& dO, const Tensor& gq, const Tensor& gk,
                                 const Tensor& gv, double scale) {
        return attn_bwd_bwd(q, k, v, o, lse, dO, gq, gk, gv, scale);
    }
    static variable_list backward(AutogradContext*, const variable_list&) {
        TORCH_CHECK(false, "ebr_fused::attn_bwd_bwd has no derivative");
    }
};

// First derivative as a differentiable node; o and lse are constants in it (their dependence is in hq, hk, hv, hdo).
struct AttnBwd : Function<AttnBwd> {
    static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v,
                                 const Tensor& o, const Tensor& lse, const Tensor& dO, double scale) {
        ctx->save_for_backward({q, k, v, o, lse, dO});
        ctx->saved_data["scale"] = scale;
        ctx->set_materialize_grads(false);  // an unused output's cotangent becomes one expanded zero row
        return attn_bwd(q, k, v, o, lse, dO, scale);
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& g) {
        const variable_list s = ctx->get_saved_variables();
        const double scale = ctx->saved_data["scale"].toDouble();
        if (!native(g))
            return python_grads("attention_bwd", 7, s[0], s[1], s[2], s[3], s[4], s[5], scale, g[0], g[1], g[2]);
        Tensor cot[3];
        for (int i = 0; i < 3; ++i)
            cot[i] = g[i].defined() ? g[i] : at::zeros({s[i].size(3)}, s[i].options()).expand(s[i].sizes());
        const variable_list h =
            recorded({s[0], s[1], s[2], s[5], cot[0], cot[1], cot[2]})
                ? AttnBwdBwd::apply(s[0], s[1], s[2], s[3], s[4], s[5], cot[0], cot[1], cot[2], scale)
                : attn_bwd_bwd(s[0], s[1], s[2], s[3], s[4], s[5], cot[0], cot[1], cot[2], scale);
        return {h[0], h[1], h[2], Tensor(), Tensor(), h[3].to(s[5].scalar_type()), Tensor()};
    }
};

struct AttnFwd : Function<AttnFwd> {
    static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v,
                                 double scale) {
        variable_list out = attn_fwd(q, k, v, scale);
        ctx->mark_non_differentiable({out[1]});
        ctx->save_for_backward({q, k, v, out[0], out[1]});
        ctx->saved_data["scale"] = scale;
        ctx->set_materialize_grads(false);
        return out;
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& g) {
        if (!g[0].defined()) return variable_list(4);  // only AttnBwd used o: nothing to add
        const variable_list s = ctx->get_saved_variables();
        const double scale = ctx->saved_data["scale"].toDouble();
        if (!native(g)) return python_grads("attention", 4, s[0], s[1], s[2], s[3], s[4], scale, g[0]);
        variable_list d = AttnBwd::apply(s[0], s[1], s[2], s[3], s[4], g[0], scale);
        d.emplace_back();
        return d;
    }
};

// fused_attention, or None for a call that stays in Python.
py::object attention(const py::handle& hq, const py::handle& hk, const py::handle& hv, std::optional<double> scale) {
    const Tensor q = plain(hq), k = plain(hk), v = plain(hv);
    if (!q.defined() || !k.defined() || !v.defined() || !plain_context()) return py::none();
    if (q.dim() != 4 || k.sizes() != q.sizes() || v.sizes() != q.sizes() || !same_kind(q, k) || !same_kind(q, v))
        return py::none();
    const int code = dtype_code(q.scalar_type());
    if (code < 0 || code == EBR_DTYPE_F64 || q.numel() == 0) return py::none();
    const int64_t D = q.size(3);
    if (D > 256 || D % (code == EBR_DTYPE_F32 ? 4 : 8) || q.numel() / D >= (int64_t(1) << 31)) return py::none();
    return py::cast(AttnFwd::apply(q, k, v, scale ? *scale : std::pow((double)D, -0.5))[0]);
}

// ---------------------------------------------------------------------------------------------------------------------
// RoPE split and merge: each other's adjoint; the tables and the temperature carry no gradient
// ---------------------------------------------------------------------------------------------------------------------

Tensor unit_last(const Tensor& t) { return t.stride(-1) == 1 ? t : t.contiguous(); }

variable_list rope_split_launch(const Tensor& qkv_, const Tensor& cos, const Tensor& sin, const Tensor& qs,
                                int64_t heads) {
    RECORD_FUNCTION("ebr_fused::rope_split", std::vector<c10::IValue>());
    const c10::DeviceGuard on(qkv_.device());
    const Tensor qkv = unit_last(qkv_);
    const int64_t B = qkv.size(0), N = qkv.size(1), D = qkv.size(2) / (3 * heads);
    variable_list out(3);
    for (Tensor& t : out) t = at::empty({B, heads, N, D}, qkv.options());
    check(ebr_rope_split(dtype_code(qkv.scalar_type()), (int)B, (int)N, (int)heads, (int)D, qkv.data_ptr(),
                         qkv.stride(0), qkv.stride(1), fptr(cos), fptr(sin), fptr(qs), out[0].data_ptr(),
                         out[1].data_ptr(), out[2].data_ptr(), stream_of(qkv)),
          "ebr_rope_split");
    return out;
}

Tensor rope_merge_launch(const Tensor& dq_, const Tensor& dk_, const Tensor& dv_, const Tensor& cos,
                         const Tensor& sin, const Tensor& qs) {
    RECORD_FUNCTION("ebr_fused::rope_merge", std::vector<c10::IValue>());
    const c10::DeviceGuard on(dq_.device());
    const auto st = dq_.scalar_type();
    const Tensor dq = unit_last(dq_), dk = unit_last(dk_.to(st)), dv = unit_last(dv_.to(st));
    const Dims d(dq);
    const Tensor g = at::empty({d.B, d.L, int64_t(3) * d.H * d.D}, dq.options());
    check(ebr_rope_merge(dtype_code(st), d.B, d.H, d.L, d.D, dq.data_ptr(), Str3(dq).s, dk.data_ptr(), Str3(dk).s,
                         dv.data_ptr(), Str3(dv).s, fptr(cos), fptr(sin), fptr(qs), g.data_ptr(), stream_of(dq)),
          "ebr_rope_merge");
    return g;
}

struct RopeMerge;

struct RopeSplit : Function<RopeSplit> {
    static variable_list forward(AutogradContext* ctx, const Tensor& qkv, const Tensor& cos, const Tensor& sin,
                                 const std::optional<Tensor>& qs_, int64_t heads) {
        const Tensor qs = qs_.value_or(Tensor());
        ctx->save_for_backward({cos, sin, qs});
        ctx->set_materialize_grads(false);
        variable_list out = rope_split_launch(qkv, cos, sin, qs, heads);
        ctx->saved_data["shape"] = out[0].sizes().vec();
        return out;
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& g);
};

struct RopeMerge : Function<RopeMerge> {
    static variable_list forward(AutogradContext* ctx, const Tensor& dq, const Tensor& dk, const Tensor& dv,
                                 const Tensor& cos, const Tensor& sin, const std::optional<Tensor>& qs_) {
        const Tensor qs = qs_.value_or(Tensor());
        ctx->save_for_backward({cos, sin, qs});
        ctx->saved_data["heads"] = dq.size(1);
        ctx->set_materialize_grads(false);
        return {rope_merge_launch(dq, dk, dv, cos, sin, qs)};
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& g) {
        if (!g[0].defined()) return variable_list(6);
        const variable_list s = ctx->get_saved_variables();
        const int64_t heads = ctx->saved_data["heads"].toInt();
        if (!native(g)) return python_grads("rope_merge", 6, s[0], s[1], s[2], heads, g[0]);
        variable_list d = RopeSplit::apply(g[0], s[0], s[1], maybe(s[2]), heads);
        d.resize(6);
        return d;
    }
};

variable_list RopeSplit::backward(AutogradContext* ctx, const variable_list& g) {
    variable_list out(5);
    const std::vector<int64_t> shape = ctx->saved_data["shape"].toIntVector();
    Tensor some;
    for (const Tensor& t : g)
        if (t.defined()) some = t;
    if (!some.defined()) return out;
    const variable_list s = ctx->get_saved_variables();
    if (!native(g)) return python_grads("rope_split", 5, s[0], s[1], s[2], shape, g[0], g[1], g[2]);
    Tensor d[3];
    for (int i = 0; i < 3; ++i) d[i] = g[i].defined() ? g[i] : at::zeros({shape[3]}, some.options()).expand(shape);
    out[0] = RopeMerge::apply(d[0], d[1], d[2], s[0], s[1], maybe(s[2]))[0];
    return out;
}

py::object rope_split(const py::handle& hqkv, const py::handle& hcos, const py::handle& hsin, int64_t heads,
                      const py::handle& hqs) {
    const Tensor qkv = plain(hqkv);
    Tensor cos = plain(hcos), sin = plain(hsin), qs;
    if (!qkv.defined() || !cos.defined() || !sin.defined() || !plain_context()) return py::none();
    if (!hqs.is_none()) {
        qs = plain(hqs);
        if (!qs.defined() || qs.numel() != heads || qs.device() != qkv.device()) return py::none();
        qs = qs.detach().to(at::kFloat).contiguous();
    }
    const int code = dtype_code(qkv.scalar_type());
    if (code < 0 || code == EBR_DTYPE_F64 || heads < 1 || qkv.dim() != 3 || qkv.numel() == 0 ||
        qkv.size(2) % (3 * heads))
        return py::none();
    const int64_t N = qkv.size(1), D = qkv.size(2) / (3 * heads);
    const std::vector<int64_t> table = {N, D};
    if (D % 4 || D > 256 || cos.sizes() != table || sin.sizes() != table || cos.device() != qkv.device() ||
        sin.device() != qkv.device())
        return py::none();
    cos = cos.to(at::kFloat).contiguous();
    sin = sin.to(at::kFloat).contiguous();
    const variable_list o = RopeSplit::apply(qkv, cos, sin, maybe(qs), heads);
    return py::make_tuple(o[0], o[1], o[2]);
}

// ---------------------------------------------------------------------------------------------------------------------
// Rotary split, temperature, attention and the heads' merge as one node: y [B, N, H D] of a projection qkv [B, N, 3 H D].
// The split's q (tempered), k and v are outputs of the node that its backward's node reads, so the second derivative's
// gradients of them come back here and the merge adds them.
// ---------------------------------------------------------------------------------------------------------------------

Tensor heads_apart(const Tensor& y, int64_t heads) {  // [B, N, H D] as [B, H, N, D]
    return y.reshape({y.size(0), y.size(1), heads, y.size(2) / heads}).transpose(1, 2);
}

Tensor heads_together(const Tensor& o) {
    return o.transpose(1, 2).reshape({o.size(0), o.size(2), o.size(1) * o.size(3)});
}

Tensor head_scratch(const Tensor& like, int64_t B, int64_t N, int64_t H, int64_t D) {
    const int64_t n = ebr_rope_graded_scratch(dtype_code(like.scalar_type()), (int)B, (int)N, (int)H, (int)D);
    return at::empty({n / 4}, like.options().dtype(at::kFloat));
}

// {q, k, v, dt}: the split of qkv with the temperature t; dt = per-head sums of w and the rotated q where w is defined.
variable_list split_graded(const Tensor& qkv, const Tensor& cos, const Tensor& sin, const Tensor& t, const Tensor& w,
                           int64_t heads) {
    RECORD_FUNCTION("ebr_fused::rope_split", std::vector<c10::IValue>());
    const c10::DeviceGuard on(qkv.device());
    const Tensor x = contig(qkv);
    const int64_t B = x.size(0), N = x.size(1), D = x.size(2) / (3 * heads);
    variable_list out(4);
    for (int i = 0; i < 3; ++i) out[i] = at::empty({B, heads, N, D}, x.options());
    Tensor part;
    if (w.defined()) {
        out[3] = at::empty({heads}, t.options());
        part = head_scratch(x, B, N, heads, D);
    }
    check(ebr_rope_split_graded(dtype_code(x.scalar_type()), (int)B, (int)N, (int)heads, (int)D, x.data_ptr(),
                                x.stride(0), x.stride(1), fptr(cos), fptr(sin), fptr(t), out[0].data_ptr(),
                                out[1].data_ptr(), out[2].data_ptr(), w.defined() ? w.data_ptr() : nullptr,
                                fptr(out[3]), fptr(part), stream_of(x)),
          "ebr_rope_split_graded");
    return out;
}

// {g, dt}: the merge of d plus add (three gradients each; add may be undefined); dt where qkv is defined.
variable_list merge_graded(const Tensor (&d_)[3], const Tensor (&add_)[3], const Tensor& cos, const Tensor& sin,
                           const Tensor& t, const Tensor& qkv_) {
    RECORD_FUNCTION("ebr_fused::rope_merge", std::vector<c10::IValue>());
    const c10::DeviceGuard on(d_[0].device());
    const auto st = d_[0].scalar_type();
    Tensor d[3], add[3];
    for (int i = 0; i < 3; ++i) {
        d[i] = rows(d_[i].to(st));
        if (add_[i].defined()) add[i] = contig(add_[i].to(st));
    }
    const Dims m(d[0]);
    const Tensor g = at::empty({m.B, m.L, int64_t(3) * m.H * m.D}, d[0].options());
    Tensor dt, part, qkv;
    if (qkv_.defined()) {
        qkv = contig(qkv_);
        dt = at::empty({m.H}, t.options());
        part = head_scratch(d[0], m.B, m.L, m.H, m.D);
    }
    const auto ptr = [](const Tensor& x) -> const void* { return x.defined() ? x.data_ptr() : nullptr; };
    check(ebr_rope_merge_graded(dtype_code(st), m.B, m.H, m.L, m.D, d[0].data_ptr(), Str3(d[0]).s, d[1].data_ptr(),
                                Str3(d[1]).s, d[2].data_ptr(), Str3(d[2]).s, ptr(add[0]), ptr(add[1]), ptr(add[2]),
                                fptr(cos), fptr(sin), fptr(t), g.data_ptr(), ptr(qkv), fptr(dt), fptr(part),
                                stream_of(g)),
          "ebr_rope_merge_graded");
    return {g, dt};
}

// The gradient of qkv from dy as a differentiable node (inputs t, q, k, v, dy; o and lse are constants in it).
struct RopeAttnBwd : Function<RopeAttnBwd> {
    static variable_list forward(AutogradContext* ctx, const Tensor& t, const Tensor& q, const Tensor& k,
                                 const Tensor& v, const Tensor& dy, const Tensor& o, const Tensor& lse,
                                 const Tensor& cos, const Tensor& sin, double scale) {
        const variable_list d = attn_bwd(q, k, v, o, lse, heads_apart(dy, q.size(1)), scale);
        ctx->save_for_backward({t, q, k, v, dy, o, lse, cos, sin, d[0]});
        ctx->saved_data["scale"] = scale;
        ctx->set_materialize_grads(false);
        return {merge_graded({d[0], d[1], d[2]}, {Tensor(), Tensor(), Tensor()}, cos, sin, t, Tensor())[0]};
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& g) {
        variable_list out(10);
        if (!g[0].defined()) return out;
        const bool want_t = ctx->needs_input_grad(0);
        const variable_list s = ctx->get_saved_variables();
        const Tensor &t = s[0], &q = s[1], &dy = s[4];
        const int64_t heads = q.size(1);
        if (!native(g))
            return python_grads("rope_attention_bwd", 10, t, q, s[2], s[3], dy, s[5], s[6], s[7], s[8], s[9],
                                ctx->saved_data["scale"].toDouble(), want_t, g[0]);
        const variable_list c = split_graded(g[0].to(q.scalar_type()), s[7], s[8], t, want_t ? s[9] : Tensor(), heads);
        const variable_list h = attn_bwd_bwd(q, s[2], s[3], s[5], s[6], heads_apart(dy, heads), c[0], c[1], c[2],
                                             ctx->saved_data["scale"].toDouble());
        variable_list d = {c[3], h[0], h[1], h[2], heads_together(h[3])};
        if (recorded({t, q, s[2], s[3], dy, g[0]})) d = last(std::move(d));
        for (size_t i = 0; i < d.size(); ++i) out[i] = d[i];
        return out;
    }
};

struct RopeAttn : Function<RopeAttn> {
    static variable_list forward(AutogradContext* ctx, const Tensor& qkv, const Tensor& t, const Tensor& cos,
                                 const Tensor& sin, int64_t heads, double scale) {
        const variable_list x = split_graded(qkv, cos, sin, t, Tensor(), heads);
        const variable_list o = attn_fwd(x[0], x[1], x[2], scale);
        ctx->save_for_backward({t.requires_grad() ? qkv : Tensor(), t, cos, sin, x[0], x[1], x[2], o[0], o[1]});
        ctx->saved_data["scale"] = scale;
        ctx->set_materialize_grads(false);
        return {heads_together(o[0]), x[0], x[1], x[2]};
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& g) {
        variable_list out(6);
        const Tensor& dy = g[0];
        const bool more = g[1].defined() || g[2].defined() || g[3].defined();
        if (!dy.defined() && !more) return out;
        const bool want_t = ctx->needs_input_grad(1);
        const variable_list s = ctx->get_saved_variables();
        const Tensor &qkv = s[0], &t = s[1], &cos = s[2], &sin = s[3], &q = s[4], &k = s[5], &v = s[6];
        const int64_t heads = q.size(1);
        const double scale = ctx->saved_data["scale"].toDouble();
        if (!native(g))
            return python_grads("rope_attention", 6, qkv, t, cos, sin, q, k, v, s[7], s[8], scale, want_t, dy, g[1],
                                g[2], g[3]);
        if (at::GradMode::is_enabled()) {
            if (!more && !want_t) {
                out[0] = RopeAttnBwd::apply(t, q, k, v, dy, s[7], s[8], cos, sin, scale)[0];
                return out;
            }
            // every part as a node of its own, for derivatives of any of them
            Tensor d[3];
            if (dy.defined()) {
                const variable_list a = AttnBwd::apply(q, k, v, s[7], s[8], heads_apart(dy, heads), scale);
                for (int i = 0; i < 3; ++i) d[i] = a[i];
            }
            for (int i = 0; i < 3; ++i) {
                if (g[i + 1].defined()) d[i] = d[i].defined() ? d[i] + g[i + 1] : g[i + 1];
                if (!d[i].defined()) d[i] = at::zeros({q.size(3)}, q.options()).expand(q.sizes());
            }
            if (want_t) {
                const Tensor rq = RopeSplit::apply(qkv, cos, sin, std::nullopt, heads)[0];
                out[1] = (d[0] * rq).sum({0, 2, 3}, false, at::kFloat).to(t.scalar_type());
            }
            const Tensor td = t.to(q.scalar_type()).view({1, heads, 1, 1});
            out[0] = RopeMerge::apply(d[0] * td, d[1], d[2], cos, sin, std::nullopt)[0];
            return out;
        }
        Tensor d[3], add[3];
        if (dy.defined()) {
            const variable_list a = attn_bwd(q, k, v, s[7], s[8], heads_apart(dy, heads), scale);
            for (int i = 0; i < 3; ++i) {
                d[i] = a[i];
                if (more) add[i] = g[i + 1].defined() ? g[i + 1] : at::zeros_like(q);
            }
        } else {
            for (int i = 0; i < 3; ++i)
                d[i] = g[i + 1].defined() ? g[i + 1] : at::zeros({q.size(3)}, q.options()).expand(q.sizes());
        }
        const variable_list m = merge_graded(d, add, cos, sin, t, want_t ? qkv : Tensor());
        out[0] = m[0];
        out[1] = m[1];
        return out;
    }
};

// Attention of a projection with the rotary tables and the temperature ``ht`` (fp32 [H], rounded to the dtype inside).
py::object rope_attention(const py::handle& hqkv, const py::handle& hcos, const py::handle& hsin, int64_t heads,
                          const py::handle& ht) {
    const Tensor qkv = plain(hqkv), cos = plain(hcos), sin = plain(hsin), t = plain(ht);
    if (!qkv.defined() || !cos.defined() || !sin.defined() || !t.defined() || !plain_context()) return py::none();
    const int code = dtype_code(qkv.scalar_type());
    if (code < 0 || code == EBR_DTYPE_F64 || heads < 1 || qkv.dim() != 3 || qkv.numel() == 0 ||
        qkv.size(2) % (3 * heads))
        return py::none();
    const int64_t B = qkv.size(0), N = qkv.size(1), D = qkv.size(2) / (3 * heads);
    const std::vector<int64_t> table = {N, D};
    if (D > 128 || cos.sizes() != table || sin.sizes() != table || t.dim() != 1 || t.size(0) != heads ||
        B * heads * N >= (int64_t(1) << 31))
        return py::none();
    for (const Tensor& x : {cos, sin, t})
        if (x.scalar_type() != at::kFloat || !x.is_contiguous() || x.device() != qkv.device() ||
            reinterpret_cast<uintptr_t>(x.data_ptr()) % (x.dim() == 2 ? 32 : 4))
            return py::none();
    if (ebr_rope_graded_scratch(code, (int)B, (int)N, (int)heads, (int)D) == 0) return py::none();
    return py::cast(RopeAttn::apply(qkv, t, cos, sin, heads, std::pow((double)D, -0.5))[0]);
}

// ---------------------------------------------------------------------------------------------------------------------
// Energy block: rms_norm and SwiGLU, each differentiable twice
// ---------------------------------------------------------------------------------------------------------------------

Tensor dense(const Tensor& t) { return t.is_contiguous() ? t : t.contiguous(); }

struct RowsOf {
    int64_t rows, width;
    explicit RowsOf(const Tensor& t) : rows(t.numel() / t.size(-1)), width(t.size(-1)) {}
};

Tensor rmsnorm(const Tensor& x_, double eps) {
    RECORD_FUNCTION("ebr_fused::block_rmsnorm", std::vector<c10::IValue>());
    const c10::DeviceGuard on(x_.device());
    const Tensor x = dense(x_), y = at::empty(x.sizes(), x.options());
    const RowsOf r(x);
    check(ebr_block_rmsnorm(dtype_code(x.scalar_type()), r.rows, (int)r.width, (float)eps, x.data_ptr(), y.data_ptr(),
                            stream_of(x)),
          "ebr_block_rmsnorm");
    return y;
}

// {sum, rms_norm(sum)} of sum = a + b
variable_list add_rmsnorm(const Tensor& a_, const Tensor& b_, double eps) {
    RECORD_FUNCTION("ebr_fused::block_add_rmsnorm", std::vector<c10::IValue>());
    const c10::DeviceGuard on(a_.device());
    const Tensor a = dense(a_), b = dense(b_), sum = at::empty(a.sizes(), a.options());
    const Tensor y = at::empty(a.sizes(), a.options());
    const RowsOf r(a);
    check(ebr_block_add_rmsnorm(dtype_code(a.scalar_type()), r.rows, (int)r.width, (float)eps, a.data_ptr(),
                                b.data_ptr(), sum.data_ptr(), y.data_ptr(), stream_of(a)),
          "ebr_block_add_rmsnorm");
    return {sum, y};
}

// ``acc``: a gradient of x that is already there and is added, or undefined.
Tensor rmsnorm_bwd(const Tensor& x_, const Tensor& dy_, const Tensor& acc_, double eps) {
    RECORD_FUNCTION("ebr_fused::block_rmsnorm_bwd", std::vector<c10::IValue>());
    const c10::DeviceGuard on(x_.device());
    const auto st = x_.scalar_type();
    const Tensor x = dense(x_), dy = dense(dy_.to(st)), dx = at::empty(x.sizes(), x.options());
    const RowsOf r(x);
    if (acc_.defined()) {
        const Tensor acc = dense(acc_.to(st));
        check(ebr_block_rmsnorm_bwd_add(dtype_code(st), r.rows, (int)r.width, (float)eps, x.data_ptr(), dy.data_ptr(),
                                        acc.data_ptr(), dx.data_ptr(), stream_of(x)),
              "ebr_block_rmsnorm_bwd_add");
    } else {
        check(ebr_block_rmsnorm_bwd(dtype_code(st), r.rows, (int)r.width, (float)eps, x.data_ptr(), dy.data_ptr(),
                                    dx.data_ptr(), stream_of(x)),
              "ebr_block_rmsnorm_bwd");
    }
    return dx;
}

variable_list rmsnorm_bwd2(const Tensor& x_, const Tensor& dy_, const Tensor& c_, double eps) {
    RECORD_FUNCTION("ebr_fused::block_rmsnorm_bwd2", std::vector<c10::IValue>());
    const c10::DeviceGuard on(x_.device());
    const auto st = x_.scalar_type();
    const Tensor x = dense(x_), dy = dense(dy_.to(st)), c = dense(c_.to(st));
    const Tensor gx = at::empty(x.sizes(), x.options()), gdy = at::empty(x.sizes(), x.options());
    const RowsOf r(x);
    check(ebr_block_rmsnorm_bwd2(dtype_code(st), r.rows, (int)r.width, (float)eps, x.data_ptr(), dy.data_ptr(),
                                 c.data_ptr(), gx.data_ptr(), gdy.data_ptr(), stream_of(x)),
          "ebr_block_rmsnorm_bwd2");
    return {gx, gdy};
}

struct RmsNormBwd : Function<RmsNormBwd> {
    static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& dy, double eps) {
        ctx->save_for_backward({x, dy});
        ctx->saved_data["eps"] = eps;
        ctx->set_materialize_grads(false);
        return {rmsnorm_bwd(x, dy, Tensor(), eps)};
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& g) {
        if (!g[0].defined()) return variable_list(3);
        const variable_list s = ctx->get_saved_variables();
        const double eps = ctx->saved_data["eps"].toDouble();
        if (!native(g)) return python_grads("rms_norm_bwd", 3, s[0], s[1], eps, g[0]);
        variable_list d = rmsnorm_bwd2(s[0], s[1], g[0], eps);
        if (recorded({s[0], s[1], g[0]})) d = last(std::move(d));
        d.emplace_back();
        return d;
    }
};

// The input of a forward node as an output of its own, which the backward's node reads: the gradients that arise there
// (the second derivative's) then come back to the forward node, whose own gradient kernel adds them.
Tensor own_input(const Tensor& x) { return x.detach(); }

// A second derivative alone passes through the forward node without using what it saved, and frees that where the caller
// keeps no graph. With the input itself saved in the backward's node that pass would not come here at all, so it must
// not use the node up: its saved input (output 1) is set aside for a later pass, until one uses it.
struct Kept {
    AutogradContext* ctx;
    bool keeps = torch::autograd::get_current_graph_task_keep_graph();

    Tensor use() {
        const auto it = ctx->saved_data.find("kept");
        if (it == ctx->saved_data.end()) {
            const Tensor x = ctx->get_saved_variables()[0];  // an error where a pass has used it up
            if (!keeps) ctx->saved_data["used"] = true;
            return x;
        }
        const Tensor x = it->second.toTensor().detach();
        TORCH_CHECK((int64_t)x._version() == ctx->saved_data["version"].toInt(),
                    "one of the variables needed for gradient computation has been modified by an inplace operation");
        if (const auto node = torch::autograd::get_current_node())
            torch::autograd::impl::set_gradient_edge(x, {node, 1});
        if (!keeps) ctx->saved_data.erase(it);
        return x;
    }
    void pass() {
        if (keeps || ctx->saved_data.count("kept") || ctx->saved_data.count("used")) return;
        const Tensor x = ctx->get_saved_variables()[0].detach();
        ctx->saved_data["version"] = (int64_t)x._version();
        ctx->saved_data["kept"] = x;
        ctx->saved_data["used"] = true;  // what the context itself saved goes with this pass
    }
};

// The gradient of a norm's input: from dy through the backward's node, plus ``acc``.
Tensor norm_grad(AutogradContext* ctx, const Tensor& dy, const Tensor& acc) {
    Kept saved{ctx};
    if (!dy.defined()) {
        saved.pass();
        return acc;
    }
    const Tensor x = saved.use();
    const double eps = ctx->saved_data["eps"].toDouble();
    if (!native({dy, acc})) return python_grads("rms_norm", 1, x, eps, dy, acc)[0];
    if (acc.defined() && !at::GradMode::is_enabled()) return rmsnorm_bwd(x, dy, acc, eps);
    const Tensor dx = RmsNormBwd::apply(x, dy, eps)[0];
    return acc.defined() ? dx + acc : dx;
}

struct RmsNorm : Function<RmsNorm> {
    static variable_list forward(AutogradContext* ctx, const Tensor& x, double eps) {
        const Tensor own = own_input(x);
        ctx->save_for_backward({own});
        ctx->saved_data["eps"] = eps;
        ctx->set_materialize_grads(false);
        return {rmsnorm(x, eps), own};
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& g) {
        return {norm_grad(ctx, g[0], g[1]), Tensor()};
    }
};

struct AddRmsNorm : Function<AddRmsNorm> {
    static variable_list forward(AutogradContext* ctx, const Tensor& a, const Tensor& b, double eps) {
        variable_list out = add_rmsnorm(a, b, eps);
        ctx->save_for_backward({out[0]});
        ctx->saved_data["eps"] = eps;
        ctx->set_materialize_grads(false);
        return {out[1], out[0]};
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& g) {
        const Tensor d = norm_grad(ctx, g[0], g[1]);
        return {d, d, Tensor()};
    }
};

Tensor swiglu_fwd(const Tensor& gu_) {
    RECORD_FUNCTION("ebr_fused::block_swiglu", std::vector<c10::IValue>());
    const c10::DeviceGuard on(gu_.device());
    const Tensor gu = dense(gu_);
    std::vector<int64_t> shape = gu.sizes().vec();
    shape.back() /= 2;
    const Tensor y = at::empty(shape, gu.options());
    const RowsOf r(gu);
    check(ebr_block_swiglu(dtype_code(gu.scalar_type()), r.rows, (int)(r.width / 2), gu.data_ptr(), y.data_ptr(),
                           stream_of(gu)),
          "ebr_block_swiglu");
    return y;
}

// ``acc``: a gradient of gu that is already there and is added, or undefined.
Tensor swiglu_bwd(const Tensor& gu_, const Tensor& dy_, const Tensor& acc_) {
    RECORD_FUNCTION("ebr_fused::block_swiglu_bwd", std::vector<c10::IValue>());
    const c10::DeviceGuard on(gu_.device());
    const Tensor gu = dense(gu_), dy = dense(dy_.to(gu_.scalar_type())), d = at::empty(gu.sizes(), gu.options());
    const RowsOf r(gu);
    if (acc_.defined()) {
        const Tensor acc = dense(acc_.to(gu.scalar_type()));
        check(ebr_block_swiglu_bwd_add(dtype_code(gu.scalar_type()), r.rows, (int)(r.width / 2), gu.data_ptr(),
                                       dy.data_ptr(), acc.data_ptr(), d.data_ptr(), stream_of(gu)),
              "ebr_block_swiglu_bwd_add");
        return d;
    }
    check(ebr_block_swiglu_bwd(dtype_code(gu.scalar_type()), r.rows, (int)(r.width / 2), gu.data_ptr(), dy.data_ptr(),
                               d.data_ptr(), stream_of(gu)),
          "ebr_block_swiglu_bwd");
    return d;
}

variable_list swiglu_bwd2(const Tensor& gu_, const Tensor& dy_, const Tensor& c_) {
    RECORD_FUNCTION("ebr_fused::block_swiglu_bwd2", std::vector<c10::IValue>());
    const c10::DeviceGuard on(gu_.device());
    const auto st = gu_.scalar_type();
    const Tensor gu = dense(gu_), dy = dense(dy_.to(st)), c = dense(c_.to(st));
    const Tensor ggu = at::empty(gu.sizes(), gu.options()), gdy = at::empty(dy.sizes(), dy.options());
    const RowsOf r(gu);
    check(ebr_block_swiglu_bwd2(dtype_code(st), r.rows, (int)(r.width / 2), gu.data_ptr(), dy.data_ptr(),
                                c.data_ptr(), ggu.data_ptr(), gdy.data_ptr(), stream_of(gu)),
          "ebr_block_swiglu_bwd2");
    return {ggu, gdy};
}

struct SwiGLUBwd : Function<SwiGLUBwd> {
    static variable_list forward(AutogradContext* ctx, const Tensor& gu, const Tensor& dy) {
        ctx->save_for_backward({gu, dy});
        ctx->set_materialize_grads(false);
        return {swiglu_bwd(gu, dy, Tensor())};
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& g) {
        if (!g[0].defined()) return variable_list(2);
        const variable_list s = ctx->get_saved_variables();
        if (!native(g)) return python_grads("swiglu_bwd", 2, s[0], s[1], g[0]);
        variable_list d = swiglu_bwd2(s[0], s[1], g[0]);
        return recorded({s[0], s[1], g[0]}) ? last(std::move(d)) : d;
    }
};

struct SwiGLU : Function<SwiGLU> {
    static variable_list forward(AutogradContext* ctx, const Tensor& gu) {
        const Tensor own = own_input(gu);
        ctx->save_for_backward({own});
        ctx->set_materialize_grads(false);
        return {swiglu_fwd(gu), own};
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& g) {
        Kept saved{ctx};
        if (!g[0].defined()) {
            saved.pass();
            return {g[1]};
        }
        const Tensor gu = saved.use();
        if (!native(g)) return python_grads("swiglu", 1, gu, g[0], g[1]);
        if (g[1].defined() && !at::GradMode::is_enabled()) return {swiglu_bwd(gu, g[0], g[1])};
        const Tensor d = SwiGLUBwd::apply(gu, g[0])[0];
        return {g[1].defined() ? d + g[1] : d};
    }
};

bool block_takes(const Tensor& x) {
    return x.defined() && x.dim() >= 1 && x.numel() > 0 && dtype_code(x.scalar_type()) >= 0 &&
           x.size(-1) < (int64_t(1) << 31) && plain_context();
}

py::object rms_norm(const py::handle& hx, double eps) {
    const Tensor x = plain(hx);
    if (!block_takes(x)) return py::none();
    return py::cast(recorded({x}) ? RmsNorm::apply(x, eps)[0] : rmsnorm(x, eps));
}

// rms_norm(a + b)
py::object add_rms_norm(const py::handle& ha, const py::handle& hb, double eps) {
    const Tensor a = plain(ha), b = plain(hb);
    if (!block_takes(a) || !b.defined() || a.sizes() != b.sizes() || !same_kind(a, b)) return py::none();
    return py::cast(recorded({a, b}) ? AddRmsNorm::apply(a, b, eps)[0] : add_rmsnorm(a, b, eps)[1]);
}

py::object swiglu(const py::handle& hgu) {
    const Tensor gu = plain(hgu);
    if (!block_takes(gu) || gu.size(-1) % 2) return py::none();
    return py::cast(recorded({gu}) ? SwiGLU::apply(gu)[0] : swiglu_fwd(gu));
}

// ---------------------------------------------------------------------------------------------------------------------
// Descent wrapper: first order only (the step size and the noise scale are constants of the schedule)
// ---------------------------------------------------------------------------------------------------------------------

void* vptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

Tensor noisy_bwd(const Tensor& z_, const Tensor& dv_, double eps) {
    RECORD_FUNCTION("ebr_fused::descent_noisy_point_bwd", std::vector<c10::IValue>());
    const c10::DeviceGuard on(z_.device());
    const Tensor z = dense(z_), dv = dense(dv_.to(z_.scalar_type())), dz = at::empty(z.sizes(), z.options());
    check(ebr_descent_noisy_point_bwd(dtype_code(z.scalar_type()), (int)z.size(0), (int)z.size(1), (int)z.size(2),
                                      (float)eps, z.data_ptr(), dv.data_ptr(), dz.data_ptr(), stream_of(z)),
          "ebr_descent_noisy_point_bwd");
    return dz;
}

variable_list step_bwd(const Tensor& v_, const Tensor& g_, const Tensor& alpha, const Tensor& active,
                       const Tensor& rms, const Tensor& dout_, double eps) {
    RECORD_FUNCTION("ebr_fused::descent_step_project_bwd", std::vector<c10::IValue>());
    const c10::DeviceGuard on(v_.device());
    const auto st = v_.scalar_type();
    const Tensor v = dense(v_), g = dense(g_.to(st)), dout = dense(dout_.to(st));
    const Tensor dv = at::empty(v.sizes(), v.options()), dg = at::empty(v.sizes(), v.options());
    const Tensor dz = active.defined() ? at::empty(v.sizes(), v.options()) : Tensor();
    const int64_t B = v.size(0);
    check(ebr_descent_step_project_bwd(dtype_code(st), (int)B, v.numel() / B, (float)eps, v.data_ptr(), g.data_ptr(),
                                       fptr(alpha), static_cast<const uint8_t*>(vptr(active)), fptr(rms),
                                       dout.data_ptr(), dv.data_ptr(), dg.data_ptr(), vptr(dz), stream_of(v)),
          "ebr_descent_step_project_bwd");
    return {dv, dg, dz};
}

struct NoisyPoint : Function<NoisyPoint> {
    static variable_list forward(AutogradContext* ctx, const Tensor& z_, const std::optional<Tensor>& noise_,
                                 const std::optional<Tensor>& sigma_, double eps) {
        const Tensor noise = noise_.value_or(Tensor()), sigma = sigma_.value_or(Tensor());
        ctx->save_for_backward({z_});
        ctx->saved_data["eps"] = eps;
        ctx->set_materialize_grads(false);
        RECORD_FUNCTION("ebr_fused::descent_noisy_point", std::vector<c10::IValue>());
        const c10::DeviceGuard on(z_.device());
        const Tensor z = dense(z_), v = at::empty(z.sizes(), z.options());
        check(ebr_descent_noisy_point(dtype_code(z.scalar_type()), (int)z.size(0), (int)z.size(1), (int)z.size(2),
                                      (float)eps, z.data_ptr(), vptr(noise), fptr(sigma), v.data_ptr(), stream_of(z)),
              "ebr_descent_noisy_point");
        return {v};
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& g) {
        variable_list out(4);
        if (!g[0].defined()) return out;
        const Tensor z = ctx->get_saved_variables()[0];
        const double eps = ctx->saved_data["eps"].toDouble();
        if (!native(g)) return python_grads("noisy_point", 4, z, eps, g[0]);
        out[0] = noisy_bwd(z, g[0], eps);
        if (recorded({z, g[0]})) out[0] = last({out[0]})[0];
        return out;
    }
};

struct StepProject : Function<StepProject> {
    static variable_list forward(AutogradContext* ctx, const Tensor& v_, const Tensor& g_, const Tensor& alpha,
                                 const std::optional<Tensor>& z_, const std::optional<Tensor>& active_, double eps) {
        const Tensor active = active_.value_or(Tensor());
        RECORD_FUNCTION("ebr_fused::descent_step_project", std::vector<c10::IValue>());
        const c10::DeviceGuard on(v_.device());
        const auto st = v_.scalar_type();
        const Tensor v = dense(v_), g = dense(g_.to(st)), z = z_ ? dense(z_->to(st)) : Tensor();
        const int64_t B = v.size(0);
        const Tensor out = at::empty(v.sizes(), v.options()), rms = at::empty({B}, v.options().dtype(at::kFloat));
        check(ebr_descent_step_project(dtype_code(st), (int)B, v.numel() / B, (float)eps, v.data_ptr(), g.data_ptr(),
                                       fptr(alpha), vptr(z), static_cast<const uint8_t*>(vptr(active)),
                                       out.data_ptr(), static_cast<float*>(rms.data_ptr()), stream_of(v)),
              "ebr_descent_step_project");
        ctx->mark_non_differentiable({rms});
        ctx->save_for_backward({v_, g_, alpha, active, rms});
        ctx->saved_data["eps"] = eps;
        ctx->set_materialize_grads(false);
        return {out, rms};
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& gr) {
        variable_list out(6);
        if (!gr[0].defined()) return out;
        const variable_list s = ctx->get_saved_variables();
        const double eps = ctx->saved_data["eps"].toDouble();
        if (!native(gr)) return python_grads("step_project", 6, s[0], s[1], s[2], s[3], s[4], eps, gr[0]);
        variable_list d = step_bwd(s[0], s[1], s[2], s[3], s[4], gr[0], eps);
        if (recorded({s[0], s[1], gr[0]})) d = last(std::move(d));
        out[0] = d[0];
        out[1] = d[1];
        out[3] = d[2];  // undefined without a mask: no row keeps z
        return out;
    }
};

// fp32 [rows] values of a per-row scalar: a Python float as given, a tensor of the data's dtype widened. Undefined for
// what the Python layer has to look at (other dtypes and shapes, a schedule value that wants a gradient).
Tensor per_row(const py::handle& x, const Tensor& like) {
    const int64_t n = like.size(0);
    if (py::isinstance<py::float_>(x) || py::isinstance<py::int_>(x))
        return at::full({n}, x.cast<double>(), like.options().dtype(at::kFloat).requires_grad(false));
    const Tensor t = plain(x);
    if (!t.defined() || (t.requires_grad() && at::GradMode::is_enabled()) || !same_kind(t, like)) return {};
    if (t.numel() != 1 && t.numel() != n) return {};
    for (int64_t i = 1; i < t.dim(); ++i)
        if (t.size(i) != 1) return {};
    return t.detach().reshape(-1).expand({n}).to(at::kFloat).contiguous();
}

bool board(const Tensor& t) {
    return t.defined() && t.dim() == 3 && t.numel() > 0 && dtype_code(t.scalar_type()) >= 0 &&
           t.scalar_type() != at::kDouble && t.size(0) < (int64_t(1) << 31) && t.size(1) < (int64_t(1) << 31) &&
           t.size(2) < (int64_t(1) << 31);
}

// rms_norm(z) + noise * sigma; ``hnoise`` None: rms_norm alone; ``hsigma`` None: the noise as it is.
py::object noisy_point(const py::handle& hz, const py::handle& hnoise, const py::handle& hsigma, double eps) {
    const Tensor z = plain(hz);
    if (!board(z) || !plain_context()) return py::none();
    Tensor noise, sigma;
    if (!hnoise.is_none()) {
        noise = plain(hnoise);
        // noise that wants a gradient takes the Python node, which has the plain formula for it
        if (!noise.defined() || noise.sizes() != z.sizes() || noise.device() != z.device() ||
            (noise.requires_grad() && at::GradMode::is_enabled()))
            return py::none();
        noise = dense(noise.detach().to(z.scalar_type()));
        if (!hsigma.is_none()) {
            sigma = per_row(hsigma, z);
            if (!sigma.defined()) return py::none();
        }
    }
    return py::cast(NoisyPoint::apply(z, maybe(noise), maybe(sigma), eps)[0]);
}

py::object step_and_project(const py::handle& hv, const py::handle& hg, const py::handle& halpha,
                            const py::handle& hz, const py::handle& hactive, double eps) {
    const Tensor v = plain(hv), g = plain(hg), z = plain(hz);
    if (!board(v) || !g.defined() || !z.defined() || !same_kind(v, g) || !same_kind(v, z) || !plain_context())
        return py::none();
    if (g.sizes() != v.sizes() || z.sizes() != v.sizes()) return py::none();
    const Tensor alpha = per_row(halpha, v);
    if (!alpha.defined()) return py::none();
    Tensor active;
    if (!hactive.is_none()) {
        active = plain(hactive);
        if (!active.defined() || active.numel() != v.size(0) || active.device() != v.device() ||
            active.scalar_type() != at::kBool)
            return py::none();
        for (int64_t i = 1; i < active.dim(); ++i)
            if (active.size(i) != 1) return py::none();
        active = active.reshape(-1).contiguous().view(at::kByte);  // a bool is one byte, 0 or 1
    }
    return py::cast(StepProject::apply(v, g, alpha, active.defined() ? maybe(z) : std::nullopt, maybe(active), eps)[0]);
}

// ---------------------------------------------------------------------------------------------------------------------
// Linear layers with split-K weight gradients (ebr_amd/linear.py states the rule and why)
// ---------------------------------------------------------------------------------------------------------------------

constexpr int64_t MIN_ROWS_PER_SPLIT = 1024;
constexpr int64_t SPLIT8_OUTPUT = 1500000;

int64_t splits(int64_t m, int64_t outputs) {
    for (int64_t s = outputs >= SPLIT8_OUTPUT ? 8 : 16; s > 1; s /= 2)
        if (m % s == 0 && m / s >= MIN_ROWS_PER_SPLIT) return s;
    return 1;
}

// a^T b over the flattened leading dims.
Tensor weight_grad(const Tensor& a, const Tensor& b) {
    const Tensor a2 = a.reshape({-1, a.size(-1)}), b2 = b.reshape({-1, b.size(-1)});
    if (recorded({a2, b2})) return at::matmul(a2.t(), b2);
    const int64_t m = a2.size(0), n = a2.size(1), k = b2.size(1);
    const int64_t s = a2.scalar_type() == at::kBFloat16 || a2.scalar_type() == at::kHalf ? splits(m, n * k) : 1;
    if (s == 1) return at::matmul(a2.t(), b2);
    const Tensor a3 = a2.contiguous().view({s, m / s, n}).transpose(1, 2);
    const Tensor b3 = b2.contiguous().view({s, m / s, k});  // the right operand stays a contiguous batch
    const Tensor part = at::bmm(a3, b3, at::kFloat);
    const c10::DeviceGuard on(a.device());
    const Tensor out = at::empty({n, k}, a2.options().requires_grad(false));
    check(ebr_block_split_sum(dtype_code(a.scalar_type()), (int)s, n * k, fptr(part), out.data_ptr(), stream_of(a)),
          "ebr_block_split_sum");
    return out;
}

struct Linear;

struct Dgrad : Function<Dgrad> {  // dX = dY W
    static variable_list forward(AutogradContext* ctx, const Tensor& dy, const Tensor& w) {
        ctx->save_for_backward({dy, w});
        ctx->set_materialize_grads(false);
        return {at::matmul(dy, w)};
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& g);
};

struct Linear : Function<Linear> {  // Y = X W^T
    static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& w) {
        ctx->save_for_backward({x, w});
        ctx->set_materialize_grads(false);
        return {at::linear(x, w)};
    }
    // Gradients that the engine will not use are not computed.
    static variable_list backward(AutogradContext* ctx, const variable_list& g) {
        variable_list out(2);
        if (!g[0].defined()) return out;
        const bool nx = ctx->needs_input_grad(0), nw = ctx->needs_input_grad(1);
        const variable_list s = ctx->get_saved_variables();
        if (!native(g)) return python_grads("linear", 2, s[0], s[1], g[0], nx, nw);
        if (nx) out[0] = Dgrad::apply(g[0], s[1])[0];
        if (nw) out[1] = weight_grad(g[0], s[0]);
        return out;
    }
};

variable_list Dgrad::backward(AutogradContext* ctx, const variable_list& g) {
    variable_list out(2);
    if (!g[0].defined()) return out;
    const bool ndy = ctx->needs_input_grad(0), nw = ctx->needs_input_grad(1);
    const variable_list s = ctx->get_saved_variables();
    if (!native(g)) return python_grads("linear_dgrad", 2, s[0], s[1], g[0], ndy, nw);
    if (ndy) out[0] = at::GradMode::is_enabled() ? Linear::apply(g[0], s[1])[0] : at::linear(g[0], s[1]);
    if (nw) out[1] = weight_grad(s[0], g[0]);
    return out;
}

py::object linear(const py::handle& hx, const py::handle& hw) {
    const Tensor x = plain(hx), w = plain(hw);
    if (!x.defined() || !w.defined() || x.dim() < 2 || w.dim() != 2 || x.size(-1) != w.size(1) || !same_kind(x, w) ||
        x.numel() == 0 || w.numel() == 0 || !at::isFloatingType(x.scalar_type()) || !plain_context())
        return py::none();
    return py::cast(Linear::apply(x, w)[0]);
}

}  // namespace

PYBIND11_MODULE(ebr_host, m) {
    if (ebr_attn_abi_version() != EBR_ATTN_ABI_VERSION)
        throw std::runtime_error("libebr_attn.so has another ABI version than this module was built for");
    m.def("attention", &attention);
    m.def("rope_split", &rope_split);
    m.def("rope_attention", &rope_attention);
    m.def("rms_norm", &rms_norm);
    m.def("add_rms_norm", &add_rms_norm);
    m.def("swiglu", &swiglu);
    m.def("noisy_point", &noisy_point);
    m.def("step_and_project", &step_and_project);
    m.def("linear", &linear);
}
