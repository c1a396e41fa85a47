// PyTorch operators over the C ABI (include/gptoss_attn.h): argument checks, allocation, launch and the autograd node in
// native code.  Stands in for the host side of the reference's `_attention` (attention_kernel.py:220-344).
//
//   gptoss_attn::fwd, gptoss_attn::bwd   the two library calls (opaque to tracing; their shape-only implementations are
//                                        registered in attention_kernel.py)
//   gptoss_attn::attention               the differentiable call made of them
//
// Why native: the calls of a training step on short rows take less time on the GPU than their host side took in Python
// (an autograd.Function around two Python custom operators and a ctypes call each: 250 us per forward + backward
// whatever the size; the same calls through this file take 60 to 90 us for two rows of 383 tokens, 88 for a sliding-window layer of
// 4096, of which 64 and 83 are kernels, and a decoding step 13 us instead of 44).  This file is built against torch; the kernels are not.
#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <pybind11/pybind11.h>
#include <torch/csrc/autograd/autograd_not_implemented_fallback.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/library.h>

#include "../../include/gptoss_attn.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;
using c10::SymInt;

constexpr int64_t kMaxSeqStride = int64_t(1) << 24;   // elements; the library refuses larger sequence strides (ERR_STRIDE)

// The kernels need unit stride along head_dim, 16-byte aligned rows and a sequence stride of at least head_dim and at most
// 2^24 elements; anything else is copied.
Tensor row_contiguous(const Tensor &t, int64_t seq_dim) {
    const auto st = t.strides();
    const int64_t eb = t.element_size();
    const bool ok = st[3] == 1 && (st[0] * eb) % 16 == 0 && (st[1] * eb) % 16 == 0 && (st[2] * eb) % 16 == 0 &&
                    reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0 && st[seq_dim] >= t.size(3) && st[seq_dim] <= kMaxSeqStride;
    return ok ? t : t.contiguous();
}

void require_on(const Tensor &q, const char *name, const Tensor &t) {
    TORCH_CHECK(t.device() == q.device(), name, " is on ", t.device(), " but q is on ", q.device(), ": every tensor must be on q's GPU");
}

// What can be looked at without a size (a traced call's sizes are symbols, and reading one as a number would tie the traced
// program to it).
void check_kinds(const Tensor &q, const Tensor &k, const Tensor &v, bool allow_cast) {
    TORCH_CHECK(q.is_cuda() && k.is_cuda() && v.is_cuda(), "gptoss attention runs on the GPU only (HIP kernels); got a CPU tensor");
    const auto dt = q.scalar_type();
    const bool ok = dt == at::kBFloat16 || dt == at::kFloat || (allow_cast && dt == at::kHalf);
    TORCH_CHECK(ok && k.scalar_type() == dt && v.scalar_type() == dt, "unsupported dtypes ", dt, "/", k.scalar_type(), "/", v.scalar_type(),
                ": q, k, v must all be bfloat16 or all be float32");
    TORCH_CHECK(q.dim() == 4 && k.dim() == 4 && v.dim() == 4, "q must be (B,H,S,D) and k, v (B,G,S_kv,D)");
}

void check_inputs(const Tensor &q, const Tensor &k, const Tensor &v, const OptTensor &sinks) {
    check_kinds(q, k, v, false);
    TORCH_CHECK(k.sizes() == v.sizes() && q.size(0) == k.size(0) && q.size(3) == k.size(3), "shape mismatch: q ", q.sizes(), ", k ", k.sizes(),
                ", v ", v.sizes());
    if (sinks) {
        TORCH_CHECK(sinks->numel() == q.size(1), "sinks must hold one logit per query head");
        require_on(q, "sinks", *sinks);
    }
    require_on(q, "k", k);
    require_on(q, "v", v);
}

// Memory for a result or for scratch, without the dispatcher: every value of it is written before it is read.  A call's allocations are a tenth of its host time.
Tensor new_tensor(at::IntArrayRef sizes, at::ScalarType dtype, const Tensor &like) {
    return Tensor(at::detail::empty_cuda(sizes, dtype, like.device(), std::nullopt));
}

void set(gptoss_attn_strides &s, const Tensor &t, bool bshd) {
    s.b = t.stride(0);
    s.h = t.stride(bshd ? 2 : 1);
    s.s = t.stride(bshd ? 1 : 2);
}

// The parameter block and the tensors it points into.
struct Call {
    gptoss_attn_params p{};
    Tensor q, k, v, sinks, seqlens, doc_start, q_offset_dev;
    int sinks_dtype = GPTOSS_ATTN_FP32;
};

void fill(Call &c, const Tensor &q, const Tensor &k, const Tensor &v, const OptTensor &sinks, double sm_scale, int64_t window, int64_t q_offset,
          const OptTensor &seqlens, const OptTensor &doc_start, const OptTensor &q_offset_dev) {
    check_inputs(q, k, v, sinks);
    c.q = row_contiguous(q, 2);
    c.k = row_contiguous(k, 2);
    c.v = row_contiguous(v, 2);
    gptoss_attn_params &p = c.p;
    p.struct_size = sizeof(p);
    p.dtype = q.scalar_type() == at::kFloat ? GPTOSS_ATTN_FP32 : GPTOSS_ATTN_BF16;
    p.B = q.size(0);
    p.H = q.size(1);
    p.Sq = q.size(2);
    p.D = q.size(3);
    p.G = k.size(1);
    p.Skv = k.size(2);
    p.window = window;
    p.q_offset = q_offset;
    p.scale = sm_scale;
    p.q = c.q.const_data_ptr();
    p.k = c.k.const_data_ptr();
    p.v = c.v.const_data_ptr();
    set(p.q_stride, c.q, false);
    set(p.k_stride, c.k, false);
    set(p.v_stride, c.v, false);
    if (sinks) {
        const bool bf16 = sinks->scalar_type() == at::kBFloat16;      // read as they are: no converted copy
        c.sinks = (bf16 ? *sinks : sinks->to(at::kFloat)).contiguous();
        c.sinks_dtype = bf16 ? GPTOSS_ATTN_BF16 : GPTOSS_ATTN_FP32;
        p.sinks = static_cast<const float *>(c.sinks.const_data_ptr());
    }
    if (seqlens) {
        c.seqlens = seqlens->to(q.device(), at::kInt).contiguous();
        TORCH_CHECK(c.seqlens.numel() == q.size(0), "seqlens must hold one length per batch row");
        p.seqlens = c.seqlens.const_data_ptr<int32_t>();
    }
    if (doc_start) {
        c.doc_start = doc_start->to(q.device(), at::kInt).contiguous();
        TORCH_CHECK(c.doc_start.dim() == 2 && c.doc_start.size(0) == q.size(0) && c.doc_start.size(1) == q.size(2),
                    "doc_start must be (B, S): the first token index of each query's document");
        p.doc_start = c.doc_start.const_data_ptr<int32_t>();
    }
    if (q_offset_dev) {
        TORCH_CHECK(q_offset_dev->device() == q.device() && q_offset_dev->numel() == 1 && !q_offset_dev->is_floating_point(),
                    "q_offset_dev must be a one-element integer tensor on the same device as q");
        c.q_offset_dev = q_offset_dev->reshape({1}).to(at::kInt).contiguous();
        p.q_offset_dev = c.q_offset_dev.const_data_ptr<int32_t>();
    }
}

void *stream_of(const Call &c) { return c10::hip::getCurrentHIPStream(c.q.device().index()).stream(); }

// A failed library call is the package's GptossAttnError wherever it happens: in a call, a backward or a traced program.
void check(const char *name, int rc) {
    if (rc == 0) return;
    const pybind11::gil_scoped_acquire gil;
    const pybind11::object type = pybind11::module_::import("oregon_gpt_oss_patching_amd._lib").attr("GptossAttnError");
    PyErr_SetObject(type.ptr(), type(name, rc, gptoss_attn_status_string(rc)).ptr());
    throw pybind11::error_already_set();
}

std::tuple<Tensor, Tensor> fwd(const Tensor &q, const Tensor &k, const Tensor &v, const OptTensor &sinks, double sm_scale, int64_t window,
                               int64_t q_offset, const OptTensor &seqlens, const OptTensor &doc_start, const OptTensor &q_offset_dev) {
    const c10::OptionalDeviceGuard guard(q.device());
    Call c;
    fill(c, q, k, v, sinks, sm_scale, window, q_offset, seqlens, doc_start, q_offset_dev);
    Tensor o = new_tensor({q.size(0), q.size(2), q.size(1), q.size(3)}, q.scalar_type(), q);
    Tensor lse = new_tensor({q.size(0), q.size(1), q.size(2)}, at::kFloat, q);
    c.p.o = o.data_ptr();
    c.p.lse = lse.data_ptr<float>();
    set(c.p.o_stride, o, true);
    // partial results of few queries' or few heads' rows, cut over their keys; records of float32 operands
    const size_t need = c.p.dtype == GPTOSS_ATTN_FP32 ? gptoss_attn_split_bytes(&c.p, 0) : gptoss_attn_fwd_workspace_bytes(&c.p);
    const Tensor scratch = need ? new_tensor({static_cast<int64_t>(need / sizeof(float))}, at::kFloat, q) : Tensor();
    check("gptoss_attn_fwd", gptoss_attn_fwd_scratch(&c.p, c.sinks_dtype, need ? scratch.data_ptr() : nullptr, need, stream_of(c)));
    return {o, lse};
}

// (an operator cannot return None: an empty dsinks stands for "not requested"; dsinks_as_sinks: in bf16 where the logits are)
std::tuple<Tensor, Tensor, Tensor, Tensor> bwd(const Tensor &q, const Tensor &k, const Tensor &v, const OptTensor &sinks, const Tensor &o_,
                                               const Tensor &lse_, const Tensor &d_o_, double sm_scale, int64_t window, int64_t q_offset,
                                               const OptTensor &seqlens, const OptTensor &doc_start, bool need_dsinks, const OptTensor &q_offset_dev,
                                               bool dsinks_as_sinks) {
    const c10::OptionalDeviceGuard guard(q.device());
    Call c;
    fill(c, q, k, v, sinks, sm_scale, window, q_offset, seqlens, doc_start, q_offset_dev);
    // the saved tensors and dO reach the kernels as raw pointers: on q's GPU and in the layout the kernels address
    const int64_t b = q.size(0), h = q.size(1), s = q.size(2), d = q.size(3);
    for (const auto &[name, t] : {std::pair<const char *, const Tensor &>("o", o_), {"lse", lse_}, {"d_o", d_o_}}) require_on(q, name, t);
    for (const auto &[name, t] : {std::pair<const char *, const Tensor &>("o", o_), {"d_o", d_o_}}) {
        TORCH_CHECK(t.scalar_type() == q.scalar_type(), name, " has dtype ", t.scalar_type(), ", expected q's dtype ", q.scalar_type());
        TORCH_CHECK(t.sizes() == at::IntArrayRef({b, s, h, d}), name, " must be (B, S, H, D) = ", at::IntArrayRef({b, s, h, d}), ", got ", t.sizes());
    }
    TORCH_CHECK(lse_.scalar_type() == at::kFloat, "lse must be float32, got ", lse_.scalar_type());
    TORCH_CHECK(lse_.sizes() == at::IntArrayRef({b, h, s}), "lse must be (B, H, S) = ", at::IntArrayRef({b, h, s}), ", got ", lse_.sizes());
    const Tensor o = row_contiguous(o_, 1), d_o = row_contiguous(d_o_, 1), lse = lse_.contiguous();

    Tensor dq = new_tensor({b, h, s, d}, q.scalar_type(), q), dk = new_tensor(k.sizes(), k.scalar_type(), q), dv = new_tensor(v.sizes(), v.scalar_type(), q);
    const bool bf16_dsinks = dsinks_as_sinks && c.sinks_dtype == GPTOSS_ATTN_BF16;
    Tensor dsinks = new_tensor({need_dsinks ? h : 0}, bf16_dsinks ? at::kBFloat16 : at::kFloat, q);
    // scratch: the row statistics, then the dK/dV partial sums of split key blocks or the window kernel's shares; the records of float32
    // operands as bf16 terms are a scratch of their own, and with them the first is two floats per row
    const size_t records = gptoss_attn_split_bytes(&c.p, 1);
    Tensor scratch = new_tensor({records ? 2 * b * h * s : static_cast<int64_t>(gptoss_attn_bwd_workspace_bytes(&c.p) / sizeof(float))}, at::kFloat, q);
    gptoss_attn_params &p = c.p;
    p.o = const_cast<void *>(o.const_data_ptr());             // (read only here)
    p.lse = const_cast<float *>(lse.const_data_ptr<float>());
    p.d_o = d_o.const_data_ptr();
    p.dq = dq.data_ptr();
    p.dk = dk.data_ptr();
    p.dv = dv.data_ptr();
    p.dsinks = need_dsinks ? static_cast<float *>(dsinks.data_ptr()) : nullptr;
    p.delta = scratch.data_ptr<float>();
    set(p.o_stride, o, true);
    set(p.do_stride, d_o, true);
    set(p.dq_stride, dq, false);
    set(p.dk_stride, dk, false);
    set(p.dv_stride, dv, false);
    const Tensor split = records ? new_tensor({static_cast<int64_t>(records / sizeof(float))}, at::kFloat, q) : Tensor();
    check("gptoss_attn_bwd", gptoss_attn_bwd_scratch(&c.p, c.sinks_dtype, bf16_dsinks ? GPTOSS_ATTN_BF16 : GPTOSS_ATTN_FP32,
                                                     records ? split.data_ptr() : nullptr, records, stream_of(c)));
    return {dq, dk, dv, dsinks};
}

// The two operators through the dispatcher (tracing modes see them).
std::tuple<Tensor, Tensor> call_fwd(const Tensor &q, const Tensor &k, const Tensor &v, const OptTensor &sinks, double sm_scale, SymInt window,
                                    SymInt q_offset, const OptTensor &seqlens, const OptTensor &doc_start, const OptTensor &q_offset_dev) {
    static const auto op = c10::Dispatcher::singleton().findSchemaOrThrow("gptoss_attn::fwd", "").typed<decltype(call_fwd)>();
    return op.call(q, k, v, sinks, sm_scale, window, q_offset, seqlens, doc_start, q_offset_dev);
}
std::tuple<Tensor, Tensor, Tensor, Tensor> call_bwd(const Tensor &q, const Tensor &k, const Tensor &v, const OptTensor &sinks, const Tensor &o,
                                                    const Tensor &lse, const Tensor &d_o, double sm_scale, SymInt window, SymInt q_offset,
                                                    const OptTensor &seqlens, const OptTensor &doc_start, bool need_dsinks,
                                                    const OptTensor &q_offset_dev, bool dsinks_as_sinks) {
    static const auto op = c10::Dispatcher::singleton().findSchemaOrThrow("gptoss_attn::bwd", "").typed<decltype(call_bwd)>();
    return op.call(q, k, v, sinks, o, lse, d_o, sm_scale, window, q_offset, seqlens, doc_start, need_dsinks, q_offset_dev, dsinks_as_sinks);
}

OptTensor optional_of(const Tensor &t) { return t.defined() ? OptTensor(t) : OptTensor(); }
Tensor tensor_of(const OptTensor &t) { return t ? *t : Tensor(); }

// float16 tensors are rounded to bfloat16 on the way in and the results cast back.
struct AttentionFunction : public torch::autograd::Function<AttentionFunction> {
    static Tensor forward(torch::autograd::AutogradContext *ctx, const Tensor &q_, const Tensor &k_, const Tensor &v_, const OptTensor &sinks,
                          double sm_scale, SymInt window, SymInt q_offset, const OptTensor &seqlens, const OptTensor &doc_start,
                          const OptTensor &q_offset_dev) {
        const at::AutoDispatchBelowADInplaceOrView below;
        const auto dtype = q_.scalar_type();
        Tensor q = q_, k = k_, v = v_;
        if (dtype == at::kHalf) {
            q = q.to(at::kBFloat16);
            k = k.to(at::kBFloat16);
            v = v.to(at::kBFloat16);
        }
        // converted once for both directions (and what is converted is a copy: the caller may move its int64 position on before
        // the backward); what is no offset at all is refused by the forward operator
        const OptTensor start = q_offset_dev && !q_offset_dev->is_floating_point() ? OptTensor(q_offset_dev->to(at::kInt)) : q_offset_dev;
        const OptTensor lens = seqlens ? OptTensor(seqlens->to(q.device(), at::kInt).contiguous()) : OptTensor();
        const OptTensor docs = doc_start ? OptTensor(doc_start->to(q.device(), at::kInt).contiguous()) : OptTensor();
        auto [o, lse] = call_fwd(q, k, v, sinks, sm_scale, window, q_offset, lens, docs, start);
        ctx->save_for_backward({q, k, v, tensor_of(sinks), o, lse, tensor_of(lens), tensor_of(docs), tensor_of(start)});
        ctx->saved_data["sm_scale"] = sm_scale;
        ctx->saved_data["window"] = window;
        ctx->saved_data["q_offset"] = q_offset;
        ctx->saved_data["half"] = dtype == at::kHalf;
        ctx->saved_data["dsinks"] = sinks && sinks->requires_grad();
        return dtype == at::kHalf ? o.to(dtype) : o;
    }

    static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const Tensor &q = saved[0], &sinks = saved[3];
        const bool half = ctx->saved_data["half"].toBool(), need_dsinks = ctx->saved_data["dsinks"].toBool();
        // a first-order backward needs no autograd bookkeeping; under create_graph the operator records that it has no second derivative
        std::optional<at::AutoDispatchBelowADInplaceOrView> below;
        if (!at::GradMode::is_enabled()) below.emplace();
        auto [dq, dk, dv, dsinks] = call_bwd(q, saved[1], saved[2], optional_of(sinks), saved[4], saved[5],
                                             grads[0].scalar_type() == q.scalar_type() ? grads[0] : grads[0].to(q.scalar_type()),
                                             ctx->saved_data["sm_scale"].toDouble(), ctx->saved_data["window"].toSymInt(),
                                             ctx->saved_data["q_offset"].toSymInt(), optional_of(saved[6]), optional_of(saved[7]), need_dsinks,
                                             optional_of(saved[8]), true);
        if (half) {
            dq = dq.to(at::kHalf);
            dk = dk.to(at::kHalf);
            dv = dv.to(at::kHalf);
        }
        // (a logit per head in one dimension, as a rule: dsinks is what it has to be)
        if (!need_dsinks) dsinks = Tensor();
        else if (dsinks.scalar_type() != sinks.scalar_type() || sinks.dim() != 1) dsinks = dsinks.to(sinks.scalar_type()).view_as(sinks);
        return {dq, dk, dv, dsinks, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

Tensor attention(const Tensor &q, const Tensor &k, const Tensor &v, const OptTensor &sinks, double sm_scale, SymInt window, SymInt q_offset,
                 const OptTensor &seqlens, const OptTensor &doc_start, const OptTensor &q_offset_dev) {
    check_kinds(q, k, v, true);        // (the shapes: gptoss_attn::fwd)
    // Nothing to differentiate (inference): no node, nothing saved; a microsecond of a decoding step's twelve.  (Dual tensors take the
    // node, which refuses them.)
    bool inference = q.scalar_type() != at::kHalf;
    for (const Tensor *t : {&q, &k, &v, sinks ? &*sinks : &q})
        inference = inference && !(at::GradMode::is_enabled() && t->requires_grad()) && !t->_fw_grad(0).defined();
    if (inference) {
        const at::AutoDispatchBelowADInplaceOrView below;
        return std::get<0>(call_fwd(q, k, v, sinks, sm_scale, window, q_offset, seqlens, doc_start, q_offset_dev));
    }
    return AttentionFunction::apply(q, k, v, sinks, sm_scale, window, q_offset, seqlens, doc_start, q_offset_dev);
}

// (B, S) int32 document starts of packed rows, see gptoss_attn_doc_start.
Tensor doc_start(const Tensor &position_ids_) {
    TORCH_CHECK(position_ids_.dim() == 2 && (position_ids_.scalar_type() == at::kLong || position_ids_.scalar_type() == at::kInt),
                "position_ids must be (B, S) of int64 or int32");
    const c10::OptionalDeviceGuard guard(position_ids_.device());
    const Tensor pos = position_ids_.size(1) > 1 && position_ids_.stride(1) != 1 ? position_ids_.contiguous() : position_ids_;
    Tensor out = at::empty(pos.sizes(), pos.options().dtype(at::kInt));
    if (pos.numel() == 0) return out;
    check("gptoss_attn_doc_start", gptoss_attn_doc_start(pos.const_data_ptr(), static_cast<int>(pos.element_size()), static_cast<int>(pos.size(0)),
                                                         static_cast<int>(pos.size(1)), pos.stride(0), out.data_ptr<int32_t>(),
                                                         c10::hip::getCurrentHIPStream(pos.device().index()).stream()));
    return out;
}

// Function transforms have no rule for the autograd node; without this vmap would run it slice by slice behind the caller's back.
void refuse_vmap(const c10::OperatorHandle &, torch::jit::Stack *) {
    TORCH_CHECK(false, "gptoss attention cannot be vmapped: its tensors have a batch dimension of their own");
}

}  // namespace

TORCH_LIBRARY(gptoss_attn, m) {
    m.def("fwd(Tensor q, Tensor k, Tensor v, Tensor? sinks, float sm_scale, SymInt window, SymInt q_offset, Tensor? seqlens, Tensor? doc_start, "
          "Tensor? q_offset_dev=None) -> (Tensor, Tensor)");
    m.def("bwd(Tensor q, Tensor k, Tensor v, Tensor? sinks, Tensor o, Tensor lse, Tensor d_o, float sm_scale, SymInt window, SymInt q_offset, "
          "Tensor? seqlens, Tensor? doc_start, bool need_dsinks, Tensor? q_offset_dev=None, bool dsinks_as_sinks=False) -> (Tensor, Tensor, Tensor, Tensor)");
    m.def("doc_start(Tensor position_ids) -> Tensor");
    m.def("attention(Tensor q, Tensor k, Tensor v, Tensor? sinks, float sm_scale, SymInt window, SymInt q_offset, Tensor? seqlens, Tensor? doc_start, "
          "Tensor? q_offset_dev=None) -> Tensor", &attention);
}
TORCH_LIBRARY_IMPL(gptoss_attn, CUDA, m) {
    m.impl("fwd", &fwd);
    m.impl("bwd", &bwd);
    m.impl("doc_start", &doc_start);
}
TORCH_LIBRARY_IMPL(gptoss_attn, Autograd, m) {
    m.impl("fwd", torch::autograd::autogradNotImplementedFallback());
    m.impl("bwd", torch::autograd::autogradNotImplementedFallback());
}
TORCH_LIBRARY_IMPL(gptoss_attn, FuncTorchBatched, m) {
    m.impl("attention", torch::CppFunction::makeFromBoxedFunction<&refuse_vmap>());
}
