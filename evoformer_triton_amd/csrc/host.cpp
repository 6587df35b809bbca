// The host side of the operator in C++: what a call does between Python and the C ABI - looking the
// tensors over, allocating results and scratch with torch, the autograd node - without the interpreter.
//
// A small call is bound by its host, not by its kernels: through Python (an autograd.Function, ctypes
// structures, the backward taking the GIL in the engine's thread) a forward took 26 us and a forward +
// backward 165 us of host time, the kernels of a small step 30 us.  The nodes below do the same work
// in C++; the backward runs in the engine's thread without the GIL.
//
// A function here returns None for a call it does not take (tensors that are not plain GPU tensors, head
// dims that need padding, empty problems, anything invalid): the caller in Python then goes its own
// way, which also words the error messages.
#include <ATen/ATen.h>
#include <ATen/autocast_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/utils/pybind.h>

#include <optional>
#include <string>
#include <vector>

#include "evoattn.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;
using torch::autograd::AutogradContext;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;
using c10::impl::tls_local_dispatch_key_set;

void check(int rc, const char *where) {
    TORCH_CHECK(rc == EVO_OK, where, " failed: ", evoattn_strerror(rc), " (code ", rc, ")");
}

int evo_dtype(at::ScalarType t) {
    switch (t) {
        case at::kBFloat16: return EVO_BF16;
        case at::kHalf: return EVO_F16;
        case at::kFloat: return EVO_F32;
        default: return EVO_NONE;
    }
}

bool head_dim_built(int64_t D) { return D == 8 || D == 16 || D == 32 || D == 64 || D == 128; }

// Whether `t` carries a tangent of forward-mode differentiation.  No node here has a formula for it, and launches drop it without a
// word, which counts as a tangent of zero.
bool dual(const Tensor &t) { return t.defined() && t._fw_grad(/*level=*/0).defined(); }

// An ordinary tensor with memory of its own kind: no subclass or mode with a dispatch in Python, no functorch wrapper,
// no tangent and no lazily negated or conjugated view, whose data pointer would not be what it stands for.
bool plain(const Tensor &t) {
    static const auto special = c10::DispatchKeySet({
        c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::FuncTorchBatched,
        c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate,
        c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor});
    return t.layout() == at::kStrided && !t.key_set().has_any(special) && !dual(t);
}

// No mode that has to see the call itself: a dispatch mode in Python, functorch, or torch.jit's tracer, which records the operators
// called here but none of the launches.
bool plain_modes() {
    static const auto modes = c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchDynamicLayerFrontMode, c10::DispatchKey::Tracer});
    return !tls_local_dispatch_key_set().included_.has_any(modes);
}

hipStream_t stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

Tensor scratch(size_t bytes, const Tensor &like) {
    return at::empty({(int64_t)std::max<size_t>(bytes, 256)}, like.options().dtype(at::kByte));
}

size_t align256(size_t n) { return (n + 255) / 256 * 256; }

// What a call's backward needs besides the tensors: the parameter block (its pointers are set anew) and the
// caller's mask and bias as they came, whose shape and dtype their gradients take.
struct Call {
    EvoAttnParams p;
    int64_t mask_b, mask_s, bias_b;
    at::ScalarType mask_dtype, bias_dtype;
    bool gated;
};

// A mask and a bias of the right shapes and dtypes into the parameter block: their addresses and strides.
void point_at(EvoAttnParams &p, Tensor &mask, Tensor &bias) {
    if (mask.defined()) {
        if (mask.stride(4) != 1) mask = mask.contiguous();
        p.mask_stride_b = mask.size(0) == p.B && p.B > 1 ? mask.stride(0) : 0;
        p.mask_stride_s = mask.size(1) == p.S && p.S > 1 ? mask.stride(1) : 0;
        p.mask = mask.data_ptr();
    }
    if (bias.defined()) {
        if (bias.stride(4) != 1 || bias.stride(3) < p.N) bias = bias.contiguous();
        p.bias_stride_b = bias.size(0) == p.B && p.B > 1 ? bias.stride(0) : 0;
        p.bias_stride_h = bias.stride(2);
        p.bias_stride_row = bias.stride(3);
        p.bias = bias.data_ptr();
    }
}

// The mask and the bias as the kernels read them; false where they do not fit the shape of Q.
bool operands(Call &c, const Tensor &q, OptTensor &mask, OptTensor &bias) {
    EvoAttnParams &p = c.p;
    p.mask_kind = EVO_MASK_NONE;
    p.bias_dtype = EVO_NONE;
    const auto qdev = q.device();
    if (mask && mask->defined()) {
        Tensor m = *mask;
        if (!plain(m) || m.device() != qdev || m.dim() != 5) return false;
        const auto sz = m.sizes();
        if (sz[2] != 1 || sz[3] != 1 || sz[4] != p.N || (sz[0] != 1 && sz[0] != p.B) || (sz[1] != 1 && sz[1] != p.S)) return false;
        c.mask_b = sz[0];
        c.mask_s = sz[1];
        c.mask_dtype = m.scalar_type();
        switch (m.scalar_type()) {
            case at::kBool: case at::kByte: p.mask_kind = EVO_MASK_BOOL; break;
            case at::kFloat: p.mask_kind = EVO_MASK_F32; break;
            case at::kBFloat16: p.mask_kind = EVO_MASK_BF16; break;
            case at::kHalf: p.mask_kind = EVO_MASK_F16; break;
            default:
                if (!at::isFloatingType(m.scalar_type()) && !at::isIntegralType(m.scalar_type(), true)) return false;
                p.mask_kind = m.is_floating_point() ? EVO_MASK_F32 : EVO_MASK_BOOL;
                m = m.is_floating_point() ? m.to(at::kFloat) : m.ne(0);
        }
        mask = m;
    } else {
        mask = Tensor();
    }
    if (bias && bias->defined()) {
        Tensor b = *bias;
        if (!plain(b) || b.device() != qdev || b.dim() != 5 || !b.is_floating_point()) return false;
        const auto sz = b.sizes();
        if (sz[1] != 1 || sz[2] != p.H || sz[3] != p.N || sz[4] != p.N || (sz[0] != 1 && sz[0] != p.B)) return false;
        c.bias_b = sz[0];
        c.bias_dtype = b.scalar_type();
        if (b.scalar_type() != at::kFloat && b.scalar_type() != q.scalar_type()) b = b.to(at::kFloat);
        p.bias_dtype = evo_dtype(b.scalar_type());
        bias = b;
    } else {
        bias = Tensor();
    }
    point_at(p, *mask, *bias);
    return true;
}

// LSE and the prepared operands share one allocation: [LSE | prep].
struct Aux {
    size_t lse_bytes;
    explicit Aux(const EvoAttnParams &p) : lse_bytes(align256((size_t)p.B * p.H * p.S * p.N * sizeof(float))) {}
    void place(EvoAttnParams &p, const Tensor &aux) const {
        char *base = (char *)aux.data_ptr();
        p.lse = (float *)base;
        p.prep = base + lse_bytes;
        p.prep_bytes = (size_t)aux.numel() - lse_bytes;
    }
};

Tensor finish_dbias(Tensor d, const Call &c) {
    const EvoAttnParams &p = c.p;
    d = d.view({p.B, 1, p.H, p.N, p.N});
    if (c.bias_b == 1 && p.B > 1) d = d.sum(0, true);
    return d.scalar_type() == c.bias_dtype ? d : d.to(c.bias_dtype);
}

Tensor finish_dmask(Tensor d, const Call &c) {
    const EvoAttnParams &p = c.p;
    d = d.view({p.B, p.S, 1, 1, p.N});
    if (c.mask_b == 1 && p.B > 1) d = d.sum(0, true);
    if (c.mask_s == 1 && p.S > 1) d = d.sum(1, true);
    return d.scalar_type() == c.mask_dtype ? d : d.to(c.mask_dtype);
}

// The backward's scratch and results beside dQ, dK, dV: allocates dBias, dMask and the workspace, sets their
// pointers in `p`, and enqueues the backward.  `p` holds the mask and the bias as the forward read them, `mask` and `bias` are
// what was saved of them: hooks on saved tensors may hand back copies, laid out otherwise, for which the forward's prepared
// operands are made anew (their form depends on strides and alignment).
void enqueue_backward(EvoAttnParams &p, const Tensor &like, Tensor mask, Tensor bias, bool want_dbias, bool want_dmask, Tensor &dbias,
                      Tensor &dmask) {
    const EvoAttnParams fwd = p;
    point_at(p, mask, bias);
    const bool same = p.mask == fwd.mask && p.bias == fwd.bias && p.mask_stride_b == fwd.mask_stride_b && p.mask_stride_s == fwd.mask_stride_s &&
                      p.bias_stride_b == fwd.bias_stride_b && p.bias_stride_h == fwd.bias_stride_h && p.bias_stride_row == fwd.bias_stride_row;
    Tensor prep;
    if (!same) {
        prep = scratch(evoattn_prep_bytes(&p), like);
        p.prep = prep.data_ptr();
        p.prep_bytes = (size_t)prep.numel();
    }
    if (want_dbias) {
        dbias = at::empty({p.B, p.H, p.N, p.N}, bias.options());
        p.dbias = dbias.data_ptr();
        p.dbias_dtype = p.bias_dtype;
    }
    if (want_dmask) {
        dmask = at::empty({p.B, p.S, p.N}, like.options().dtype(at::kFloat));
        p.dmask = (float *)dmask.data_ptr();
    }
    Tensor ws = scratch(evoattn_bwd_workspace_bytes(&p), like);
    p.workspace = ws.data_ptr();
    p.workspace_bytes = (size_t)ws.numel();
    if (same) p.flags |= EVO_FLAG_PREP_VALID;
    check(evoattn_bwd(&p, stream_of(like)), "evoattn_bwd");
}

// Gradients of gradients are not formed: as torch's once_differentiable does, results of a backward that is itself
// recorded become inputs of a node that says so when it is differentiated.
variable_list once_differentiable(variable_list outs, bool recorded) {
    if (!recorded) return outs;
    std::vector<size_t> at_;
    variable_list defined;
    for (size_t i = 0; i < outs.size(); ++i)
        if (outs[i].defined()) {
            at_.push_back(i);
            defined.push_back(outs[i].detach().set_requires_grad(true));
        }
    torch::autograd::DelayedError err("trying to differentiate twice a function that was marked with @once_differentiable",
                                      (int64_t)defined.size());
    variable_list wrapped = err.apply(std::move(defined));
    for (size_t i = 0; i < at_.size(); ++i) outs[at_[i]] = wrapped[i];
    return outs;
}

// A node whose saved tensors lie in one list.
struct SavingNode : Node {
    std::vector<SavedVariable> saved;
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        for (auto &s : saved) s.reset_data();
    }
    void save(const Tensor &t, bool is_output = false) { saved.emplace_back(t, is_output); }
    template <typename... T>
    static bool wanted(const T &...t) {
        return at::GradMode::is_enabled() && ((t.defined() && t.requires_grad()) || ...);
    }
};

template <typename N, typename... T>
std::shared_ptr<N> make_node(const T &...inputs) {
    std::shared_ptr<N> node(new N(), torch::autograd::deleteNode);
    node->set_next_edges(torch::autograd::collect_next_edges(inputs...));
    return node;
}

// ------------------------------------------------------------------ attention

struct AttentionNode : SavingNode {
    Call c{};
    std::string name() const override { return c.gated ? "GatedAttentionBackward" : "EvoformerAttentionBackward"; }

    // grads[0]: the gradient of the output; results: Q, K, V, mask, bias, gate
    variable_list apply(variable_list &&grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        const bool rec = at::GradMode::is_enabled();
        variable_list out(6);
        {
            at::AutoDispatchBelowADInplaceOrView guard;
            const Tensor q = saved[0].unpack().contiguous(), k = saved[1].unpack().contiguous(), v = saved[2].unpack().contiguous(),
                         mask = saved[3].unpack(), bias = saved[4].unpack(), aux = saved[5].unpack(),
                         o = saved[6].unpack(shared_from_this()).contiguous();
            const Tensor gate = c.gated ? saved[7].unpack().contiguous() : Tensor();
            c10::DeviceGuard on(q.device());
            Tensor dO = grads[0].defined() ? grads[0].contiguous() : at::zeros_like(q);
            if (dO.scalar_type() != q.scalar_type()) dO = dO.to(q.scalar_type());
            EvoAttnParams p = c.p;
            Aux(p).place(p, aux);
            p.q = q.data_ptr();
            p.k = k.data_ptr();
            p.v = v.data_ptr();
            p.dout = dO.data_ptr();
            Tensor dbias, dmask;
            for (int i = 0; i < 3; ++i) out[i] = at::empty_like(q);
            p.dq = out[0].data_ptr();
            p.dk = out[1].data_ptr();
            p.dv = out[2].data_ptr();
            if (c.gated) {   // o is the gated output, dO its gradient
                out[5] = at::empty_like(q);
                p.o = nullptr;
                p.o_gated = o.data_ptr();
                p.gate = gate.data_ptr();
                p.dgate = out[5].data_ptr();
            } else {
                p.o = o.data_ptr();
            }
            const bool want_dmask = mask.defined() && mask.is_floating_point() && task_should_compute_output(3);
            const bool want_dbias = bias.defined() && task_should_compute_output(4);
            enqueue_backward(p, q, mask, bias, want_dbias, want_dmask, dbias, dmask);
            if (want_dbias) out[4] = finish_dbias(dbias, c);
            if (want_dmask) out[3] = finish_dmask(dmask, c);
        }
        return once_differentiable(std::move(out), rec);
    }
};

// The attention on dense [B,S,N,H,D] tensors with the reference's flat-reshape heads or (per_head) true ones, with a
// gate sigmoid(gate) * O; none where this path does not take the call.
OptTensor attention(const Tensor &Q, const Tensor &K, const Tensor &V, OptTensor mask, OptTensor bias, const OptTensor &gate, bool per_head,
                    int64_t flags) {
    if (!plain(Q) || !plain(K) || !plain(V) || !Q.is_cuda() || Q.dim() != 5 || !plain_modes()) return std::nullopt;
    if (!K.sizes().equals(Q.sizes()) || !V.sizes().equals(Q.sizes()) || K.device() != Q.device() || V.device() != Q.device()) return std::nullopt;
    const auto dt = Q.scalar_type();
    if (K.scalar_type() != dt || V.scalar_type() != dt || evo_dtype(dt) == EVO_NONE || Q.numel() == 0 || !head_dim_built(Q.size(4)))
        return std::nullopt;
    for (int i = 0; i < 5; ++i)
        if (Q.size(i) > INT32_MAX) return std::nullopt;
    const bool gated = gate && gate->defined();
    if (gated && (!plain(*gate) || !gate->sizes().equals(Q.sizes()) || gate->scalar_type() != dt || gate->device() != Q.device())) return std::nullopt;

    Call c{};
    EvoAttnParams &p = c.p;
    p.B = (int32_t)Q.size(0);
    p.S = (int32_t)Q.size(1);
    p.N = (int32_t)Q.size(2);
    p.H = (int32_t)Q.size(3);
    p.D = (int32_t)Q.size(4);
    p.dtype = evo_dtype(dt);
    p.dbias_dtype = EVO_F32;
    p.flags = (int32_t)flags;
    p.scale = (float)(1.0 / std::sqrt((double)p.D));
    const int64_t row = (int64_t)p.N * p.D;
    p.stride_b = (int64_t)p.S * p.H * row;
    p.stride_h = per_head ? p.D : p.S * row;
    p.stride_s = per_head ? p.H * row : row;
    p.stride_n = per_head ? (int64_t)p.H * p.D : p.D;
    c.gated = gated;

    OptTensor mask_in = mask, bias_in = bias;
    const Tensor mask0 = mask ? *mask : Tensor(), bias0 = bias ? *bias : Tensor(), gate0 = gated ? *gate : Tensor();
    const bool wanted = SavingNode::wanted(Q, K, V, mask0, bias0, gate0);
    if (!wanted) p.flags |= EVO_FLAG_FORWARD_ONLY;
    Tensor q, k, v, g, o, aux;
    {
        at::AutoDispatchBelowADInplaceOrView guard;
        if (!operands(c, Q, mask, bias)) return std::nullopt;
        c10::DeviceGuard on(Q.device());
        q = Q.contiguous();
        k = K.contiguous();
        v = V.contiguous();
        o = at::empty_like(q);
        const Aux layout(p);
        aux = scratch(layout.lse_bytes + evoattn_prep_bytes(&p), q);
        layout.place(p, aux);
        p.q = q.data_ptr();
        p.k = k.data_ptr();
        p.v = v.data_ptr();
        if (gated) {   // only the gated output is written: the backward's gate pass forms delta from it
            g = gate0.contiguous();
            p.gate = g.data_ptr();
            p.o_gated = o.data_ptr();
        } else {
            p.o = o.data_ptr();
        }
        if (evoattn_fwd(&p, stream_of(q)) != EVO_OK) return std::nullopt;
    }
    if (wanted) {
        auto node = make_node<AttentionNode>(Q, K, V, mask0, bias0, gate0);
        node->c = c;
        node->c.p.gate = nullptr;
        torch::autograd::set_history(o, node);
        node->saved.reserve(gated ? 8 : 7);
        node->save(q);
        node->save(k);
        node->save(v);
        node->save(*mask);
        node->save(*bias);
        node->save(aux);
        node->save(o, true);
        if (gated) node->save(g);
    }
    return o;
}

// Q, K, V (and the gate) as slots of one [B,S,N,W,H,D] tensor (`_SlotAttention` in evoformer.py describes the buffers).
struct SlotAttention : torch::autograd::Function<SlotAttention> {
    static void strides(EvoAttnParams &p, const Tensor &P) {
        const int64_t W = P.size(3), tok = W * p.H * p.D;
        p.stride_b = (int64_t)p.S * p.N * tok;
        p.stride_h = p.D;
        p.stride_s = p.N * tok;
        p.stride_n = tok;
    }
    static char *slot(const Tensor &t, const EvoAttnParams &p, int i) {
        return (char *)t.data_ptr() + (size_t)i * p.H * p.D * t.element_size();
    }

    // What the forward leaves for the backward.  `ob` [B,S,N,W,H,D]: slot 1 (gated, else 0) the output, slot 2 room for its gradient.
    struct Run {
        Call c{};
        Tensor ob, aux;
        OptTensor mask, bias;
    };
    static Run enqueue(const Tensor &P, const OptTensor &mask, const OptTensor &bias, bool gated, int64_t flags) {
        Run r;
        Call &c = r.c;
        EvoAttnParams &p = c.p;
        p.B = (int32_t)P.size(0);
        p.S = (int32_t)P.size(1);
        p.N = (int32_t)P.size(2);
        p.H = (int32_t)P.size(4);
        p.D = (int32_t)P.size(5);
        p.dtype = evo_dtype(P.scalar_type());
        p.dbias_dtype = EVO_F32;
        p.flags = (int32_t)flags;
        p.scale = (float)(1.0 / std::sqrt((double)p.D));
        strides(p, P);
        c.gated = gated;
        r.mask = mask;
        r.bias = bias;
        TORCH_CHECK_VALUE(operands(c, P, r.mask, r.bias), "the mask must be [B,S,1,1,N] and the pair bias [B,1,H,N,N] (B and the mask's S may be 1), on P's device");
        c10::DeviceGuard on(P.device());
        r.ob = at::empty_like(P);
        const Aux layout(p);
        r.aux = scratch(layout.lse_bytes + evoattn_prep_bytes(&p), P);
        layout.place(p, r.aux);
        p.q = slot(P, p, 0);
        p.k = slot(P, p, 1);
        p.v = slot(P, p, 2);
        if (gated) {   // the gated output alone: slot 0 stays unwritten
            p.gate = slot(P, p, 3);
            p.o_gated = slot(r.ob, p, 1);
        } else {
            p.o = slot(r.ob, p, 0);
        }
        check(evoattn_fwd(&p, stream_of(P)), "evoattn_fwd");
        p.gate = nullptr;
        p.o_gated = nullptr;
        return r;
    }
    // the gradient of P; that of the output lies at `dout` (slot 2 of the forward's buffer)
    static Tensor enqueue_gradients(const Call &c, const Tensor &P, const Tensor &mask, const Tensor &bias, const Tensor &aux, void *out, void *dout,
                                    bool want_dbias, bool want_dmask, Tensor &dbias, Tensor &dmask) {
        c10::DeviceGuard on(P.device());
        Tensor DP = P.size(3) == (c.gated ? 4 : 3) ? at::empty_like(P) : at::zeros_like(P);
        EvoAttnParams p = c.p;
        Aux(p).place(p, aux);
        p.q = slot(P, p, 0);
        p.k = slot(P, p, 1);
        p.v = slot(P, p, 2);
        p.dout = dout;
        p.dq = slot(DP, p, 0);
        p.dk = slot(DP, p, 1);
        p.dv = slot(DP, p, 2);
        if (c.gated) {   // slot 2 is the node's own memory: the gradient of the ungated output takes its place
            p.o = nullptr;
            p.gate = slot(P, p, 3);
            p.dgate = slot(DP, p, 3);
            p.o_gated = out;
            p.flags |= EVO_FLAG_GATE_DOUT_INPLACE;
        } else {
            p.o = out;
        }
        enqueue_backward(p, P, mask, bias, want_dbias, want_dmask, dbias, dmask);
        return DP;
    }

    static variable_list forward(AutogradContext *ctx, const Tensor &P, OptTensor mask, OptTensor bias, bool gated, int64_t flags) {
        const Run r = enqueue(P, mask, bias, gated, flags);
        const Call &c = r.c;
        const Tensor &ob = r.ob, &aux = r.aux;
        Tensor out = ob.select(3, gated ? 1 : 0);
        // `out` is what the backward reads: saved like any output, so that a consumer who changes it in place is told so
        // by autograd's version check.  Slot 2 alone is kept under a version counter of its own: the consumer
        // writes the incoming gradient there in place, which must not look like a change of `out` (the same memory object).
        Tensor grad_slot = ob.variable_data().select(3, 2);
        ctx->save_for_backward({P, *r.mask, *r.bias, aux, out});
        ctx->saved_data["slot"] = grad_slot;
        ctx->saved_data["call"] = std::string((const char *)&c, sizeof c);
        ctx->mark_non_differentiable({grad_slot});
        ctx->set_materialize_grads(false);   // (no tensor of zeros for the second output's gradient, which nobody has)
        return {out, grad_slot};
    }

    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const bool rec = at::GradMode::is_enabled();
        variable_list res(5);
        {
            at::AutoDispatchBelowADInplaceOrView guard;
            const auto saved = ctx->get_saved_variables();
            const Tensor P = saved[0].contiguous(), &mask = saved[1], &bias = saved[2], &aux = saved[3];
            Call c;
            const std::string bytes = ctx->saved_data["call"].toStringRef();
            memcpy(&c, bytes.data(), sizeof c);
            const Tensor slot2 = ctx->saved_data["slot"].toTensor();
            if (!grads[0].defined()) {   // the output took no part in what is differentiated
                res[0] = at::zeros_like(P);
                return res;
            }
            // (a hook on saved tensors may hand back a copy whose rows do not lie as slots do)
            Tensor out = saved[4];
            if (!out.strides().equals(slot2.strides())) {
                const Tensor ob = at::empty_like(P);
                out = ob.select(3, 0).copy_(out);
            }
            const Tensor &dout = grads[0];
            bool in_place = dout.data_ptr() == slot2.data_ptr() && dout.scalar_type() == slot2.scalar_type() && dout.sizes().equals(slot2.sizes());
            for (int i = 0; in_place && i < 5; ++i) in_place = slot2.size(i) == 1 || dout.stride(i) == slot2.stride(i);
            c10::DeviceGuard on(P.device());
            if (!in_place) const_cast<Tensor &>(slot2).copy_(dout);
            // (edges are those of the tensors that were given)
            size_t edge = 1;
            const bool want_dmask = mask.defined() && ctx->needs_input_grad(edge) && mask.is_floating_point();
            if (mask.defined()) ++edge;
            const bool want_dbias = bias.defined() && ctx->needs_input_grad(edge);
            Tensor dbias, dmask;
            res[0] = enqueue_gradients(c, P, mask, bias, aux, out.data_ptr(), slot2.data_ptr(), want_dbias, want_dmask, dbias, dmask);
            if (want_dmask) res[1] = finish_dmask(dmask, c);
            if (want_dbias) res[2] = finish_dbias(dbias, c);
        }
        return once_differentiable(std::move(res), rec);
    }
};

variable_list slot_attention(const Tensor &P, const OptTensor &mask, const OptTensor &bias, bool gated, int64_t flags) {
    TORCH_CHECK_NOT_IMPLEMENTED(!dual(P) && !(mask && dual(*mask)) && !(bias && dual(*bias)),
                                "slot_attention has no formula for forward mode differentiation");
    TORCH_CHECK_VALUE(plain(P) && P.is_cuda() && P.dim() == 6 && P.numel() > 0 && P.is_contiguous() && P.size(3) >= (gated ? 4 : 3) &&
                          (P.scalar_type() == at::kBFloat16 || P.scalar_type() == at::kHalf) && head_dim_built(P.size(5)),
                      "P must be a contiguous 16-bit [B,S,N,W,H,D] tensor with W >= 3 (4 with a gate) and a head dim the library is built for");
    return SlotAttention::apply(P, mask, bias, gated, flags);
}

// ------------------------------------------------------------------ the layers of the block around the attention

// Slices of the rows that a weight gradient is summed over (`_row_slices` in block.py: the same rule, and why).
int64_t row_slices(int64_t rows, int64_t n_out, int64_t n_in) {
    const int64_t tiles = ((n_out + 127) / 128) * ((n_in + 127) / 128);
    int64_t g = 1;
    while (g * tiles < 512 && rows % (2 * g) == 0 && rows / (2 * g) >= 256) g *= 2;
    return g;
}

Tensor weight_grad(const Tensor &dy2, const Tensor &x2) {
    const int64_t rows = dy2.size(0), g = row_slices(rows, dy2.size(1), x2.size(1));
    if (g == 1) return dy2.t().mm(x2);
    return at::bmm(dy2.view({g, rows / g, -1}).transpose(1, 2), x2.view({g, rows / g, -1})).sum(0);
}

Tensor bias_grad(const Tensor &dy2) {
    const int64_t rows = dy2.size(0), cols = dy2.size(1);
    const int dt = evo_dtype(dy2.scalar_type());
    if (rows && dy2.is_cuda() && dt != EVO_NONE && cols <= INT32_MAX && dy2.stride(1) == 1 && dy2.stride(0) >= cols && dy2.stride(0) % 8 == 0 &&
        (uintptr_t)dy2.data_ptr() % 16 == 0) {
        if (const size_t bytes = evoattn_colsum_workspace_bytes(rows, (int32_t)cols, dt)) {
            c10::DeviceGuard on(dy2.device());
            Tensor out = at::empty({cols}, dy2.options()), ws = scratch(bytes, dy2);
            check(evoattn_colsum(dy2.data_ptr(), dy2.stride(0), out.data_ptr(), ws.data_ptr(), (size_t)ws.numel(), rows, (int32_t)cols, dt,
                                 stream_of(dy2)), "evoattn_colsum");
            return out;
        }
    }
    return dy2.sum(0);
}

Tensor as_rows(const Tensor &t) { return t.reshape({-1, t.size(-1)}); }

// The products of the Linear layers: through the library's kernels (csrc/linear.hip) where they take the operands, else torch's.
bool lin_rows_ok(const Tensor &t, at::ScalarType dt) {
    return plain(t) && t.is_cuda() && t.dim() == 2 && t.scalar_type() == dt && t.stride(1) == 1 && t.stride(0) % 8 == 0 && t.stride(0) >= t.size(1) &&
           (uintptr_t)t.data_ptr() % 16 == 0;
}
// `a`: rows of a matrix to be multiplied by the stacked weights [n, k]
bool lin_ok(const Tensor &a, const std::vector<Tensor> &w) {
    const auto dt = a.scalar_type();
    if ((dt != at::kBFloat16 && dt != at::kHalf) || w.empty() || w.size() > 4 || !plain_modes() || !lin_rows_ok(a, dt) || a.size(0) == 0) return false;
    for (const Tensor &t : w)
        if (!lin_rows_ok(t, dt) || t.device() != a.device() || !t.is_contiguous() || !t.sizes().equals(w[0].sizes())) return false;
    const int64_t rows = w[0].size(0), n = rows * (int64_t)w.size(), k = w[0].size(1);
    return n <= INT32_MAX && k <= INT32_MAX && rows % 64 == 0 && evoattn_linear_dw_workspace_bytes(a.size(0), (int32_t)n, (int32_t)k, evo_dtype(dt)) != 0;
}
// Where the library's kernels take over.  They run a large product in half to three quarters of the time of linear.hip's (which waits
// for memory once per 64 of the contraction), and cost 18 us of host time and, with several weights, 6 us for a copy of them
// (forward: 20 with the padded bias).  linear.hip takes 1.2 us for each stage of 64 of each round of 512 workgroups; up to 64 of these the
// two are level, or what the library saves is less than what it costs.  bf16, back to back, rows, n, k (stages in all rounds): own / library, us:
//   y    8192, 1024, 1024 (16) 22 / 22; 32 768, 1024, 256 (16) 30 / 30; 98 304, 1024, 256 (48) 84 / 77; 8192, 4096, 1024 (64) 83 / 56;
//        beyond: 16 384, 3072, 768 (72) 100 / 68; 32 768, 2048, 2048 300 / 191; 131 072, 4096, 4096 5044 / 2878
//   dx   32 768, 1024, 256 (16) 25 / 23; 98 304, 1024, 256 (48) 71 / 54; 2048, 4096, 1024 (64) 65 / 33; beyond: 16 384, 3072, 768 (96)
//        108 / 68; 32 768, 2048, 2048 342 / 216
// Whole block steps, linear.hip throughout / the library beyond, us: 131 072 rows of 256 (64 for y) 1102 / 1137; 32 768 of 512, n = 2048 (64)
// 793 / 808; 32 768 of 768, n = 1536 (72) 866 / 797; 65 536 of 512, n = 2048 (128) 1490 / 1430; 16 384 of 1024, n = 4096 (128) 1115 / 1014.
bool lin_rows_pay(int64_t rows, int64_t outs, int64_t depth) {
    const int64_t tiles = ((rows + 127) / 128) * ((outs + 127) / 128);
    return (tiles + 511) / 512 * ((depth + 63) / 64) <= 64;
}
// dW and the column sums, of which the library's way takes 42 us of host time: level at 64 of its stages.  32 768,
// 1024, 256 38 / 51; 131 072, 1024, 256 124 / 131; 32 768, 1024, 1024 99 / 94; beyond: 32 768, 768, 768 99 / 70; 65 536, 1024, 1024 213 / 171;
// 8192, 4096, 4096 367 / 245; and where a slice's gradient in fp32 is itself large: 1024, 4096, 1024 29 / 44, but 1024, 4096, 4096 72 / 53.
bool lin_weight_pays(int64_t rows, int64_t n, int64_t k, size_t workspace) {
    const int64_t slices = (int64_t)(workspace / ((size_t)(n * k + n) * sizeof(float))), wgs = ((n + 127) / 128) * ((k + 127) / 128) * slices;
    return n * k <= (int64_t)1 << 22 && (wgs + 511) / 512 * ((rows + slices * 64 - 1) / (slices * 64)) <= 64;
}

struct WeightPtrs {
    const void *p[4] = {};
    explicit WeightPtrs(const std::vector<Tensor> &w) {
        for (size_t i = 0; i < w.size(); ++i) p[i] = w[i].data_ptr();
    }
};

// a w^T (+ bias on the last columns) as [rows, n]; not defined where the kernels do not take it
Tensor lin_forward(const Tensor &a, const std::vector<Tensor> &w, const Tensor &bias) {
    if (at::autocast::is_autocast_enabled(at::kCUDA) || !lin_ok(a, w) || a.size(1) != w[0].size(1)) return Tensor();
    const int64_t n = w[0].size(0) * (int64_t)w.size();
    if (!lin_rows_pay(a.size(0), n, a.size(1))) return Tensor();
    const int64_t from = bias.defined() ? n - bias.numel() : 0;
    if (bias.defined() && (!plain(bias) || bias.dim() != 1 || bias.scalar_type() != a.scalar_type() || bias.device() != a.device() || !bias.is_contiguous() ||
                           from < 0 || from % 16 || (uintptr_t)bias.data_ptr() % 16))
        return Tensor();
    c10::DeviceGuard on(a.device());
    Tensor y = at::empty({a.size(0), n}, a.options());
    check(evoattn_linear_fwd(a.data_ptr(), a.stride(0), WeightPtrs(w).p, (int32_t)w.size(), (int32_t)w[0].size(0), bias.defined() ? bias.data_ptr() : nullptr,
                             (int32_t)from, y.data_ptr(), n, a.size(0), (int32_t)n, (int32_t)a.size(1), evo_dtype(a.scalar_type()), stream_of(a)),
          "evoattn_linear_fwd");
    return y;
}

// dy w into `dx`, whose rows may lie apart; false where the kernels do not take it
bool lin_input_grad(const Tensor &dy, const std::vector<Tensor> &w, const Tensor &dx) {
    if (!lin_ok(dy, w) || !lin_rows_ok(dx, dy.scalar_type()) || dy.size(1) != w[0].size(0) * (int64_t)w.size() || dx.size(0) != dy.size(0) ||
        dx.size(1) != w[0].size(1) || dx.device() != dy.device() || !lin_rows_pay(dy.size(0), dx.size(1), dy.size(1)))
        return false;
    c10::DeviceGuard on(dy.device());
    check(evoattn_linear_dx(dy.data_ptr(), dy.stride(0), WeightPtrs(w).p, (int32_t)w.size(), (int32_t)w[0].size(0), dx.data_ptr(), dx.stride(0), dy.size(0),
                            (int32_t)dy.size(1), (int32_t)dx.size(1), evo_dtype(dy.scalar_type()), stream_of(dy)), "evoattn_linear_dx");
    return true;
}

// dy^T x and, if asked for, the column sums of dy
std::pair<Tensor, Tensor> lin_weight_grad(const Tensor &dy, const Tensor &x, bool sums) {
    const auto dt = dy.scalar_type();
    const int64_t rows = dy.size(0), n = dy.size(1), k = x.size(1);
    size_t bytes = 0;
    if ((dt == at::kBFloat16 || dt == at::kHalf) && plain_modes() && lin_rows_ok(dy, dt) && lin_rows_ok(x, dt) && x.device() == dy.device() &&
        n <= INT32_MAX && k <= INT32_MAX)
        bytes = evoattn_linear_dw_workspace_bytes(rows, (int32_t)n, (int32_t)k, evo_dtype(dt));
    if (!bytes || !lin_weight_pays(rows, n, k, bytes)) return {weight_grad(dy, x), sums ? bias_grad(dy) : Tensor()};
    c10::DeviceGuard on(dy.device());
    Tensor out = at::empty({n * k + (sums ? n : 0)}, dy.options()), ws = scratch(bytes, dy);
    check(evoattn_linear_dw(dy.data_ptr(), dy.stride(0), x.data_ptr(), x.stride(0), out.data_ptr(), sums, ws.data_ptr(), (size_t)ws.numel(), rows, (int32_t)n,
                            (int32_t)k, evo_dtype(dt), stream_of(dy)), "evoattn_linear_dw");
    return {out.narrow(0, 0, n * k).view({n, k}), sums ? out.narrow(0, n * k, n) : Tensor()};
}

struct LinearNode : SavingNode {
    bool has_bias = false;
    Tensor dx_place;
    std::string name() const override { return "LinearBackward"; }
    variable_list apply(variable_list &&grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        const bool rec = at::GradMode::is_enabled();
        variable_list out(3);
        if (!grads[0].defined()) return out;
        {
            at::AutoDispatchBelowADInplaceOrView guard;
            const Tensor x = saved[0].unpack(), w = saved[1].unpack(), dy2 = as_rows(grads[0]);
            if (task_should_compute_output(0)) {
                out[0] = dx_place.defined() ? dx_place : at::empty_like(x, at::MemoryFormat::Contiguous);
                Tensor rows = out[0].view({-1, x.size(-1)});
                if (!lin_input_grad(dy2, {w}, rows)) at::mm_out(rows, dy2, w);
            }
            const bool sums = has_bias && task_should_compute_output(2);
            if (task_should_compute_output(1)) std::tie(out[1], out[2]) = lin_weight_grad(dy2, as_rows(x), sums);
            else if (sums) out[2] = bias_grad(dy2);
        }
        return once_differentiable(std::move(out), rec);
    }
};

// x W^T + b with the weight gradient summed over slices of the rows; `dx_place` (shaped like x, rows may lie apart): where
// the input gradient is to be written.  None under a mode or for tensors that a hand-made node does not stand for.
OptTensor linear(const Tensor &x, const Tensor &weight, const OptTensor &bias, const OptTensor &dx_place) {
    if (!plain_modes() || !plain(x) || !plain(weight) || (bias && bias->defined() && !plain(*bias))) return std::nullopt;
    Tensor y;
    {
        at::AutoDispatchBelowADInplaceOrView guard;
        // (as a matrix: for an input of more dimensions whose rows lie apart torch multiplies and then adds the
        // bias in a pass of its own)
        const Tensor rows = as_rows(x);
        y = lin_forward(rows, {weight}, bias ? *bias : Tensor());
        if (!y.defined()) y = at::linear(rows, weight, bias);
        auto shape = x.sizes().vec();
        shape.back() = weight.size(0);
        y = y.view(shape);
    }
    const Tensor b = bias ? *bias : Tensor();
    if (SavingNode::wanted(x, weight, b)) {
        auto node = make_node<LinearNode>(x, weight, b);
        node->has_bias = b.defined();
        if (dx_place) node->dx_place = *dx_place;
        torch::autograd::set_history(y, node);
        node->save(x);
        node->save(weight);
    }
    return y;
}

struct StackedNode : SavingNode {
    std::vector<int64_t> sizes;
    bool has_bias = false;
    std::string name() const override { return "StackedProjectionBackward"; }
    // results: x, gate_bias, the weights
    variable_list apply(variable_list &&grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        const bool rec = at::GradMode::is_enabled();
        variable_list out(2 + sizes.size());
        if (!grads[0].defined()) return out;
        {
            at::AutoDispatchBelowADInplaceOrView guard;
            const Tensor x = saved[0].unpack(), dp2 = as_rows(grads[0]);
            std::vector<Tensor> w;
            for (size_t i = 0; i < sizes.size(); ++i) w.push_back(saved[1 + i].unpack());
            if (task_should_compute_output(0)) {
                out[0] = at::empty_like(x, at::MemoryFormat::Contiguous);
                Tensor rows = as_rows(out[0]);
                if (!lin_input_grad(dp2, w, rows)) at::mm_out(rows, dp2, at::cat(w, 0));
            }
            const bool sums = has_bias && task_should_compute_output(1);
            bool any = false;
            for (size_t i = 0; i < sizes.size(); ++i) any |= task_should_compute_output(2 + i);
            if (any) {
                auto [dw, db] = lin_weight_grad(dp2, as_rows(x), sums);
                auto parts = dw.split_with_sizes(sizes, 0);
                for (size_t i = 0; i < sizes.size(); ++i) out[2 + i] = parts[i];
                if (sums) out[1] = db.narrow(0, db.size(0) - sizes.back(), sizes.back());
            } else if (sums) {
                out[1] = bias_grad(dp2.narrow(1, dp2.size(1) - sizes.back(), sizes.back()));
            }
        }
        return once_differentiable(std::move(out), rec);
    }
};

// x [rows, k] times the stacked weights, `gb` on the last columns
Tensor stacked_forward(const Tensor &x, const std::vector<Tensor> &weights, const Tensor &gb) {
    const Tensor y = lin_forward(x, weights, gb);
    if (y.defined()) return y;
    const Tensor w = at::cat(weights, 0);
    OptTensor bias;
    if (gb.defined()) bias = at::constant_pad_nd(gb, {w.size(0) - gb.size(0), 0});
    return at::linear(x, w, bias);
}

// Several projections of one input as one GEMM with their weights stacked; `gate_bias` is added on the last layer's columns.
// None as above.
OptTensor stacked_projection(const Tensor &x, const OptTensor &gate_bias, const std::vector<Tensor> &weights) {
    Tensor y;
    const Tensor gb = gate_bias ? *gate_bias : Tensor();
    bool taken = plain_modes() && plain(x) && (!gb.defined() || plain(gb));
    for (const Tensor &t : weights) taken = taken && plain(t);
    if (!taken) return std::nullopt;
    {
        at::AutoDispatchBelowADInplaceOrView guard;
        y = stacked_forward(as_rows(x), weights, gb);
        auto shape = x.sizes().vec();
        shape.back() = y.size(1);
        y = y.view(shape);
    }
    bool needed = SavingNode::wanted(x, gb);
    for (const auto &t : weights) needed |= SavingNode::wanted(t);
    if (needed) {
        std::shared_ptr<StackedNode> node(new StackedNode(), torch::autograd::deleteNode);
        variable_list inputs{x, gb};
        inputs.insert(inputs.end(), weights.begin(), weights.end());
        node->set_next_edges(torch::autograd::collect_next_edges(inputs));
        for (const auto &t : weights) node->sizes.push_back(t.size(0));
        node->has_bias = gb.defined();
        torch::autograd::set_history(y, node);
        node->save(x);
        for (const auto &t : weights) node->save(t);
    }
    return y;
}

// mean, then 1 / deviation of every row, each on a 16-byte boundary
Tensor ln_stats(const Tensor &x, int64_t rows) { return at::empty({2 * ((rows + 3) / 4 * 4)}, x.options().dtype(at::kFloat)); }
const void *ptr_or_null(const Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }

bool ln_ok(const Tensor &x, const Tensor &w, const Tensor &b) {
    const int dt = evo_dtype(x.scalar_type());
    if (!plain(x) || !plain_modes() || !x.is_cuda() || x.dim() < 1 || x.numel() == 0 || dt == EVO_NONE || x.size(-1) > INT32_MAX) return false;
    for (const Tensor *t : {&w, &b})
        if (t->defined() && (!plain(*t) || t->scalar_type() != x.scalar_type() || t->device() != x.device() || t->dim() != 1 || t->size(0) != x.size(-1)))
            return false;
    return evoattn_layernorm_bwd_workspace_bytes(1, (int32_t)x.size(-1), dt) != 0;
}
// (x, w, b contiguous)
Tensor ln_forward(const Tensor &x, const Tensor &w, const Tensor &b, double eps, const Tensor &stats) {
    c10::DeviceGuard on(x.device());
    const int64_t cols = x.size(-1), rows = x.numel() / cols;
    Tensor y = at::empty_like(x);
    float *mean = (float *)stats.data_ptr();
    check(evoattn_layernorm_fwd(x.data_ptr(), ptr_or_null(w), ptr_or_null(b), y.data_ptr(), mean, mean + stats.numel() / 2, rows, (int32_t)cols,
                                evo_dtype(x.scalar_type()), (float)eps, stream_of(x)), "evoattn_layernorm_fwd");
    return y;
}
void ln_backward(const Tensor &dy, const Tensor &x, const Tensor &w, const Tensor &stats, bool need_x, bool need_w, bool need_b, Tensor &dx, Tensor &dw,
                 Tensor &db) {
    if (!need_x && !need_w && !need_b) return;
    c10::DeviceGuard on(x.device());
    const int64_t cols = x.size(-1), rows = x.numel() / cols;
    const int dt = evo_dtype(x.scalar_type());
    Tensor ws;
    if (need_x) dx = at::empty_like(x);
    if (need_w) dw = at::empty({cols}, x.options());
    if (need_b) db = at::empty({cols}, x.options());
    if (need_w || need_b) ws = scratch(evoattn_layernorm_bwd_workspace_bytes(rows, (int32_t)cols, dt), x);
    const float *mean = (const float *)stats.data_ptr();
    check(evoattn_layernorm_bwd(dy.data_ptr(), x.data_ptr(), ptr_or_null(w), mean, mean + stats.numel() / 2, const_cast<void *>(ptr_or_null(dx)),
                                const_cast<void *>(ptr_or_null(dw)), const_cast<void *>(ptr_or_null(db)), const_cast<void *>(ptr_or_null(ws)),
                                ws.defined() ? (size_t)ws.numel() : 0, rows, (int32_t)cols, dt, stream_of(x)), "evoattn_layernorm_bwd");
}

struct LayerNormNode : SavingNode {
    bool has_bias = false;
    std::string name() const override { return "LayerNormBackward"; }
    variable_list apply(variable_list &&grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        const bool rec = at::GradMode::is_enabled();
        variable_list out(3);
        if (!grads[0].defined()) return out;
        {
            at::AutoDispatchBelowADInplaceOrView guard;
            const Tensor x = saved[0].unpack().contiguous(), w = saved[1].unpack(), stats = saved[2].unpack();
            ln_backward(grads[0].contiguous(), x, w, stats, task_should_compute_output(0), w.defined() && task_should_compute_output(1),
                        has_bias && task_should_compute_output(2), out[0], out[1], out[2]);
        }
        return once_differentiable(std::move(out), rec);
    }
};

// LayerNorm over the last dimension through the library's kernels: x and y cross HBM once in the forward, x, dy and dx once in
// the backward.  None for rows, dtypes or devices that those kernels do not take.
OptTensor layer_norm(const Tensor &x, const OptTensor &weight, const OptTensor &bias, double eps) {
    const Tensor w0 = weight ? *weight : Tensor(), b0 = bias ? *bias : Tensor();
    if (!ln_ok(x, w0, b0)) return std::nullopt;
    Tensor y, xc, w, stats;
    {
        at::AutoDispatchBelowADInplaceOrView guard;
        xc = x.contiguous();
        w = w0.defined() ? w0.contiguous() : Tensor();
        stats = ln_stats(xc, xc.numel() / xc.size(-1));
        y = ln_forward(xc, w, b0.defined() ? b0.contiguous() : Tensor(), eps, stats);
    }
    if (SavingNode::wanted(x, w0, b0)) {
        auto node = make_node<LayerNormNode>(x, w0, b0);
        node->has_bias = b0.defined();
        torch::autograd::set_history(y, node);
        node->save(xc);
        node->save(w);
        node->save(stats);
    }
    return y;
}

// The pair bias (csrc/pair_bias.hip): contiguous 16-byte aligned operands, and whether the kernels take them.
struct PairOperands {
    Tensor z, lw, lb, w;
    int64_t B, pairs;
    int32_t C, H;
    int dt;
    size_t workspace;
    PairOperands(const Tensor &z_, const Tensor &lw_, const Tensor &lb_, const Tensor &w_) : z(z_), lw(lw_), lb(lb_), w(w_) {
        B = z.size(0);
        pairs = z.size(1) * z.size(2);
        C = (int32_t)z.size(3);
        H = (int32_t)w.size(0);
        dt = evo_dtype(z.scalar_type());
        workspace = evoattn_pair_bias_workspace_bytes(B, pairs, C, H, dt);
    }
    static bool ok(const Tensor &z, const Tensor &lw, const Tensor &lb, const Tensor &w) {
        if (!plain(z) || !plain_modes() || at::autocast::is_autocast_enabled(at::kCUDA) || !z.is_cuda() || z.dim() != 4 || z.numel() == 0 || !plain(w) ||
            w.dim() != 2 || w.size(1) != z.size(3) || w.size(1) > 4096 || w.size(0) > 4096)
            return false;
        for (const Tensor *t : {&lw, &lb, &w})
            if (t->defined() && (!plain(*t) || t->scalar_type() != z.scalar_type() || t->device() != z.device())) return false;
        for (const Tensor *t : {&lw, &lb})
            if (t->defined() && (t->dim() != 1 || t->size(0) != z.size(3))) return false;
        return evoattn_pair_bias_workspace_bytes(z.size(0), z.size(1) * z.size(2), (int32_t)z.size(3), (int32_t)w.size(0), evo_dtype(z.scalar_type())) != 0;
    }
    static Tensor ready(const Tensor &t) {
        Tensor c = t.defined() ? t.contiguous() : t;
        return c.defined() && (uintptr_t)c.data_ptr() % 16 ? c.clone() : c;
    }
    Tensor forward(double eps, Tensor &stats) const {
        c10::DeviceGuard on(z.device());
        Tensor out = at::empty({B, 1, H, z.size(1), z.size(2)}, z.options());
        stats = at::empty({2 * B * pairs}, z.options().dtype(at::kFloat));   // mean, then 1 / deviation
        float *mean = (float *)stats.data_ptr();
        check(evoattn_pair_bias_fwd(z.data_ptr(), ptr_or_null(lw), ptr_or_null(lb), w.data_ptr(), out.data_ptr(), mean, mean + B * pairs, B, pairs, C, H, dt,
                                    (float)eps, stream_of(z)), "evoattn_pair_bias_fwd");
        return out;
    }
    // dparams [2 + H, C]: LayerNorm weight, LayerNorm bias, projection
    void backward(const Tensor &dbias, const Tensor &stats, bool need_z, bool need_params, Tensor &dz, Tensor &dparams) const {
        if (!need_z && !need_params) return;
        c10::DeviceGuard on(z.device());
        Tensor ws;
        if (need_z) dz = at::empty_like(z);
        if (need_params) {
            dparams = at::empty({2 + H, C}, z.options());
            ws = scratch(workspace, z);
        }
        const float *mean = (const float *)stats.data_ptr();
        check(evoattn_pair_bias_bwd(dbias.data_ptr(), z.data_ptr(), ptr_or_null(lw), ptr_or_null(lb), w.data_ptr(), mean, mean + B * pairs,
                                    const_cast<void *>(ptr_or_null(dz)), const_cast<void *>(ptr_or_null(dparams)), const_cast<void *>(ptr_or_null(ws)),
                                    ws.defined() ? (size_t)ws.numel() : 0, B, pairs, C, H, dt, stream_of(z)), "evoattn_pair_bias_bwd");
    }
};

struct PairBiasNode : SavingNode {
    std::string name() const override { return "PairBiasBackward"; }
    // results: z, the LayerNorm's weight and bias, the projection's weight
    variable_list apply(variable_list &&grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        const bool rec = at::GradMode::is_enabled();
        variable_list out(4);
        if (!grads[0].defined()) return out;
        {
            at::AutoDispatchBelowADInplaceOrView guard;
            const PairOperands o(PairOperands::ready(saved[0].unpack()), saved[1].unpack(), saved[2].unpack(), PairOperands::ready(saved[3].unpack()));
            const bool lw = task_should_compute_output(1), lb = task_should_compute_output(2), w = task_should_compute_output(3);
            Tensor dparams;
            o.backward(grads[0].contiguous(), saved[4].unpack(), task_should_compute_output(0), lw || lb || w, out[0], dparams);
            if (lw) out[1] = dparams.select(0, 0);
            if (lb) out[2] = dparams.select(0, 1);
            if (w) out[3] = dparams.narrow(0, 2, o.H);
        }
        return once_differentiable(std::move(out), rec);
    }
};

// LayerNorm of the pair representation, its projection to heads and the permute to [B,1,H,N,N] in one pass.  None for what
// the kernels do not take.
OptTensor pair_bias(const Tensor &z, const OptTensor &ln_weight, const OptTensor &ln_bias, double eps, const Tensor &weight) {
    const Tensor lw = ln_weight ? *ln_weight : Tensor(), lb = ln_bias ? *ln_bias : Tensor();
    if (!PairOperands::ok(z, lw, lb, weight)) return std::nullopt;
    std::optional<PairOperands> o;
    Tensor out, stats;
    {
        at::AutoDispatchBelowADInplaceOrView guard;
        o.emplace(PairOperands::ready(z), PairOperands::ready(lw), PairOperands::ready(lb), PairOperands::ready(weight));
        out = o->forward(eps, stats);
    }
    if (SavingNode::wanted(z, lw, lb, weight)) {
        auto node = make_node<PairBiasNode>(z, lw, lb, weight);
        torch::autograd::set_history(out, node);
        for (const Tensor *t : {&o->z, &o->lw, &o->lb, &o->w, &stats}) node->save(*t);
    }
    return out;
}

// ------------------------------------------------------------------ the whole block

// Inputs of the block in the order of its node's results.
enum BlockInput { kM, kZ, kNormMW, kNormMB, kQ, kK, kV, kG, kGBias, kO, kOBias, kNormZW, kNormZB, kZW, kBlockInputs };

// One node for what the layers above do in five, with the tensors between them its own: a training step of a small block
// spent a third of its host time between those nodes (the engine's bookkeeping, views, the interpreter).
struct BlockNode : SavingNode {
    Call c{};
    // saved: the inputs, then
    enum { kX = kBlockInputs, kStatsM, kP, kMask, kBias, kAux, kOut, kStatsZ, kSaved };
    std::string name() const override { return "GatedAttentionBlockBackward"; }
    variable_list apply(variable_list &&grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        const bool rec = at::GradMode::is_enabled();
        variable_list out(kBlockInputs);
        if (!grads[0].defined()) return out;
        {
            at::AutoDispatchBelowADInplaceOrView guard;
            Tensor t[kSaved];
            for (int i = 0; i < kSaved; ++i) t[i] = saved[i].unpack();
            for (int i : {(int)kM, (int)kX, (int)kP, (int)kOut}) t[i] = t[i].contiguous();   // (after a hook on saved tensors)
            bool want[kBlockInputs], inner = false;
            for (int i = 0; i < kBlockInputs; ++i) {
                want[i] = t[i].defined() && task_should_compute_output(i);
                inner |= want[i] && i != kO && i != kOBias;
            }
            Tensor dy = grads[0].scalar_type() == t[kM].scalar_type() ? as_rows(grads[0]) : as_rows(grads[0].to(t[kM].scalar_type()));
            const int64_t rows = dy.size(0), W = t[kP].size(3), hd = t[kP].size(4) * t[kP].size(5);
            const Tensor slots = t[kOut].view({rows, W * hd}), o = slots.narrow(1, (c.gated ? 1 : 0) * hd, hd);
            if (want[kO] || want[kOBias]) {
                std::tie(out[kO], out[kOBias]) = lin_weight_grad(dy, o, want[kOBias]);
                if (!want[kO]) out[kO] = Tensor();
            }
            if (inner) {
                Tensor dout = slots.narrow(1, 2 * hd, hd), dbias, dmask;
                if (!lin_input_grad(dy, {t[kO]}, dout)) at::mm_out(dout, dy, t[kO]);
                const bool z_side = want[kZ] || want[kNormZW] || want[kNormZB] || want[kZW];
                const Tensor DP = SlotAttention::enqueue_gradients(c, t[kP], t[kMask], t[kBias], t[kAux], o.data_ptr(), dout.data_ptr(), z_side, false, dbias,
                                                                   dmask);
                if (z_side) {
                    Tensor dparams;
                    PairOperands(t[kZ], t[kNormZW], t[kNormZB], t[kZW])
                        .backward(dbias, t[kStatsZ], want[kZ], want[kNormZW] || want[kNormZB] || want[kZW], out[kZ], dparams);
                    if (want[kNormZW]) out[kNormZW] = dparams.select(0, 0);
                    if (want[kNormZB]) out[kNormZB] = dparams.select(0, 1);
                    if (want[kZW]) out[kZW] = dparams.narrow(0, 2, dparams.size(0) - 2);
                }
                const Tensor dp2 = DP.view({rows, W * hd}), x2 = as_rows(t[kX]);
                bool weights = want[kGBias];
                for (int i = 0; i < W; ++i) weights |= want[kQ + i];
                if (weights) {
                    auto [dw, db] = lin_weight_grad(dp2, x2, want[kGBias]);
                    for (int i = 0; i < W; ++i)
                        if (want[kQ + i]) out[kQ + i] = dw.narrow(0, i * hd, hd);
                    if (want[kGBias]) out[kGBias] = db.narrow(0, (W - 1) * hd, hd);
                }
                if (want[kM] || want[kNormMW] || want[kNormMB]) {
                    Tensor dx = at::empty_like(x2);
                    std::vector<Tensor> w(t + kQ, t + kQ + W);
                    if (!lin_input_grad(dp2, w, dx)) at::mm_out(dx, dp2, at::cat(w, 0));
                    ln_backward(dx, t[kM], t[kNormMW], t[kStatsM], want[kM], want[kNormMW], want[kNormMB], out[kM], out[kNormMW], out[kNormMB]);
                }
            }
        }
        return once_differentiable(std::move(out), rec);
    }
};

// The block around the attention, in.size() == kBlockInputs (those that a block does not have undefined); `keep` [B,S,N], 1 where a
// key counts.  None where some part of it does not take the call.
OptTensor block(const std::vector<OptTensor> &in, const OptTensor &keep, int64_t heads, double eps_m, double eps_z, double inf, int64_t flags) {
    Tensor t[kBlockInputs];
    TORCH_CHECK(in.size() == kBlockInputs, "block: wrong number of inputs");
    for (int i = 0; i < kBlockInputs; ++i)
        if (in[i]) t[i] = *in[i];
    const Tensor &m = t[kM];
    for (const Tensor &i : t)
        if (i.defined() && !plain(i)) return std::nullopt;
    if (m.dim() != 4 || !m.is_cuda() || m.numel() == 0 || at::autocast::is_autocast_enabled(at::kCUDA)) return std::nullopt;
    const bool gated = t[kG].defined();
    const int W = gated ? 4 : 3;
    if (!t[kQ].defined() || t[kQ].dim() != 2 || !t[kK].defined() || !t[kV].defined() || !t[kO].defined()) return std::nullopt;
    const int64_t B = m.size(0), S = m.size(1), N = m.size(2), hd = t[kQ].size(0), D = hd / heads, rows = B * S * N;
    if (hd != heads * D || !head_dim_built(D) || B > INT32_MAX || S > INT32_MAX || N > INT32_MAX || heads > INT32_MAX) return std::nullopt;
    if (!ln_ok(m, t[kNormMW], t[kNormMB])) return std::nullopt;
    const std::vector<Tensor> w(t + kQ, t + kQ + W);
    if (m.size(3) != t[kQ].size(1) || !m.is_contiguous() || !lin_ok(m.view({rows, m.size(3)}), w) || !plain(t[kO]) || t[kO].dim() != 2 ||
        t[kO].size(1) != hd || t[kO].scalar_type() != m.scalar_type() || t[kO].device() != m.device())
        return std::nullopt;
    if (keep && (!plain(*keep) || keep->requires_grad() || keep->dim() != 3 || keep->size(0) != B || keep->size(1) != S || keep->size(2) != N ||
                 keep->device() != m.device()))
        return std::nullopt;
    if (t[kZ].defined() && (t[kZ].scalar_type() != m.scalar_type() || t[kZ].device() != m.device() || t[kZW].size(0) != heads ||
                            !PairOperands::ok(t[kZ], t[kNormZW], t[kNormZB], t[kZW]) || t[kZ].size(0) != B || t[kZ].size(1) != N || t[kZ].size(2) != N))
        return std::nullopt;
    Tensor y, x, stats_m, stats_z, P;
    SlotAttention::Run r;
    {
        at::AutoDispatchBelowADInplaceOrView guard;
        c10::DeviceGuard on(m.device());
        for (int i : {kNormMW, kNormMB}) t[i] = t[i].defined() ? t[i].contiguous() : t[i];
        stats_m = ln_stats(m, rows);
        x = ln_forward(m, t[kNormMW], t[kNormMB], eps_m, stats_m);
        P = stacked_forward(as_rows(x), w, t[kGBias]).view({B, S, N, W, heads, D});
        OptTensor mask, bias;
        if (keep) {
            const Tensor k = keep->to(at::kFloat).contiguous();
            mask = at::empty({B, S, 1, 1, N}, k.options());
            check(evoattn_keep_mask((const float *)k.data_ptr(), (float *)mask->data_ptr(), rows, (float)inf, stream_of(k)), "evoattn_keep_mask");
        }
        if (t[kZ].defined()) {
            for (int i : {kZ, kNormZW, kNormZB, kZW}) t[i] = PairOperands::ready(t[i]);
            bias = PairOperands(t[kZ], t[kNormZW], t[kNormZB], t[kZW]).forward(eps_z, stats_z);
        }
        r = SlotAttention::enqueue(P, mask, bias, gated, flags);
        const Tensor o = r.ob.view({rows, W * hd}).narrow(1, (gated ? 1 : 0) * hd, hd);
        y = lin_forward(o, {t[kO]}, t[kOBias]);
        if (!y.defined()) y = at::linear(o, t[kO], t[kOBias].defined() ? OptTensor(t[kOBias]) : OptTensor());
        y = y.view({B, S, N, t[kO].size(0)});
    }
    bool wanted = false;
    variable_list inputs;
    for (int i = 0; i < kBlockInputs; ++i) {
        inputs.push_back(in[i] ? *in[i] : Tensor());
        wanted |= SavingNode::wanted(inputs.back());
    }
    if (wanted) {
        std::shared_ptr<BlockNode> node(new BlockNode(), torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(inputs));
        node->c = r.c;
        torch::autograd::set_history(y, node);
        node->saved.reserve(BlockNode::kSaved);
        for (const Tensor &i : t) node->save(i);
        for (const Tensor &i : {x, stats_m, P, *r.mask, *r.bias, r.aux, r.ob, stats_z}) node->save(i);
    }
    return y;
}

}  // namespace

PYBIND11_MODULE(_host, m) {
    namespace py = pybind11;
    const py::call_guard<py::gil_scoped_release> no_gil;
    m.def("attention", &attention, no_gil, py::arg("Q"), py::arg("K"), py::arg("V"), py::arg("res_mask"), py::arg("pair_bias"), py::arg("gate"),
          py::arg("per_head"), py::arg("flags"));
    m.def("slot_attention", &slot_attention, no_gil, py::arg("P"), py::arg("res_mask"), py::arg("pair_bias"), py::arg("gated"), py::arg("flags"));
    m.def("linear", &linear, no_gil, py::arg("x"), py::arg("weight"), py::arg("bias"), py::arg("dx_place"));
    m.def("stacked_projection", &stacked_projection, no_gil, py::arg("x"), py::arg("gate_bias"), py::arg("weights"));
    m.def("layer_norm", &layer_norm, no_gil, py::arg("x"), py::arg("weight"), py::arg("bias"), py::arg("eps"));
    m.def("pair_bias", &pair_bias, no_gil, py::arg("z"), py::arg("ln_weight"), py::arg("ln_bias"), py::arg("eps"), py::arg("weight"));
    m.def("block", &block, no_gil, py::arg("inputs"), py::arg("keep"), py::arg("heads"), py::arg("eps_m"), py::arg("eps_z"), py::arg("inf"),
          py::arg("flags"));
}
