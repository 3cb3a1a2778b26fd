// The differentiable operators of a rank that has no peers as native autograd nodes. A small training step is host work: a node
// of Python's (its context, the casting decorators, the interpreter lock that the backward thread takes) costs 20 to 30 us forward and
// backward beside its launches, a native one 3 to 5.
//
// A call that is not the ordinary one returns None, and the caller takes its Python node, which behaves as it always did: tensors that
// are no plain tensors, tracing, functional transforms, forward-mode levels, dispatch modes, operands on other devices or of other shapes than the
// operator's own (the Python node raises for those).
#include "host_ops.h"

#include <ATen/autocast_mode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

namespace cw_host {
namespace {

using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

bool ordinary() {
    return !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
           !c10::impl::TorchDispatchModeTLS::any_modes_set() && !torch::jit::tracer::isTracing() &&
           torch::autograd::ForwardADLevel::try_get_by_idx(0) == nullptr;
}
// A plain CUDA tensor (or parameter), or None where that is allowed (an undefined tensor).
bool take(py::handle h, Tensor& t, bool optional = false) {
    if (h.is_none()) return optional;
    if (!THPVariable_CheckTypeExact(Py_TYPE(h.ptr()))) return false;
    t = THPVariable_Unpack(h.ptr());
    return t.is_cuda() && t.layout() == at::kStrided && !t.is_neg() && !t.is_conj();
}
bool together(std::initializer_list<Tensor> ts) {
    const Tensor& first = *ts.begin();
    for (const auto& t : ts)
        if (t.defined() && t.device() != first.device()) return false;
    return true;
}
bool half_type(at::ScalarType t) { return t == at::kBFloat16 || t == at::kHalf; }
OptTensor opt(const Tensor& t) { return t.defined() ? OptTensor(t) : OptTensor(); }
Tensor def(const OptTensor& t) { return t ? *t : Tensor(); }

// What custom_fwd does to inputs in an autocast region (nothing outside one), and the state in which the bodies run.
void cast_inputs(std::initializer_list<Tensor*> ts, at::ScalarType type) {
    Tensor none, *cast[CW_MAX_CASTS] = {&none, &none, &none, &none};
    int n = 0;
    for (Tensor* t : ts)
        if (t->defined() && t->is_floating_point() && t->scalar_type() != at::kDouble) cast[n++] = t;
    cast_together({cast[0], cast[1], cast[2], cast[3]}, type);
}
bool autocast() { return at::autocast::is_autocast_enabled(at::kCUDA); }
struct Body {
    at::AutoGradMode no_grad{false};
    c10::impl::ExcludeDispatchKeyGuard no_autocast{c10::DispatchKey::AutocastCUDA};
};

void keep(AutogradContext* ctx, std::vector<int64_t> meta) { ctx->saved_data["meta"] = std::move(meta); }
std::vector<int64_t> kept(const AutogradContext* ctx) { return ctx->saved_data.at("meta").toIntVector(); }

// A 16-bit operand of two products with rows that begin at multiples of 16 bytes (ops.aligned_rows).
Tensor aligned_rows(const Tensor& t_in) {
    const Tensor t = rows(t_in);
    if (t.element_size() != 2 || t.size(0) < 2 || (aligned16(t) && ld(t) % 8 == 0)) return t;
    Tensor out = empty({t.size(0), (t.size(1) + 7) / 8 * 8}, t).narrow(1, 0, t.size(1));
    return out.copy_(t);
}

// Which of the tensors are fp32, as bits.
int64_t fp32_inputs(std::initializer_list<const Tensor*> ts) {
    int64_t bits = 0, bit = 1;
    for (const Tensor* t : ts) {
        if (t->defined() && t->scalar_type() == at::kFloat) bits |= bit;
        bit *= 2;
    }
    return bits;
}

// act(x W + bias) + residual, W [in, out] (CW_NN) or [out, in] (CW_NT): parallel_2d._operation._SUMMA_AB, parallel_1d._operation._LinearNT.
struct Linear : Function<Linear> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x_in, const Tensor& w_in, const OptTensor& bias_in, const OptTensor& residual_in,
                          int64_t layout, int64_t act) {
        Tensor x = x_in, w = w_in, bias = def(bias_in), residual = def(residual_in);
        const bool cast = autocast();
        const auto asked = cast ? at::autocast::get_autocast_dtype(at::kCUDA) : at::kHalf;
        const int64_t given = fp32_inputs({&x, &w, &bias});
        Body body;
        if (cast) cast_inputs({&x, &w, &bias, &residual}, half_type(asked) ? asked : at::kHalf);
        const int64_t N = w.size(layout == CW_NN ? 1 : 0);
        std::vector<Tensor> addends;
        if (residual.defined()) addends.push_back(residual.reshape({-1, N}));
        // ReLU needs no separate pre-activation: its derivative [pre > 0] is [out > 0], so the output serves
        auto [out, pre] = gemm_ksteps((int)layout, {x.reshape({-1, x.size(-1)})}, {w}, opt(bias),
                                      act != CW_ACT_NONE ? (int)act : bias.defined() ? CW_EPI_BIAS : CW_EPI_NONE, addends,
                                      act != CW_ACT_NONE && act != CW_ACT_RELU, {});
        ctx->save_for_backward({x, w, act == CW_ACT_RELU ? out : def(pre)});
        keep(ctx, {layout, act, bias.defined() ? (int64_t)bias.scalar_type() : -1, residual.defined(), given & ~fp32_inputs({&x, &w, &bias})});
        auto shape = x.sizes().vec();
        shape.back() = N;
        return out.reshape(shape);
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        Body body;
        const auto saved = ctx->get_saved_variables();
        const auto meta = kept(ctx);
        const Tensor &x = saved[0], &w = saved[1], &pre = saved[2];
        const int layout = (int)meta[0], act = (int)meta[1];
        const bool has_bias = meta[2] >= 0, need_x = ctx->needs_input_grad(0), need_w = ctx->needs_input_grad(1);
        const auto sum_type = has_bias ? std::optional((at::ScalarType)meta[2]) : std::nullopt;
        const Tensor x2 = x.reshape({-1, x.size(-1)});
        Tensor g = grads[0].reshape({-1, grads[0].size(-1)}), dbias, dx, dw;
        if (act != CW_ACT_NONE) {
            auto [dpre, sums] = act_bwd_colsum(act, g, pre, has_bias, sum_type);
            g = dpre;
            dbias = def(sums);
        } else if (has_bias) {
            dbias = colsum(g, sum_type);
        }
        if (layout == CW_NT && need_x && need_w) g = aligned_rows(g);
        if (need_x) dx = std::get<0>(gemm_ksteps(layout == CW_NN ? CW_NT : CW_NN, {g}, {w}, {}, CW_EPI_NONE, {}, false, {})).reshape(x.sizes());
        if (need_w)
            dw = std::get<0>(layout == CW_NN ? gemm_ksteps(CW_TN, {x2}, {g}, {}, CW_EPI_NONE, {}, false, {})
                                             : gemm_ksteps(CW_TN, {g}, {x2}, {}, CW_EPI_NONE, {}, false, {}));
        // gradients of inputs that were cast, which autograd would cast one by one
        if (const int64_t was_fp32 = meta[4]; was_fp32 != 0) {
            Tensor none;
            cast_together({was_fp32 & 1 ? &dx : &none, was_fp32 & 2 ? &dw : &none, was_fp32 & 4 ? &dbias : &none}, at::kFloat);
        }
        // absent operands are no inputs of the node, and have no index there
        const bool need_residual = has_residual(*ctx) && ctx->needs_input_grad(has_bias ? 3 : 2);
        return {dx, dw, dbias, need_residual ? grads[0] : Tensor(), Tensor(), Tensor()};
    }
    static bool has_residual(const AutogradContext& ctx) { return kept(&ctx)[3] != 0; }
};

py::object linear(py::handle x_in, py::handle w_in, py::handle bias_in, py::handle residual_in, int layout, int act) {
    Tensor x, w, bias, residual;
    if (!ordinary() || !take(x_in, x) || !take(w_in, w) || !take(bias_in, bias, true) || !take(residual_in, residual, true)) return py::none();
    if (x.dim() < (layout == CW_NN ? 2 : 1) || w.dim() != 2 || x.size(-1) != w.size(layout == CW_NN ? 0 : 1) || x.size(-1) == 0 || (residual.defined() && act != CW_ACT_NONE) ||
        !together({x, w, bias, residual}))
        return py::none();
    auto shape = x.sizes().vec();
    shape.back() = w.size(layout == CW_NN ? 1 : 0);
    if (shape.back() == 0 || (residual.defined() && residual.sizes() != at::IntArrayRef(shape))) return py::none();
    Tensor out;
    {
        py::gil_scoped_release no_gil;
        out = Linear::apply(x, w, opt(bias), opt(residual), (int64_t)layout, (int64_t)act);
    }
    return py::cast(out);
}

// parallel_2d._operation._Layernorm2D over rows that are whole on this rank.
struct LayerNorm : Function<LayerNorm> {
    static variable_list forward(AutogradContext* ctx, const Tensor& x_in, const Tensor& w_in, const Tensor& b_in, double eps, bool fork) {
        Tensor x = x_in, w = w_in, b = b_in;
        const bool cast = autocast();
        Body body;
        if (cast) cast_inputs({&x, &w, &b}, at::kFloat);
        auto [out, mean_rstd] = ln_forward(x, {}, {}, 0, eps, w, b, CW_LN_ONE_PASS, true);
        ctx->save_for_backward({x, w, *mean_rstd});
        keep(ctx, {(int64_t)w.scalar_type(), (int64_t)b.scalar_type()});
        if (fork) return {out, x.view_as(x)};
        return {out};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        Body body;
        const auto saved = ctx->get_saved_variables();
        const auto meta = kept(ctx);
        const auto wt = (at::ScalarType)meta[0], bt = (at::ScalarType)meta[1];
        auto [dx, dw, db] = ln_backward_fused(grads[0], saved[0], saved[2], saved[1], true, wt == bt ? std::optional(wt) : std::nullopt,
                                              grads.size() > 1 ? opt(grads[1]) : OptTensor());
        return {dx, dw->to(wt), db->to(bt), Tensor(), Tensor()};
    }
};

py::object layernorm(py::handle x_in, py::handle w_in, py::handle b_in, double eps, bool fork) {
    Tensor x, w, b;
    if (!ordinary() || !take(x_in, x) || !take(w_in, w) || !take(b_in, b)) return py::none();
    if (x.dim() < 1 || w.dim() != 1 || b.dim() != 1 || w.size(0) != x.size(-1) || b.size(0) != x.size(-1) || x.numel() == 0 || !together({x, w, b}))
        return py::none();
    for (const Tensor* t : {&x, &w, &b})
        if (t->scalar_type() != at::kFloat && !half_type(t->scalar_type())) return py::none();
    variable_list out;
    {
        py::gil_scoped_release no_gil;
        out = LayerNorm::apply(x, w, b, eps, fork);
    }
    return fork ? py::object(py::make_tuple(out[0], out[1])) : py::cast(out[0]);
}

// ops._AttentionCore for heads that the kernels read as they lie in a contiguous qkv.
struct Attention : Function<Attention> {
    static Tensor forward(AutogradContext* ctx, const Tensor& qkv, int64_t heads, double scale, bool causal) {
        Body body;
        const int64_t B = qkv.size(0), S = qkv.size(1), D = qkv.size(2) / (3 * heads);
        Tensor out = empty({B, S, heads * D}, qkv), lse = empty({B, heads, S}, qkv, at::kFloat);
        const auto* p = (const uint16_t*)ptr(qkv);
        const bool narrow = D != 64 && D != 128;
        check((narrow ? lib.cw_attn_narrow_fwd : lib.cw_attn_fwd)(B, heads, S, D, p, p + D, p + 2 * D, S * heads * 3 * D, heads * 3 * D, 3 * D,
                                                                  (float)scale, causal, ptr(out), S * heads * D, heads * D, D, (float*)ptr(lse),
                                                                  dtype_code(qkv.scalar_type()), stream()),
              narrow ? "cw_attn_narrow_fwd" : "cw_attn_fwd");
        ctx->save_for_backward({qkv, out, lse});
        keep(ctx, {heads, causal});
        ctx->saved_data["scale"] = scale;
        return out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        Body body;
        const auto saved = ctx->get_saved_variables();
        const auto meta = kept(ctx);
        const Tensor &qkv = saved[0], &out = saved[1];
        const int64_t heads = meta[0], B = qkv.size(0), S = qkv.size(1), D = qkv.size(2) / (3 * heads);
        const bool narrow = D != 64 && D != 128;
        Tensor d_out = grads[0].contiguous(), dqkv = empty(qkv.sizes(), qkv), ws = bytes(std::max<int64_t>(lib.cw_attn_bwd_workspace_bytes(B, heads, S), 16), qkv);
        if (narrow && !aligned16(d_out)) d_out = d_out.clone();
        const auto* p = (const uint16_t*)ptr(qkv);
        auto* g = (uint16_t*)ptr(dqkv);
        const int64_t sb = S * heads * 3 * D, st = heads * 3 * D, sh = 3 * D;
        check((narrow ? lib.cw_attn_narrow_bwd : lib.cw_attn_bwd)(B, heads, S, D, p, p + D, p + 2 * D, sb, st, sh, ptr(out), ptr(d_out), S * heads * D,
                                                                  heads * D, D, (const float*)ptr(saved[2]), (float)ctx->saved_data["scale"].toDouble(),
                                                                  meta[1] != 0, g, g + D, g + 2 * D, sb, st, sh, ptr(ws), ws.numel(),
                                                                  dtype_code(qkv.scalar_type()), stream()),
              narrow ? "cw_attn_narrow_bwd" : "cw_attn_bwd");
        return {dqkv, Tensor(), Tensor(), Tensor()};
    }
};

py::object attention(py::handle qkv_in, int64_t heads, std::optional<double> scale, bool causal) {
    Tensor qkv;
    if (!ordinary() || !take(qkv_in, qkv)) return py::none();
    if (qkv.dim() != 3 || heads < 1 || !half_type(qkv.scalar_type()) || !qkv.is_contiguous() || qkv.numel() == 0 || qkv.size(2) % (3 * heads) != 0)
        return py::none();
    const int64_t D = qkv.size(2) / (3 * heads);
    if (D != 64 && D != 128 && !(D % 8 == 0 && D < 128 && aligned16(qkv) && qkv.size(2) < (1 << 23))) return py::none();
    Tensor out;
    {
        py::gil_scoped_release no_gil;
        out = Attention::apply(qkv, heads, scale.value_or(std::pow((double)D, -0.5)), causal);
    }
    return py::cast(out);
}

// ops._VocabEmbedding.
struct Embedding : Function<Embedding> {
    static Tensor forward(AutogradContext* ctx, const Tensor& ids, const Tensor& weight, int64_t start, int64_t skip_row) {
        Body body;
        const Tensor w = rows(weight), flat = ids.reshape({-1}).to(at::kLong).contiguous();
        auto shape = ids.sizes().vec();
        shape.push_back(w.size(1));
        Tensor out = empty(shape, w);
        check(lib.cw_embed_fwd(flat.numel(), w.size(1), (const int64_t*)ptr(flat), start, w.size(0), ptr(w), ld(w), ptr(out), w.size(1),
                               dtype_code(w.scalar_type()), stream()),
              "cw_embed_fwd");
        ctx->save_for_backward({ids});
        keep(ctx, {w.size(0), start, skip_row});
        return out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        Body body;
        const Tensor ids = ctx->get_saved_variables()[0], g = rows(grads[0].reshape({-1, grads[0].size(-1)})), flat = ids.reshape({-1}).to(at::kLong).contiguous();
        const auto meta = kept(ctx);
        const int64_t T = g.size(0), E = g.size(1), V = meta[0], start = meta[1], skip = meta[2];
        const int dt = dtype_code(g.scalar_type());
        Tensor dw = empty({V, E}, g);
        bool done = false;
        if (lib.cw_embed_bwd_ids_supported(T, E, ptr(g), ld(g), ptr(dw), ld(dw), dt)) {
            const int rc = lib.cw_embed_bwd_ids(T, E, (const int64_t*)ptr(flat), start, V, skip, ptr(g), ld(g), ptr(dw), ld(dw), dt, stream());
            done = rc != CW_ERR_UNSUPPORTED;
            if (done) check(rc, "cw_embed_bwd_ids");
        }
        if (!done) {
            const int64_t need = lib.cw_embed_sort_workspace_bytes(T);
            Tensor sorted = empty({T}, flat), order = empty({T}, flat), ws = bytes(need, flat);
            check(lib.cw_embed_sort_ids(T, (const int64_t*)ptr(flat), start, V, (int64_t*)ptr(sorted), (int64_t*)ptr(order), need > 0 ? ptr(ws) : nullptr, need,
                                        stream()),
                  "cw_embed_sort_ids");
            check(lib.cw_embed_bwd(T, E, (const int64_t*)ptr(sorted), (const int64_t*)ptr(order), start, V, skip, ptr(g), ld(g), ptr(dw), ld(dw), dt, stream()),
                  "cw_embed_bwd");
        }
        return {Tensor(), dw, Tensor(), Tensor()};
    }
};

py::object embedding(py::handle ids_in, py::handle weight_in, int64_t start, int64_t skip_row) {
    Tensor ids, weight;
    if (!ordinary() || !take(ids_in, ids) || !take(weight_in, weight)) return py::none();
    if ((ids.scalar_type() != at::kLong && ids.scalar_type() != at::kInt) || weight.dim() != 2 || ids.numel() == 0 || weight.numel() == 0 ||
        !together({ids, weight}))
        return py::none();
    Tensor out;
    {
        py::gil_scoped_release no_gil;
        out = Embedding::apply(ids, weight, start, skip_row);
    }
    return py::cast(out);
}

// Whether the gradient that the running node hands to its first input's node is read by that node's own kernels alone, those of a
// layer without a residual (which would hand the gradient on as it is): no hook before, at or behind that node sees it and nobody asked
// for it. It may then have rows that begin at multiples of 16 bytes whatever their length, as both gradient products read them.
// (autograd's other readers, a logits tensor with a second use among them, take any strides.)
bool for_a_product_only() {
    const auto node = torch::autograd::get_current_node();
    const auto* asked = torch::autograd::get_current_graph_task_exec_info();  // empty for backward() without inputs
    if (!node || !node->post_hooks().empty() || asked == nullptr || !asked->empty() || node->num_outputs() == 0) return false;
    const auto& next = node->next_edge(0).function;
    const auto* linear = dynamic_cast<torch::autograd::CppNode<Linear>*>(next.get());
    return linear != nullptr && !Linear::has_residual(linear->ctx_) && next->pre_hooks().empty() && next->tensor_pre_hooks().empty() &&
           next->retains_grad_hooks().empty() && next->post_hooks().empty();
}

// loss._operation._VocabParallelCrossEntropyMean.
struct MeanLoss : Function<MeanLoss> {
    static Tensor forward(AutogradContext* ctx, const Tensor& logits, const Tensor& targets, int64_t start, const std::vector<Tensor>* peers) {
        Body body;
        const Tensor flat = logits.reshape({-1, logits.size(-1)}), t = targets.reshape({-1});
        auto [loss, total] = vpce_mean(flat, t, start, *peers);
        ctx->save_for_backward({flat, t, total});
        auto meta = logits.sizes().vec();
        meta.push_back(start);
        keep(ctx, std::move(meta));
        return loss;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        Body body;
        const auto saved = ctx->get_saved_variables();
        auto shape = kept(ctx);
        const int64_t start = shape.back();
        shape.pop_back();
        // rows of an odd vocabulary: dense ones would be copied for the products (1023 x 50257 bf16: 43 us, 0.2 GB)
        const bool aligned = saved[0].element_size() == 2 && saved[0].size(1) % 8 != 0 && for_a_product_only();
        return {vpce_mean_bwd(saved[0], saved[1], start, saved[2], grads[0], aligned).reshape(shape), Tensor(), Tensor(), Tensor()};
    }
};

py::object mean_loss(py::handle logits_in, py::handle targets_in, int64_t start, const std::vector<Tensor>& peers) {
    Tensor logits, targets;
    if (!ordinary() || !take(logits_in, logits) || !take(targets_in, targets)) return py::none();
    if (logits.dim() < 1 || logits.numel() == 0 || (logits.scalar_type() != at::kFloat && !half_type(logits.scalar_type())) || !together({logits, targets}))
        return py::none();
    Tensor out;
    {
        py::gil_scoped_release no_gil;
        out = MeanLoss::apply(logits, targets, start, &peers);
    }
    return py::cast(out);
}

}  // namespace

void def_nodes(py::module_& m) {
    m.def("linear", &linear);
    m.def("layernorm", &layernorm);
    m.def("attention", &attention);
    m.def("embedding", &embedding);
    m.def("mean_loss", &mean_loss);
}

}  // namespace cw_host
