// The operators' host side as one native call each: shape and type checks, output and scratch allocation through torch, the
// current stream, the C ABI entry point. A small training step is bound by this work (a block of 128 tokens: about 30
// launches, 0.2 ms on the GPU), and through Python and ctypes an operator costs 15 to 30 us of it; here 5 to 8 us, most of
// them the launches.
// The entry points' addresses come from the library that cubework_amd._lib loaded (bind), so a measurement build selected
// there is the one that runs. Calls run without the interpreter lock. Errors: ValueError, TypeError and RuntimeError as
// the Python wrappers document, CubeworkHipError (raised by cubework_amd._lib.check) for a status of the library.
#include "host_ops.h"

#include <c10/hip/HIPStream.h>

namespace cw_host {

Entries lib;

void bind(const std::map<std::string, uintptr_t>& addresses) {
#define X(name) lib.name = reinterpret_cast<decltype(lib.name)>(addresses.at(#name));
    CW_HOST_ENTRIES(X)
#undef X
}

void check(int status, const char* what) {
    if (status == 0) return;
    py::gil_scoped_acquire gil;
    py::module_::import("cubework_amd._lib").attr("check")(status, what);
}

int dtype_code(at::ScalarType t) {
    if (t == at::kBFloat16) return CW_BF16;
    if (t == at::kFloat) return CW_F32;
    if (t == at::kHalf) return CW_F16;
    TORCH_CHECK_TYPE(false, "the cubework_amd kernels take bfloat16, float16 or float32 tensors, got ", t);
}
// Type of column sums and parameter gradients: fp32 unless the caller names another.
at::ScalarType sum_type(std::optional<at::ScalarType> t) {
    const at::ScalarType s = t.value_or(at::kFloat);
    TORCH_CHECK_TYPE(s == at::kFloat || s == at::kBFloat16 || s == at::kHalf,
                     "column sums are stored as float32, bfloat16 or float16, not ", s);
    return s;
}

void on_device(const Tensor& t) {
    TORCH_CHECK(t.is_cuda(), "cubework_amd operators run on the GPU only (got a ", t.device(), " tensor); there is no CPU fallback");
}
void on_device(const OptTensor& t) {
    if (t) on_device(*t);
}

Tensor rows(const Tensor& t) {
    Tensor r = t.dim() == 2 ? t : t.reshape({-1, t.size(-1)});
    if (r.stride(1) != 1 || (r.size(0) > 1 && r.stride(0) < r.size(1))) r = r.contiguous();
    return r;
}
int64_t ld(const Tensor& t) { return t.size(0) > 1 ? t.stride(0) : std::max<int64_t>(t.size(1), 1); }
int64_t ld(const OptTensor& t) { return t ? ld(*t) : 0; }
void* ptr(const OptTensor& t) { return t ? t->data_ptr() : nullptr; }
void* stream() { return c10::hip::getCurrentHIPStream().stream(); }
OptTensor vec(const OptTensor& t, at::ScalarType type) {
    if (!t) return t;
    return t->to(type).contiguous();
}
Tensor colsum_workspace(int64_t M, int64_t N, const Tensor& like) { return bytes(std::max<int64_t>(lib.cw_colsum_workspace_bytes(M, N), 16), like); }

// The other ranks' summands of a vector or of rows' pairs. The kernels read them where they arrived if they are what a rank of this
// kind sends (fp32, contiguous, as many elements); anything else that torch can add is added here, in the same order.
using Peers = std::vector<Tensor>;
bool direct(const Peers& peers, const Tensor& own) {
    if (peers.size() > CW_MAX_ADDENDS || own.scalar_type() != at::kFloat) return false;
    for (const auto& t : peers)
        if (t.scalar_type() != at::kFloat || t.sizes() != own.sizes() || !t.is_contiguous() || t.device() != own.device()) return false;
    return true;
}
std::vector<const float*> pointers(const Peers& peers) {
    std::vector<const float*> p;
    for (const auto& t : peers) p.push_back((const float*)ptr(t));
    return p;
}
Tensor add_peers(Tensor own, const Peers& peers) {
    for (const auto& t : peers) own = own + t;
    return own;
}
// This rank's share of column sums that are reduce-scattered over `world` ranks, stored as `type`.
struct Scatter {
    Peers peers;
    int64_t world = 1, rank = 0;
    at::ScalarType type = at::kFloat;
    bool fused(const Tensor& own) const {
        return !peers.empty() && own.dim() == 1 && own.size(0) % world == 0 && (type == at::kFloat || type == at::kBFloat16 || type == at::kHalf) &&
               direct(peers, own);
    }
    int64_t count(const Tensor& own) const { return own.size(0) / world; }
    Tensor general(const Tensor& own) const { return add_peers(own, peers).chunk(world, -1).at(rank).contiguous().to(type); }
};

// -> (C, preact or None). See ops.gemm_ksteps.
std::tuple<Tensor, OptTensor> gemm_ksteps(int layout, std::vector<Tensor> A, std::vector<Tensor> B, const OptTensor& bias_in, int epilogue,
                                          std::vector<Tensor> addends, bool want_preact, const OptTensor& out_in) {
    TORCH_CHECK_VALUE(!A.empty() && A.size() == B.size(), "need the same, non-zero number of A and B step operands");
    for (auto& t : A) t = rows(t);
    for (auto& t : B) t = rows(t);
    for (const auto& t : A) on_device(t);
    for (const auto& t : B) on_device(t);
    on_device(bias_in);
    for (const auto& t : addends) on_device(t);
    const Tensor &a0 = A[0], &b0 = B[0];
    const at::ScalarType type = a0.scalar_type();
    const int dt = dtype_code(type);
    const int64_t M = a0.size(layout == CW_TN ? 1 : 0), K = a0.size(layout == CW_TN ? 0 : 1);
    const int64_t N = b0.size(layout == CW_NT ? 0 : 1), Kb = b0.size(layout == CW_NT ? 1 : 0);
    TORCH_CHECK_VALUE(K == Kb, "reduction sizes differ: A ", a0.sizes(), ", B ", b0.sizes(), " for layout ", layout == CW_NN ? "NN" : layout == CW_NT ? "NT" : "TN");
    const int64_t lda = ld(a0), ldb = ld(b0);
    bool al_a = true, al_b = true;
    for (const auto* set : {&A, &B})
        for (const auto& t : *set) TORCH_CHECK_TYPE(t.scalar_type() == type, "all GEMM operands must share one dtype");
    for (const auto& t : A) {
        TORCH_CHECK_VALUE(t.sizes() == a0.sizes() && ld(t) == lda, "A step operands must share shape and leading dimension");
        al_a = al_a && aligned16(t);
    }
    for (const auto& t : B) {
        TORCH_CHECK_VALUE(t.sizes() == b0.sizes() && ld(t) == ldb, "B step operands must share shape and leading dimension");
        al_b = al_b && aligned16(t);
    }
    if (bias_in) TORCH_CHECK_VALUE(bias_in->numel() == N, "bias has ", bias_in->numel(), " elements, output width is ", N);
    const OptTensor bias = vec(bias_in, type);
    for (auto& t : addends) {
        t = rows(t);
        TORCH_CHECK_VALUE(t.size(0) == M && t.size(1) == N && t.scalar_type() == type, "addends must be [M,N] of the operand dtype");
    }
    // the C ABI takes one leading dimension for all addends: copy those that are laid out differently
    int64_t ldadd = addends.empty() ? 0 : ld(addends[0]);
    bool same = true;
    for (auto& t : addends) {
        if (ld(t) != ldadd) t = t.contiguous();
        same = same && ld(t) == ldadd;
    }
    if (!same) {
        ldadd = N;
        for (auto& t : addends) t = t.contiguous();
    }
    bool al_add = ldadd % 8 == 0;
    for (const auto& t : addends) al_add = al_add && aligned16(t);
    if (out_in)
        TORCH_CHECK_VALUE(out_in->dim() == 2 && out_in->size(0) == M && out_in->size(1) == N && out_in->scalar_type() == type && out_in->stride(1) == 1,
                          "out must be a row-major [M,N] tensor of the operand dtype");
    Tensor out = out_in ? *out_in : empty({M, N}, a0);
    OptTensor pre;
    if (want_preact) pre = empty({M, N}, a0);
    std::vector<const void*> pa, pb, pd;
    for (const auto& t : A) pa.push_back(ptr(t));
    for (const auto& t : B) pb.push_back(ptr(t));
    for (const auto& t : addends) pd.push_back(ptr(t));
    // scratch for tiles cut along k and for copies of operands with unaligned rows
    const int n = (int)A.size(), n_add = (int)addends.size();
    const int64_t need = lib.cw_gemm_scratch_bytes(layout, M, N, K, n, lda, ldb, al_a, al_b, al_add ? 0 : n_add, dt);
    OptTensor ws;
    if (need > 0) ws = bytes(need, a0);
    check(lib.cw_gemm_ksteps_ws(layout, M, N, K, n, pa.data(), lda, pb.data(), ldb, ptr(bias), epilogue, ptr(out), ld(out), ptr(pre),
                                ld(pre), pd.data(), n_add, ldadd, ptr(ws), need, dt, stream()),
          "cw_gemm_ksteps_ws");
    return {out, pre};
}

void cast_together(std::initializer_list<Tensor*> ts, at::ScalarType type) {
    auto half = [](at::ScalarType t) { return t == at::kBFloat16 || t == at::kHalf; };
    const void* src[CW_MAX_CASTS];
    void* dst[CW_MAX_CASTS];
    int64_t n[CW_MAX_CASTS];
    Tensor to[CW_MAX_CASTS], *of[CW_MAX_CASTS];
    int count = 0;
    at::ScalarType from = at::kFloat;
    for (Tensor* t : ts) {
        if (!t->defined() || t->scalar_type() == type) continue;
        const at::ScalarType own = t->scalar_type();
        const bool ours = (own == at::kFloat ? half(type) : half(own) && type == at::kFloat) && (count == 0 || own == from) && count < CW_MAX_CASTS &&
                          t->is_contiguous() && aligned16(*t) && t->numel() > 0 && t->numel() < ((int64_t)1 << 33);
        if (!ours) {
            *t = t->to(type);
            continue;
        }
        from = own;
        to[count] = empty(t->sizes(), *t, type);
        src[count] = ptr(*t);
        dst[count] = ptr(to[count]);
        n[count] = t->numel();
        of[count++] = t;
    }
    if (count == 0) return;
    check(lib.cw_cast_many(count, src, dst, n, dtype_code(from), dtype_code(type), stream()), "cw_cast_many");
    for (int i = 0; i < count; ++i) *of[i] = to[i];
}

Tensor colsum(const Tensor& dy_in, std::optional<at::ScalarType> out_type) {
    const Tensor dy = rows(dy_in);
    on_device(dy);
    const at::ScalarType st = sum_type(out_type);
    const int64_t M = dy.size(0), N = dy.size(1);
    Tensor out = empty({N}, dy, st), ws = colsum_workspace(M, N, dy);
    check(lib.cw_colsum(M, N, ptr(dy), ld(dy), ptr(out), dtype_code(st), ptr(ws), ws.numel(), dtype_code(dy.scalar_type()), stream()), "cw_colsum");
    return out;
}

std::tuple<Tensor, OptTensor> act_bwd_colsum(int activation, const Tensor& dy_in, const Tensor& pre_in, bool want_dbias,
                                             std::optional<at::ScalarType> out_type) {
    const Tensor dy = rows(dy_in), pre = rows(pre_in);
    on_device(dy);
    on_device(pre);
    TORCH_CHECK_VALUE(dy.sizes() == pre.sizes() && dy.scalar_type() == pre.scalar_type(), "dy and preact must agree in shape and dtype");
    const at::ScalarType st = sum_type(out_type);
    const int64_t M = dy.size(0), N = dy.size(1);
    Tensor dpre = empty({M, N}, dy);
    OptTensor dbias, ws;
    if (want_dbias) {
        dbias = empty({N}, dy, st);
        ws = colsum_workspace(M, N, dy);
    }
    check(lib.cw_act_bwd_colsum(activation, M, N, ptr(dy), ld(dy), ptr(pre), ld(pre), ptr(dpre), ld(dpre), ptr(dbias), dtype_code(st), ptr(ws),
                                ws ? ws->numel() : 0, dtype_code(dy.scalar_type()), stream()),
          "cw_act_bwd_colsum");
    return {dpre, dbias};
}

// Column sums (of dPre = dy * act'(pre) if there is an activation) reduce-scattered over the ranks: -> (dPre or None, this rank's share).
std::tuple<OptTensor, Tensor> colsum_scattered(const Tensor& dy_in, int activation, const OptTensor& pre_in, Peers peers, int64_t world,
                                               int64_t rank, at::ScalarType type) {
    const Tensor dy = rows(dy_in);
    on_device(dy);
    const int64_t M = dy.size(0), N = dy.size(1);
    const Scatter sc{std::move(peers), world, rank, type};
    Tensor own = empty({N}, dy, at::kFloat), ws = colsum_workspace(M, N, dy);
    const bool fused = sc.fused(own);
    const int64_t count = fused ? sc.count(own) : 0;
    OptTensor reduced, pre, dpre;
    if (fused) reduced = empty({count}, dy, sum_type(type));
    const auto table = pointers(fused ? sc.peers : Peers{});
    if (pre_in) {
        pre = rows(*pre_in);
        on_device(pre);
        TORCH_CHECK_VALUE(dy.sizes() == pre->sizes() && dy.scalar_type() == pre->scalar_type(), "dy and preact must agree in shape and dtype");
        dpre = empty({M, N}, dy);
        check(lib.cw_act_bwd_colsum_peers(activation, M, N, ptr(dy), ld(dy), ptr(pre), ld(pre), ptr(dpre), ld(dpre), ptr(own), CW_F32, ptr(ws),
                                          ws.numel(), table.data(), (int)table.size(), rank * count, count, ptr(reduced),
                                          fused ? dtype_code(type) : CW_F32, dtype_code(dy.scalar_type()), stream()),
              "cw_act_bwd_colsum_peers");
    } else {
        check(lib.cw_colsum_peers(M, N, ptr(dy), ld(dy), ptr(own), CW_F32, ptr(ws), ws.numel(), table.data(), (int)table.size(), rank * count,
                                  count, ptr(reduced), fused ? dtype_code(type) : CW_F32, dtype_code(dy.scalar_type()), stream()),
              "cw_colsum_peers");
    }
    return {dpre, fused ? *reduced : sc.general(own)};
}

// Statistics of x and, by the same launch, the affine parameters gathered from their ranks' parts: -> (stats, gamma, beta).
std::tuple<Tensor, Tensor, Tensor> ln_partial_stats_gather(const Tensor& x_in, std::vector<Tensor> gammas, std::vector<Tensor> betas) {
    const Tensor x = rows(x_in);
    on_device(x);
    const int64_t R = x.size(0), C = x.size(1), n = (int64_t)gammas.size();
    bool fused = R > 0 && n >= 1 && n <= CW_MAX_ADDENDS && betas.size() == gammas.size() && C % n == 0;
    for (const auto* set : {&gammas, &betas})
        for (const auto& t : *set)
            fused = fused && t.dim() == 1 && t.numel() * n == C && t.scalar_type() == x.scalar_type() && t.is_contiguous() && t.device() == x.device();
    Tensor stats = empty({R, 2}, x, at::kFloat);
    if (!fused) {
        check(lib.cw_ln_partial_stats(R, C, ptr(x), ld(x), CW_LN_ONE_PASS, nullptr, (float*)ptr(stats), dtype_code(x.scalar_type()), stream()),
              "cw_ln_partial_stats");
        return {stats, at::cat(gammas, -1), at::cat(betas, -1)};
    }
    Tensor gamma = empty({C}, x), beta = empty({C}, x);
    std::vector<const void*> pg, pb;
    for (const auto& t : gammas) pg.push_back(ptr(t));
    for (const auto& t : betas) pb.push_back(ptr(t));
    check(lib.cw_ln_partial_stats_gather(R, C, ptr(x), ld(x), (float*)ptr(stats), pg.data(), pb.data(), (int)n, ptr(gamma), ptr(beta),
                                         dtype_code(x.scalar_type()), stream()),
          "cw_ln_partial_stats_gather");
    return {stats, gamma, beta};
}

Tensor ln_partial_stats(const Tensor& x_in, int mode, const OptTensor& mean_in) {
    const Tensor x = rows(x_in);
    on_device(x);
    on_device(mean_in);
    Tensor stats = empty({x.size(0), 2}, x, at::kFloat);
    OptTensor mean;
    if (mean_in) {
        mean = mean_in->reshape({-1}).to(at::kFloat).contiguous();
        TORCH_CHECK_VALUE(mean->numel() == x.size(0), "mean must have one entry per row");
    }
    check(lib.cw_ln_partial_stats(x.size(0), x.size(1), ptr(x), ld(x), mode, (const float*)ptr(mean), (float*)ptr(stats),
                                  dtype_code(x.scalar_type()), stream()),
          "cw_ln_partial_stats");
    return stats;
}

// stats given: ln_normalize of their sum with the peers'; else ln_forward_fused.
std::tuple<Tensor, OptTensor> ln_forward(const Tensor& x_in, const OptTensor& stats_in, Peers peers, int64_t hidden, double eps,
                                         const OptTensor& gamma_in, const OptTensor& beta_in, int mode, bool save_mean_rstd) {
    const Tensor x = rows(x_in);
    on_device(x);
    on_device(stats_in);
    on_device(gamma_in);
    on_device(beta_in);
    const int64_t R = x.size(0), C = x.size(1);
    OptTensor stats;
    if (stats_in) {
        if (!direct(peers, *stats_in)) stats = add_peers(*stats_in, std::exchange(peers, {}));
        stats = stats.value_or(*stats_in).reshape({R, 2}).to(at::kFloat).contiguous();
    }
    const auto table = pointers(peers);
    const OptTensor gamma = vec(gamma_in, x.scalar_type()), beta = vec(beta_in, x.scalar_type());
    if (stats)
        for (const auto* v : {&gamma, &beta}) TORCH_CHECK_VALUE(!*v || (*v)->numel() == C, "gamma/beta must have C elements");
    Tensor y = empty({R, C}, x);
    OptTensor mr;
    if (save_mean_rstd) mr = empty({R, 2}, x, at::kFloat);
    const int dt = dtype_code(x.scalar_type());
    if (stats)
        check(lib.cw_ln_normalize_peers(R, C, ptr(x), ld(x), (const float*)ptr(stats), table.data(), (int)table.size(), mode, hidden, (float)eps,
                                        ptr(gamma), ptr(beta), ptr(y), ld(y), (float*)ptr(mr), dt, stream()),
              "cw_ln_normalize_peers");
    else
        check(lib.cw_ln_forward_fused(R, C, ptr(x), ld(x), mode, (float)eps, ptr(gamma), ptr(beta), ptr(y), ld(y), (float*)ptr(mr), dt, stream()),
              "cw_ln_forward_fused");
    return {y.sizes() == x_in.sizes() ? y : y.reshape(x_in.sizes()), mr};
}

struct LnBackward {
    Tensor dy, x;
    OptTensor gamma;
    int64_t R, C;
    int dt;
};
LnBackward ln_backward_inputs(const Tensor& dy_in, const Tensor& x_in, const Tensor& mean_rstd, const OptTensor& row_sums, const OptTensor& gamma) {
    LnBackward b{rows(dy_in), rows(x_in), {}, 0, 0, 0};
    on_device(b.dy);
    on_device(b.x);
    on_device(mean_rstd);
    on_device(row_sums);
    on_device(gamma);
    TORCH_CHECK_VALUE(b.dy.sizes() == b.x.sizes() && b.dy.scalar_type() == b.x.scalar_type(), "dy and x must agree in shape and dtype");
    b.gamma = vec(gamma, b.x.scalar_type());
    b.R = b.x.size(0);
    b.C = b.x.size(1);
    b.dt = dtype_code(b.x.scalar_type());
    return b;
}

std::tuple<Tensor, OptTensor, OptTensor> ln_backward_fused(const Tensor& dy_in, const Tensor& x_in, const Tensor& mean_rstd,
                                                           const OptTensor& gamma, bool want_param_grads,
                                                           std::optional<at::ScalarType> param_type, const OptTensor& addend) {
    const LnBackward b = ln_backward_inputs(dy_in, x_in, mean_rstd, {}, gamma);
    Tensor row_sums = empty({b.R, 2}, b.x, at::kFloat), dx = empty({b.R, b.C}, b.x);
    const at::ScalarType pt = sum_type(param_type);
    OptTensor dgamma, dbeta, ws, add;
    if (want_param_grads) {
        dgamma = empty({b.C}, b.x, pt);
        dbeta = empty({b.C}, b.x, pt);
        ws = colsum_workspace(b.R, b.C, b.x);
    }
    if (addend) {
        add = rows(*addend);
        TORCH_CHECK_VALUE(add->sizes() == b.x.sizes() && add->scalar_type() == b.x.scalar_type(), "dx_addend must agree with x in shape and dtype");
        on_device(add);
    }
    auto call = [&](const OptTensor& a) {
        return lib.cw_ln_backward_fused(b.R, b.C, ptr(b.dy), ld(b.dy), ptr(b.x), ld(b.x), (const float*)ptr(mean_rstd), ptr(b.gamma),
                                        (float*)ptr(row_sums), ptr(dx), ld(dx), ptr(a), ld(a), ptr(dgamma), ptr(dbeta), dtype_code(pt), ptr(ws),
                                        ws ? ws->numel() : 0, b.dt, stream());
    };
    int rc = call(add);
    if (rc == CW_ERR_UNSUPPORTED && add) {  // a shape of the two-kernel path: add separately
        rc = call({});
        check(rc, "cw_ln_backward_fused");
        dx = dx + *add;
    }
    check(rc, "cw_ln_backward_fused");
    return {dx.sizes() == x_in.sizes() ? dx : dx.reshape(x_in.sizes()), dgamma, dbeta};
}

// -> (row_sums, workspace, number of partial rows in it)
std::tuple<Tensor, Tensor, int64_t> ln_bwd_partials_open(const Tensor& dy_in, const Tensor& x_in, const Tensor& mean_rstd, const OptTensor& gamma) {
    const LnBackward b = ln_backward_inputs(dy_in, x_in, mean_rstd, {}, gamma);
    Tensor row_sums = empty({b.R, 2}, b.x, at::kFloat), ws = colsum_workspace(b.R, b.C, b.x);
    int64_t parts = 0;
    check(lib.cw_ln_bwd_partials_open(b.R, b.C, ptr(b.dy), ld(b.dy), ptr(b.x), ld(b.x), (const float*)ptr(mean_rstd), ptr(b.gamma),
                                      (float*)ptr(row_sums), ptr(ws), ws.numel(), &parts, b.dt, stream()),
          "cw_ln_bwd_partials_open");
    return {row_sums, ws, parts};
}

// sums: this rank's; the row peers' are added. With column peers dgamma and dbeta come back reduce-scattered, as the given types.
std::tuple<Tensor, Tensor, Tensor> ln_bwd_dx_close(const Tensor& dy_in, const Tensor& x_in, const Tensor& mean_rstd, const Tensor& sums_in,
                                                   Peers row_peers, int64_t hidden, const Tensor& ws, int64_t parts, const OptTensor& gamma,
                                                   std::optional<at::ScalarType> param_type, Peers dgamma_peers, Peers dbeta_peers, int64_t world,
                                                   int64_t rank, at::ScalarType gamma_type, at::ScalarType beta_type) {
    const LnBackward b = ln_backward_inputs(dy_in, x_in, mean_rstd, sums_in, gamma);
    const bool rows_direct = direct(row_peers, sums_in);
    const Tensor sums = (rows_direct ? sums_in : add_peers(sums_in, row_peers)).reshape({b.R, 2}).to(at::kFloat).contiguous();
    const at::ScalarType pt = sum_type(param_type);
    Tensor dx = empty({b.R, b.C}, b.x), dgamma = empty({b.C}, b.x, pt), dbeta = empty({b.C}, b.x, pt);
    const Scatter sg{std::move(dgamma_peers), world, rank, gamma_type}, sb{std::move(dbeta_peers), world, rank, beta_type};
    const bool fused = sg.fused(dgamma) && sb.fused(dbeta) && sg.peers.size() == sb.peers.size() && gamma_type == beta_type;
    const int64_t count = fused ? sg.count(dgamma) : 0;
    OptTensor rg, rb;
    if (fused) {
        rg = empty({count}, b.x, sum_type(gamma_type));
        rb = empty({count}, b.x, gamma_type);
    }
    const auto tr = pointers(rows_direct ? row_peers : Peers{}), tg = pointers(fused ? sg.peers : Peers{}), tb = pointers(fused ? sb.peers : Peers{});
    check(lib.cw_ln_bwd_dx_close_peers(b.R, b.C, ptr(b.dy), ld(b.dy), ptr(b.x), ld(b.x), (const float*)ptr(mean_rstd), ptr(b.gamma),
                                       (const float*)ptr(sums), tr.data(), (int)tr.size(), hidden, ptr(dx), ld(dx), ptr(ws), parts, ptr(dgamma),
                                       ptr(dbeta), dtype_code(pt), tg.data(), tb.data(), (int)tg.size(), rank * count, count, ptr(rg), ptr(rb),
                                       fused ? dtype_code(gamma_type) : CW_F32, b.dt, stream()),
          "cw_ln_bwd_dx_close_peers");
    if (fused) {
        dgamma = *rg;
        dbeta = *rb;
    } else if (world > 1) {
        dgamma = sg.general(dgamma);
        dbeta = sb.general(dbeta);
    }
    return {dx.sizes() == x_in.sizes() ? dx : dx.reshape(x_in.sizes()), dgamma, dbeta};
}

// Mean vocabulary-parallel loss of [T, V] logits, T >= 1: -> (loss, [2, T] global maxima and sums). peers: as ops.vpce_finalize_peers.
std::tuple<Tensor, Tensor> vpce_mean(const Tensor& logits_in, const Tensor& targets_in, int64_t vocab_start, std::vector<Tensor> peers) {
    const Tensor logits = rows(logits_in);
    on_device(logits);
    on_device(targets_in);
    const int64_t T = logits.size(0), V = logits.size(1);
    const Tensor targets = targets_in.reshape({-1}).to(at::kLong).contiguous();
    TORCH_CHECK_VALUE(targets.numel() == T, "one target per logits row is required");
    Tensor own = empty({3, T}, logits, at::kFloat), mask = bytes(T, logits), total = empty({2, T}, logits, at::kFloat);
    Tensor loss = empty({}, logits, at::kFloat), ws = bytes(lib.cw_vpce_mean_workspace_bytes(T), logits);
    float *f = (float*)ptr(own), *g = (float*)ptr(total);
    uint8_t* m = (uint8_t*)ptr(mask);
    int64_t n = 0;
    TORCH_CHECK_VALUE(peers.empty() || peers.size() == 4, "the peers' max, sumexp, pred and mask must come from the same ranks");
    for (size_t i = 0; i < peers.size(); ++i) {
        on_device(peers[i]);
        peers[i] = peers[i].to(i < 3 ? at::kFloat : at::kByte).reshape({-1, T}).contiguous();
        n = peers[0].size(0);
        TORCH_CHECK_VALUE(peers[i].size(0) == n, "the peers' max, sumexp, pred and mask must come from the same ranks");
    }
    auto peer = [&](size_t i) { return peers.empty() ? nullptr : ptr(peers[i]); };
    check(lib.cw_vpce_fwd_local_mean(T, V, ptr(logits), ld(logits), (const int64_t*)ptr(targets), vocab_start, f, f + T, f + 2 * T, m, (int*)ptr(ws),
                                     dtype_code(logits.scalar_type()), stream()),
          "cw_vpce_fwd_local_mean");
    check(lib.cw_vpce_finalize_mean(T, (int)n, f, f + T, f + 2 * T, m, (const float*)peer(0), (const float*)peer(1), (const float*)peer(2),
                                    (const uint8_t*)peer(3), (float*)ptr(loss), g, g + T, ptr(ws), ws.numel(), stream()),
          "cw_vpce_finalize_mean");
    return {loss, total};
}

// Gradient of the logits, of their type, for the gradient `dloss` of vpce_mean's loss: contiguous, or with rows that begin at multiples
// of 16 bytes.
Tensor vpce_mean_bwd(const Tensor& logits_in, const Tensor& targets_in, int64_t vocab_start, const Tensor& total, const Tensor& dloss_in,
                     bool aligned) {
    const Tensor logits = rows(logits_in), targets = targets_in.reshape({-1}).to(at::kLong).contiguous(), dloss = dloss_in.to(at::kFloat);
    on_device(logits);
    on_device(dloss);
    const int64_t T = logits.size(0), V = logits.size(1);
    const int64_t unit = aligned ? 16 / logits.element_size() : 1;
    Tensor grad = empty({T, (V + unit - 1) / unit * unit}, logits).narrow(1, 0, V);
    const float* g = (const float*)ptr(total);
    const int dt = dtype_code(logits.scalar_type());
    check(lib.cw_vpce_bwd_mean(T, V, ptr(logits), ld(logits), (const int64_t*)ptr(targets), vocab_start, g, g + T, (const float*)ptr(dloss), ptr(grad),
                               ld(grad), dt, dt, stream()),
          "cw_vpce_bwd_mean");
    return grad;
}

}  // namespace cw_host

using namespace cw_host;

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.def("bind", &bind);
#define CW_HOST_DEF(name) m.def(#name, torch::wrap_pybind_function_no_gil(name))
    CW_HOST_DEF(gemm_ksteps);
    CW_HOST_DEF(colsum);
    CW_HOST_DEF(act_bwd_colsum);
    CW_HOST_DEF(colsum_scattered);
    CW_HOST_DEF(ln_partial_stats);
    CW_HOST_DEF(ln_partial_stats_gather);
    CW_HOST_DEF(ln_forward);
    CW_HOST_DEF(ln_backward_fused);
    CW_HOST_DEF(ln_bwd_partials_open);
    CW_HOST_DEF(ln_bwd_dx_close);
    CW_HOST_DEF(vpce_mean);
    CW_HOST_DEF(vpce_mean_bwd);
    def_nodes(m);
}
