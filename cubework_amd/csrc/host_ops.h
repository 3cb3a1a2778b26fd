// The operators' host side, shared by the calls (host_ops.cpp) and the autograd nodes (host_nodes.cpp).
#pragma once
#include <torch/extension.h>

#include "cubework_hip.h"

namespace cw_host {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

#define CW_HOST_ENTRIES(X)                                                                                             \
    X(cw_gemm_scratch_bytes) X(cw_gemm_ksteps_ws) X(cw_colsum_workspace_bytes) X(cw_colsum) X(cw_act_bwd_colsum)       \
    X(cw_colsum_peers) X(cw_act_bwd_colsum_peers) X(cw_ln_partial_stats) X(cw_ln_partial_stats_gather)                 \
    X(cw_ln_normalize_peers) X(cw_ln_forward_fused) X(cw_ln_backward_fused) X(cw_ln_bwd_partials_open)                 \
    X(cw_ln_bwd_dx_close_peers) X(cw_vpce_fwd_local_mean) X(cw_vpce_mean_workspace_bytes) X(cw_vpce_finalize_mean)     \
    X(cw_vpce_bwd_mean) X(cw_attn_fwd) X(cw_attn_narrow_fwd) X(cw_attn_bwd) X(cw_attn_narrow_bwd)                      \
    X(cw_attn_bwd_workspace_bytes) X(cw_embed_fwd) X(cw_embed_bwd_ids_supported) X(cw_embed_bwd_ids)                   \
    X(cw_embed_sort_workspace_bytes) X(cw_embed_sort_ids) X(cw_embed_bwd) X(cw_cast_many)
struct Entries {
#define X(name) decltype(&::name) name = nullptr;
    CW_HOST_ENTRIES(X)
#undef X
};
extern Entries lib;

// Raises CubeworkHipError for a status of the library.
void check(int status, const char* what);
int dtype_code(at::ScalarType t);
void on_device(const Tensor& t);
// View as [rows, cols] with unit column stride (copy only if unavoidable), and its leading dimension.
Tensor rows(const Tensor& t);
int64_t ld(const Tensor& t);
void* stream();
inline void* ptr(const Tensor& t) { return t.data_ptr(); }
inline bool aligned16(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }
inline Tensor empty(at::IntArrayRef shape, const Tensor& like, at::ScalarType t) { return at::empty(shape, like.options().dtype(t)); }
inline Tensor empty(at::IntArrayRef shape, const Tensor& like) { return at::empty(shape, like.options()); }
inline Tensor bytes(int64_t n, const Tensor& like) { return empty({n}, like, at::kByte); }

std::tuple<Tensor, OptTensor> gemm_ksteps(int layout, std::vector<Tensor> A, std::vector<Tensor> B, const OptTensor& bias_in, int epilogue,
                                          std::vector<Tensor> addends, bool want_preact, const OptTensor& out_in);
// Each of the tensors (undefined ones stay so) as `type`: those that are contiguous between fp32 and a 16-bit type in one launch.
void cast_together(std::initializer_list<Tensor*> ts, at::ScalarType type);
Tensor colsum(const Tensor& dy_in, std::optional<at::ScalarType> out_type);
std::tuple<Tensor, OptTensor> act_bwd_colsum(int activation, const Tensor& dy_in, const Tensor& pre_in, bool want_dbias,
                                             std::optional<at::ScalarType> out_type);
std::tuple<Tensor, OptTensor> ln_forward(const Tensor& x_in, const OptTensor& stats_in, std::vector<Tensor> peers, int64_t hidden, double eps,
                                         const OptTensor& gamma_in, const OptTensor& beta_in, int mode, bool save_mean_rstd);
std::tuple<Tensor, OptTensor, OptTensor> ln_backward_fused(const Tensor& dy_in, const Tensor& x_in, const Tensor& mean_rstd,
                                                           const OptTensor& gamma, bool want_param_grads,
                                                           std::optional<at::ScalarType> param_type, const OptTensor& addend);
std::tuple<Tensor, Tensor> vpce_mean(const Tensor& logits_in, const Tensor& targets_in, int64_t vocab_start, std::vector<Tensor> peers);
Tensor vpce_mean_bwd(const Tensor& logits_in, const Tensor& targets_in, int64_t vocab_start, const Tensor& total, const Tensor& dloss_in,
                     bool aligned);

void def_nodes(py::module_& m);

}  // namespace cw_host
