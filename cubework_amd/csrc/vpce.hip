// Vocab-parallel cross-entropy, one rank's vocabulary slice, for gfx950.
// forward: one online pass (running max + rescaled sum of exponentials) over a
// row per 256-thread block, 16-byte loads, wavefront-shuffle reductions, plus
// the bit-exact target mask / shifted index / gather. backward: recomputes the
// softmax from the logits and the global (max, sum) and writes the gradient;
// the logits are never modified.
// Both are bound by memory. 16-byte accesses serve rows of any alignment (an odd vocabulary puts every row at another
// offset): 1023 x 50257 bf16, forward 19 us where single elements took 75, backward 41 us for 44; aligned rows
// (8192 x 12568 bf16, 33 and 69 us, 6 TB/s) run as they did with loads that assumed their alignment.
#include <type_traits>

#include "cw_common.h"

namespace cw {

namespace {

constexpr int kCeBlock = 256;
constexpr int kCeUnroll = 3;     // 16-byte loads in flight per thread, forward
// Backward: one block of 16 wavefronts per row, every thread's share of the row requested at once. Measured on
// 8192 x 12568 bf16 -> fp32 (8-byte loads, 16-byte stores): 256 threads per row 118 us, 512: 116, 1024: 107.
constexpr int kCeBwdBlock = 1024;
constexpr float kNegInf = -__builtin_huge_valf();

// Running (max m, sum s of exp(x - m)) kept in the exp2 domain: m2 = m*log2(e).
struct OnlineLse {
    float m;   // running maximum of the logits seen (exact input value)
    float m2;  // m * log2(e), or 0 while m is -inf
    float s;   // sum of exp2(x*log2e - m2)
};

template <int V>
__device__ __forceinline__ float chunk_max(const float (&v)[V]) {
    float cm = v[0];
#pragma unroll
    for (int e = 1; e < V; ++e) cm = fmaxf(cm, v[e]);
    return cm;
}

// Adds U chunks with one rescale of the running sum.
template <int V, int U>
__device__ __forceinline__ void lse_add_chunks(OnlineLse& st, const float (&v)[U][V]) {
    float cm = chunk_max<V>(v[0]);
#pragma unroll
    for (int u = 1; u < U; ++u) cm = fmaxf(cm, chunk_max<V>(v[u]));
    const float m_new = fmaxf(st.m, cm);
    const float m2_new = (m_new == kNegInf) ? 0.0f : m_new * kLog2e;
    const float scale = (st.m == kNegInf) ? 0.0f : __builtin_amdgcn_exp2f(st.m2 - m2_new);
    float s = st.s * scale;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        float su = 0.0f;  // per-chunk partial sums keep the add chains short
#pragma unroll
        for (int e = 0; e < V; ++e) su += __builtin_amdgcn_exp2f(__builtin_fmaf(v[u][e], kLog2e, -m2_new));
        s += su;
    }
    st.m = m_new;
    st.m2 = m2_new;
    st.s = s;
}

template <int V>
__device__ __forceinline__ void lse_add_chunk(OnlineLse& st, const float (&v)[V]) {
    const float cm = chunk_max<V>(v);
    const float m_new = fmaxf(st.m, cm);
    const float m2_new = (m_new == kNegInf) ? 0.0f : m_new * kLog2e;
    // rescale the old sum; an empty state (m == -inf) has s == 0 and stays 0
    const float scale = (st.m == kNegInf) ? 0.0f : __builtin_amdgcn_exp2f(st.m2 - m2_new);
    float s = st.s * scale;
#pragma unroll
    for (int e = 0; e < V; ++e) s += __builtin_amdgcn_exp2f(__builtin_fmaf(v[e], kLog2e, -m2_new));
    st.m = m_new;
    st.m2 = m2_new;
    st.s = s;
}

__device__ __forceinline__ void lse_add_one(OnlineLse& st, float x) {
    const float v[1] = {x};
    lse_add_chunk<1>(st, v);
}

// Merge (m_b, s_b) into (m_a, s_a).
__device__ __forceinline__ void lse_merge(float& m_a, float& s_a, float m_b, float s_b) {
    const float m = fmaxf(m_a, m_b);
    const float fa = (m_a == kNegInf) ? 0.0f : __builtin_amdgcn_exp2f((m_a - m) * kLog2e);
    const float fb = (m_b == kNegInf) ? 0.0f : __builtin_amdgcn_exp2f((m_b - m) * kLog2e);
    s_a = s_a * fa + s_b * fb;
    m_a = m;
}

// 1 for a row of 16-bit elements that begins off a multiple of 4 bytes: where ODD, its vectors are taken from the second element on. 16-byte
// loads at odd elements take the load unit longer, at even ones they run as aligned ones do (1023 x 50257 bf16, where every other row
// is odd, forward 24.5 -> 18.9 us, as at 50258 columns; 8192 x 12567 forward 42.4 -> 34.7, backward 81 -> 72, at 12568 33 and 68).
// Long rows only, for it costs every wavefront some 20 instructions, of which a block of short rows does little else (us, without / with it:
// forward 8192 x 4097 20.1 / 19.5, 1853 x 4097 6.2 / 6.3, 1853 x 3073 5.9 / 6.0; backward 8192 x 8193 56.2 / 51.9, 437 x 8193 4.8 / 5.0, 8192 x
// 6145 43.9 / 43.9, 8192 x 1097 25.9 / 31.0).
template <bool ODD, typename T>
__device__ __forceinline__ int odd_row(const T* row) {
    return ODD ? (int)(reinterpret_cast<uintptr_t>(row) >> 1) & 1 : 0;
}
constexpr int64_t kOddForward = 4096, kOddBackward = 8192;  // columns
template <typename T>
bool odd_rows(const void* p, int64_t ld, int64_t rows) {
    return sizeof(T) == 2 && ((reinterpret_cast<uintptr_t>(p) >> 1 & 1) != 0 || (rows > 1 && ld % 2 != 0));
}

// MEAN: for the launch of the mean behind this one (MeanOut); a test of every block for it took 8192 rows of 301 from 11.1 to 11.6 us.
template <typename T, bool ODD, bool MEAN>
__global__ __launch_bounds__(kCeBlock) void vpce_fwd_kernel(int64_t T_rows, int64_t V_cols,
                                                            const T* __restrict__ logits, int64_t ld,
                                                            const int64_t* __restrict__ targets, int64_t vocab_start,
                                                            float* __restrict__ out_max, float* __restrict__ out_sumexp,
                                                            float* __restrict__ out_pred, uint8_t* __restrict__ out_mask,
                                                            int* __restrict__ arrived) {
    if (MEAN && blockIdx.x == 0 && threadIdx.x == 0) *arrived = 0;
    constexpr int V = elem<T>::kVec;
    __shared__ float red_m[kCeBlock / 64];
    __shared__ float red_s[kCeBlock / 64];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    for (int64_t row = blockIdx.x; row < T_rows; row += gridDim.x) {
        const T* row_begin = logits + row * ld;
        const int odd = odd_row<ODD>(row_begin);
        const T* xr = row_begin + odd;
        const int64_t cols = V_cols - odd;
        OnlineLse st{kNegInf, 0.0f, 0.0f};
        if (odd != 0 && tid == kCeBlock - 1) lse_add_one(st, load_elem(row_begin));
        const int64_t nvec = cols / V;
        int64_t i = tid;
        // kCeUnroll independent 16-byte streaming loads in flight per trip
        for (; i + (kCeUnroll - 1) * kCeBlock < nvec; i += kCeUnroll * kCeBlock) {
            raw16_t raw[kCeUnroll];
#pragma unroll
            for (int u = 0; u < kCeUnroll; ++u) raw[u] = load_raw_stream_any(xr + (i + u * kCeBlock) * V);
            float v[kCeUnroll][V];
#pragma unroll
            for (int u = 0; u < kCeUnroll; ++u) unpack_raw(raw[u], v[u], (const T*)nullptr);
            lse_add_chunks<V, kCeUnroll>(st, v);
        }
        for (; i < nvec; i += kCeBlock) {
            float v0[V];
            unpack_raw(load_raw_stream_any(xr + i * V), v0, (const T*)nullptr);
            lse_add_chunk<V>(st, v0);
        }
        for (int64_t c = nvec * V + tid; c < cols; c += kCeBlock) lse_add_one(st, load_elem(xr + c));
        // wavefront, then block
        float m = st.m, s = st.s;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const float mo = __shfl_xor(m, off, 64);
            const float so = __shfl_xor(s, off, 64);
            lse_merge(m, s, mo, so);
        }
        if (lane == 0) {
            red_m[wave] = m;
            red_s[wave] = s;
        }
        __syncthreads();
        if (tid == 0) {
            float gm = red_m[0], gs = red_s[0];
#pragma unroll
            for (int w = 1; w < kCeBlock / 64; ++w) lse_merge(gm, gs, red_m[w], red_s[w]);
            out_max[row] = gm;
            out_sumexp[row] = gs;
            // target bookkeeping: integer-exact
            const int64_t t = targets[row];
            const bool masked = (t < vocab_start) || (t >= vocab_start + V_cols);
            const int64_t idx = masked ? 0 : (t - vocab_start);
            out_mask[row] = masked ? 1 : 0;
            out_pred[row] = masked ? 0.0f : load_elem(row_begin + idx);
        }
        __syncthreads();
    }
}

// One slice's statistics, [T] each; for the peers' [n_peers, T].
struct CeStats {
    const float* max;
    const float* sumexp;
    const float* pred;
    const uint8_t* mask;
};
// The mean over the rows, finished by the launch that forms the losses: every block leaves its sum, and the one that arrives last
// (`arrived`, zeroed by the launch of the statistics) adds the blocks' sums in block order. Behind a launch of per-row losses the
// mean was one more (4.8 us at 8192 rows, where this takes the launch from 4.0 to 5.5 us), and its backward two autograd nodes and
// a launch that writes dloss / T for every row (2.9 us), which the gradient kernel now reads as one scalar.
struct MeanOut {
    float* mean;      // nullptr: the losses of the rows are wanted
    float* partials;  // one a block
    int* arrived;
};
constexpr int kMeanBlocks = 128;  // blocks at most; each release of a partial sum costs its XCD's L2 a write-back

// This rank's statistics and the peers' as they arrived, combined in that order: stacking them first took four launches
// (14 us of the GPU at 8192 rows of 4 ranks, and as much of the host) in front of this one (5 us): the loss, forward and
// backward, 173 -> 144 us.
__global__ __launch_bounds__(256) void vpce_finalize_kernel(int64_t T_rows, int n_peers, const CeStats own, const CeStats peers,
                                                            float* __restrict__ loss, float* __restrict__ gmax,
                                                            float* __restrict__ gsum, const MeanOut mean) {
    __shared__ float red[256 / 64];
    __shared__ int last;
    float total = 0.0f;
    for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < T_rows; t += (int64_t)gridDim.x * 256) {
        float m = own.max[t];
        for (int r = 0; r < n_peers; ++r) m = fmaxf(m, peers.max[(int64_t)r * T_rows + t]);
        float s = 0.0f, p = 0.0f;
        auto add = [&](const CeStats& st, int64_t i) {
            const float mr = st.max[i];
            const float f = (mr == kNegInf) ? 0.0f : expf(mr - m);
            s += st.sumexp[i] * f;
            if (st.mask[i] == 0) p += st.pred[i] - m;
        };
        add(own, t);
        for (int r = 0; r < n_peers; ++r) add(peers, (int64_t)r * T_rows + t);
        const float l = logf(s) - p;
        total += l;
        if (loss != nullptr) loss[t] = l;
        if (gmax != nullptr) gmax[t] = m;
        if (gsum != nullptr) gsum[t] = s;
    }
    if (mean.mean == nullptr) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    total = wave_sum(total);
    if (lane == 0) red[wave] = total;
    __syncthreads();
    if (threadIdx.x == 0) {
        float block = red[0];
        for (int w = 1; w < 256 / 64; ++w) block += red[w];
        __hip_atomic_store(mean.partials + blockIdx.x, block, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last = __hip_atomic_fetch_add(mean.arrived, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == (int)gridDim.x - 1;
    }
    __syncthreads();
    if (!last || wave != 0) return;
    float sum = 0.0f;
    for (int b = lane; b < (int)gridDim.x; b += 64) sum += __hip_atomic_load(mean.partials + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    sum = wave_sum(sum);
    if (lane == 0) *mean.mean = sum / (float)T_rows;
}

// The gradient is written once and not read again by this kernel: streaming stores.
template <int V>
__device__ __forceinline__ void store_grad(bf16_t* p, const float (&v)[V]) {
    static_assert(V == 8, "bf16 gradients are written 8 at a time");
    store_raw_stream_any(p, pack_raw(v, (const bf16_t*)nullptr));
}
template <int V>
__device__ __forceinline__ void store_grad(f16_t* p, const float (&v)[V]) {
    static_assert(V == 8, "fp16 gradients are written 8 at a time");
    store_raw_stream_any(p, pack_raw(v, (const f16_t*)nullptr));
}
template <int V>
__device__ __forceinline__ void store_grad(float* p, const float (&v)[V]) {
#pragma unroll
    for (int e = 0; e < V; e += 4) {
        const float q[4] = {v[e], v[e + 1], v[e + 2], v[e + 3]};
        store_raw_stream_any(p + e, pack_raw(q, (const float*)nullptr));
    }
}

// One 16-byte vector of the gradient row: softmax * scale, minus dl at the target column.
template <typename T, typename G, int V>
__device__ __forceinline__ void grad_vector(raw16_t raw, int64_t i, int64_t tcol, float m2, float scale, float dl,
                                            G* __restrict__ gr) {
    float v[V];
    unpack_raw(raw, v, (const T*)nullptr);
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(v[e], kLog2e, -m2)) * scale;
    const int64_t rel = tcol - i * V;
    if (rel >= 0 && rel < V) {
#pragma unroll
        for (int e = 0; e < V; ++e)
            if (e == rel) v[e] -= dl;
    }
    store_grad<V>(gr + i * V, v);
}

// fp32 gradient of 16-bit logits: four logits (8 bytes) in, four floats (16 bytes) out per lane, so that the
// stores of one instruction cover one contiguous 1 KB span. With 16-byte loads a lane would write 32
// bytes in two stores that each leave every other 16 bytes to the next instruction.
typedef uint32_t raw8_t __attribute__((ext_vector_type(2)));
typedef uint32_t raw8_any_t __attribute__((ext_vector_type(2), aligned(2)));
template <typename T>
__device__ __forceinline__ void grad_quad(raw8_t raw, int64_t i, int64_t tcol, float m2, float scale, float dl,
                                          float* __restrict__ gr) {
    float v[4] = {half_conv<T>::lo(raw.x), half_conv<T>::hi(raw.x), half_conv<T>::lo(raw.y), half_conv<T>::hi(raw.y)};
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(v[e], kLog2e, -m2)) * scale;
    const int64_t rel = tcol - i * 4;
    if (rel >= 0 && rel < 4) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (e == rel) v[e] -= dl;
    }
    store_raw_stream_any(gr + i * 4, pack_raw(v, (const float*)nullptr));
}

// The loss's gradient: one value a row, or one for all (stride 0), times scale; no pointer: scale alone.
struct DLoss {
    const float* p;
    int stride;
    float scale;
};

// Per-row scalars of the backward: fetched after the row's first loads have been issued.
struct CeRowScalars {
    float m2, dl, scale;
    int64_t tcol;
};
__device__ __forceinline__ CeRowScalars ce_row_scalars(int64_t row, int64_t V_cols, const int64_t* __restrict__ targets,
                                                       int64_t vocab_start, const float* __restrict__ gmax,
                                                       const float* __restrict__ gsum, const DLoss& dloss) {
    CeRowScalars r;
    r.m2 = gmax[row] * kLog2e;
    r.dl = (dloss.p != nullptr ? dloss.p[row * dloss.stride] : 1.0f) * dloss.scale;
    r.scale = r.dl / gsum[row];
    const int64_t t = targets[row];
    const bool masked = (t < vocab_start) || (t >= vocab_start + V_cols);
    r.tcol = masked ? -1 : (t - vocab_start);
    return r;
}

template <typename T, typename G, bool ODD>
__global__ __launch_bounds__(kCeBwdBlock) void vpce_bwd_kernel(int64_t T_rows, int64_t V_cols,
                                                               const T* __restrict__ logits, int64_t ld,
                                                               const int64_t* __restrict__ targets, int64_t vocab_start,
                                                               const float* __restrict__ gmax,
                                                               const float* __restrict__ gsum,
                                                               const DLoss dloss, G* __restrict__ grad, int64_t ld_grad) {
    constexpr int V = elem<T>::kVec;
    constexpr int B = kCeBwdBlock;
    const int tid = threadIdx.x;
    for (int64_t row = blockIdx.x; row < T_rows; row += gridDim.x) {
        const T* xr = logits + row * ld;
        G* gr = grad + row * ld_grad;
        if constexpr (sizeof(T) == 2 && std::is_same<G, float>::value) {
            // fp32 gradient of 16-bit logits: batches of U quads (8 bytes in, 16 out) per thread, all requested
            // before the first is worked on; a position past the end of the row re-reads the last quad (no
            // load under a branch) and stores nothing
            constexpr int U = 4;
            const int64_t nq = V_cols / 4;
            const uint16_t* xb = reinterpret_cast<const uint16_t*>(xr);
            float* gf = reinterpret_cast<float*>(gr);
            CeRowScalars rs;
            for (int64_t base = tid; base < nq; base += (int64_t)U * B) {
                raw8_t raw[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int64_t i = base + (int64_t)u * B;
                    raw[u] = __builtin_nontemporal_load(reinterpret_cast<const raw8_any_t*>(xb + (i < nq ? i : nq - 1) * 4));
                }
                if (base == tid) rs = ce_row_scalars(row, V_cols, targets, vocab_start, gmax, gsum, dloss);
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int64_t i = base + (int64_t)u * B;
                    if (i < nq) grad_quad<T>(raw[u], i, rs.tcol, rs.m2, rs.scale, rs.dl, gf);
                }
            }
            if (nq * 4 < V_cols) {
                rs = ce_row_scalars(row, V_cols, targets, vocab_start, gmax, gsum, dloss);
                for (int64_t c = nq * 4 + tid; c < V_cols; c += B) {
                    float y = __builtin_amdgcn_exp2f(__builtin_fmaf(load_elem(xr + c), kLog2e, -rs.m2)) * rs.scale;
                    if (c == rs.tcol) y -= rs.dl;
                    store_elem(gr + c, y);
                }
            }
        } else {
            // where logits and gradient are odd rows both, the vectors of both begin at the second element
            const int odd = odd_row<ODD>(xr) & odd_row<ODD>(gr);
            const int64_t nvec = (V_cols - odd) / V;
            CeRowScalars rs;
            if constexpr (sizeof(T) == 2) {
                // 16-bit in, 16-bit out: one vector per thread and trip. Sixteen wavefronts per row and two rows
                // per compute unit keep enough loads in flight; batching loads per thread measured slower here.
                rs = ce_row_scalars(row, V_cols, targets, vocab_start, gmax, gsum, dloss);
                for (int64_t i = tid; i < nvec; i += B)
                    grad_vector<T, G, V>(load_raw_stream_any(xr + odd + i * V), i, rs.tcol - odd, rs.m2, rs.scale, rs.dl, gr + odd);
            } else {
                constexpr int U = 4;  // 16-byte vectors per thread and batch
                for (int64_t base = tid; base < nvec; base += (int64_t)U * B) {
                    raw16_t raw[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const int64_t i = base + (int64_t)u * B;
                        raw[u] = load_raw_stream_any(xr + (i < nvec ? i : nvec - 1) * V);
                    }
                    if (base == tid) rs = ce_row_scalars(row, V_cols, targets, vocab_start, gmax, gsum, dloss);
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const int64_t i = base + (int64_t)u * B;
                        if (i < nvec) grad_vector<T, G, V>(raw[u], i, rs.tcol, rs.m2, rs.scale, rs.dl, gr);
                    }
                }
            }
            if (odd + nvec * V < V_cols || odd != 0) {
                rs = ce_row_scalars(row, V_cols, targets, vocab_start, gmax, gsum, dloss);
                // the columns behind the vectors, and the first one of an odd row
                for (int64_t c = odd + nvec * V + tid; c < V_cols + odd; c += B) {
                    const int64_t col = c < V_cols ? c : 0;
                    float y = __builtin_amdgcn_exp2f(__builtin_fmaf(load_elem(xr + col), kLog2e, -rs.m2)) * rs.scale;
                    if (col == rs.tcol) y -= rs.dl;
                    store_elem(gr + col, y);
                }
            }
        }
    }
}

int ce_grid(int64_t T_rows) {
    const int64_t cap = (int64_t)1 << 20;  // one block per row: finished blocks are replaced one by one
    return (int)(T_rows < cap ? T_rows : cap);
}

template <typename T, typename G>
int bwd_impl(int64_t T_rows, int64_t V_cols, const void* logits, int64_t ld, const int64_t* targets,
             int64_t vocab_start, const float* gmax, const float* gsum, const DLoss& dloss, void* grad, int64_t ld_grad,
             hipStream_t s) {
    auto launch = [&](auto odd) {
        hipLaunchKernelGGL((vpce_bwd_kernel<T, G, decltype(odd)::value>), dim3(ce_grid(T_rows)), dim3(kCeBwdBlock), 0, s, T_rows, V_cols,
                           (const T*)logits, ld, targets, vocab_start, gmax, gsum, dloss, (G*)grad, ld_grad);
        return check_launch("vpce_bwd_kernel");
    };
    if constexpr (sizeof(G) == 2)
        if (V_cols >= kOddBackward && odd_rows<T>(logits, ld, T_rows) && odd_rows<G>(grad, ld_grad, T_rows)) return launch(std::true_type{});
    return launch(std::false_type{});
}

}  // namespace
}  // namespace cw

using namespace cw;

extern "C" int cw_vpce_fwd_local(int64_t T, int64_t V, const void* logits, int64_t ld, const int64_t* targets,
                                 int64_t vocab_start, float* out_max, float* out_sumexp, float* out_pred,
                                 uint8_t* out_mask, int io_dtype, void* stream) {
    return cw_vpce_fwd_local_mean(T, V, logits, ld, targets, vocab_start, out_max, out_sumexp, out_pred, out_mask, nullptr, io_dtype, stream);
}

extern "C" int cw_vpce_fwd_local_mean(int64_t T, int64_t V, const void* logits, int64_t ld, const int64_t* targets, int64_t vocab_start,
                                      float* out_max, float* out_sumexp, float* out_pred, uint8_t* out_mask, int* arrived, int io_dtype,
                                      void* stream) {
    if (T < 0 || V <= 0) return fail(CW_ERR_INVALID, "cw_vpce_fwd_local: bad shape T=%lld V=%lld", (long long)T, (long long)V);
    if (io_dtype != CW_BF16 && io_dtype != CW_F32 && io_dtype != CW_F16)
        return fail(CW_ERR_INVALID, "cw_vpce_fwd_local: bad io_dtype %d", io_dtype);
    if (vocab_start < 0) return fail(CW_ERR_INVALID, "cw_vpce_fwd_local: negative vocab_start");
    if (T == 0) return CW_OK;
    if (logits == nullptr || targets == nullptr || out_max == nullptr || out_sumexp == nullptr ||
        out_pred == nullptr || out_mask == nullptr || ld < V)
        return fail(CW_ERR_INVALID, "cw_vpce_fwd_local: null pointer or ld < V");
    if (const int drc = require_gfx950("cw_vpce_fwd_local"); drc != CW_OK) return drc;
    hipStream_t s = (hipStream_t)stream;
    return with_elem_type(io_dtype, [&](auto* tag) {
        using E = std::remove_pointer_t<decltype(tag)>;
        auto launch = [&](auto odd, auto mean) {
            hipLaunchKernelGGL((vpce_fwd_kernel<E, decltype(odd)::value, decltype(mean)::value>), dim3(ce_grid(T)), dim3(kCeBlock), 0, s, T, V,
                               (const E*)logits, ld, targets, vocab_start, out_max, out_sumexp, out_pred, out_mask, arrived);
            return check_launch("vpce_fwd_kernel");
        };
        auto any = [&](auto odd) { return arrived != nullptr ? launch(odd, std::true_type{}) : launch(odd, std::false_type{}); };
        if constexpr (sizeof(E) == 2)
            if (V >= kOddForward && odd_rows<E>(logits, ld, T)) return any(std::true_type{});
        return any(std::false_type{});
    });
}

extern "C" int cw_vpce_finalize(int64_t T, int n_ranks, const float* max_all, const float* sumexp_all,
                                const float* pred_all, const uint8_t* mask_all, float* loss, float* gmax,
                                float* gsum, void* stream) {
    if (T < 0 || n_ranks < 1) return fail(CW_ERR_INVALID, "cw_vpce_finalize: bad T=%lld or n_ranks=%d", (long long)T, n_ranks);
    if (T == 0) return CW_OK;
    if (max_all == nullptr || sumexp_all == nullptr || pred_all == nullptr || mask_all == nullptr || loss == nullptr)
        return fail(CW_ERR_INVALID, "cw_vpce_finalize: null pointer");
    return cw_vpce_finalize_peers(T, n_ranks - 1, max_all, sumexp_all, pred_all, mask_all, max_all + T, sumexp_all + T,
                                  pred_all + T, mask_all + T, loss, gmax, gsum, stream);
}

extern "C" int cw_vpce_finalize_peers(int64_t T, int n_peers, const float* max, const float* sumexp, const float* pred,
                                      const uint8_t* mask, const float* max_peers, const float* sumexp_peers,
                                      const float* pred_peers, const uint8_t* mask_peers, float* loss, float* gmax,
                                      float* gsum, void* stream) {
    if (T < 0 || n_peers < 0) return fail(CW_ERR_INVALID, "cw_vpce_finalize_peers: bad T=%lld or n_peers=%d", (long long)T, n_peers);
    if (T == 0) return CW_OK;
    if (max == nullptr || sumexp == nullptr || pred == nullptr || mask == nullptr || loss == nullptr ||
        (n_peers > 0 && (max_peers == nullptr || sumexp_peers == nullptr || pred_peers == nullptr || mask_peers == nullptr)))
        return fail(CW_ERR_INVALID, "cw_vpce_finalize_peers: null pointer");
    if (const int drc = require_gfx950("cw_vpce_finalize_peers"); drc != CW_OK) return drc;
    hipLaunchKernelGGL(vpce_finalize_kernel, dim3((unsigned)((T + 255) / 256)), dim3(256), 0, (hipStream_t)stream, T, n_peers,
                       (CeStats{max, sumexp, pred, mask}), (CeStats{max_peers, sumexp_peers, pred_peers, mask_peers}), loss, gmax, gsum, MeanOut{});
    return check_launch("vpce_finalize_kernel");
}

extern "C" int64_t cw_vpce_mean_workspace_bytes(int64_t T) {
    const int64_t blocks = (T + 255) / 256;
    return T <= 0 ? 0 : (1 + (blocks < kMeanBlocks ? blocks : kMeanBlocks)) * (int64_t)sizeof(float);
}

extern "C" int cw_vpce_finalize_mean(int64_t T, int n_peers, const float* max, const float* sumexp, const float* pred, const uint8_t* mask,
                                     const float* max_peers, const float* sumexp_peers, const float* pred_peers,
                                     const uint8_t* mask_peers, float* loss_mean, float* gmax, float* gsum, void* workspace,
                                     int64_t workspace_bytes, void* stream) {
    if (T <= 0 || n_peers < 0) return fail(CW_ERR_INVALID, "cw_vpce_finalize_mean: bad T=%lld or n_peers=%d", (long long)T, n_peers);
    if (max == nullptr || sumexp == nullptr || pred == nullptr || mask == nullptr || loss_mean == nullptr || workspace == nullptr ||
        (n_peers > 0 && (max_peers == nullptr || sumexp_peers == nullptr || pred_peers == nullptr || mask_peers == nullptr)))
        return fail(CW_ERR_INVALID, "cw_vpce_finalize_mean: null pointer");
    const int64_t need = cw_vpce_mean_workspace_bytes(T);
    if (workspace_bytes < need || (reinterpret_cast<uintptr_t>(workspace) & 3u) != 0)
        return fail(CW_ERR_INVALID, "cw_vpce_finalize_mean: workspace too small (%lld bytes) or not 4-byte aligned", (long long)workspace_bytes);
    if (const int drc = require_gfx950("cw_vpce_finalize_mean"); drc != CW_OK) return drc;
    hipLaunchKernelGGL(vpce_finalize_kernel, dim3((unsigned)(need / (int64_t)sizeof(float) - 1)), dim3(256), 0, (hipStream_t)stream, T, n_peers,
                       (CeStats{max, sumexp, pred, mask}), (CeStats{max_peers, sumexp_peers, pred_peers, mask_peers}), nullptr, gmax, gsum,
                       (MeanOut{loss_mean, (float*)workspace + 1, (int*)workspace}));
    return check_launch("vpce_finalize_kernel (mean)");
}

static int vpce_bwd(int64_t T, int64_t V, const void* logits, int64_t ld, const int64_t* targets, int64_t vocab_start,
                    const float* gmax, const float* gsum, const DLoss& dloss, void* grad, int64_t ld_grad, int io_dtype,
                    int grad_dtype, void* stream);

extern "C" int cw_vpce_bwd(int64_t T, int64_t V, const void* logits, int64_t ld, const int64_t* targets,
                           int64_t vocab_start, const float* gmax, const float* gsum, const float* dloss_rows,
                           float dloss_scale, void* grad, int64_t ld_grad, int io_dtype, int grad_dtype,
                           void* stream) {
    return vpce_bwd(T, V, logits, ld, targets, vocab_start, gmax, gsum, DLoss{dloss_rows, 1, dloss_scale}, grad, ld_grad, io_dtype,
                    grad_dtype, stream);
}

extern "C" int cw_vpce_bwd_mean(int64_t T, int64_t V, const void* logits, int64_t ld, const int64_t* targets, int64_t vocab_start,
                                const float* gmax, const float* gsum, const float* dloss, void* grad, int64_t ld_grad, int io_dtype,
                                int grad_dtype, void* stream) {
    if (dloss == nullptr) return fail(CW_ERR_INVALID, "cw_vpce_bwd_mean: null pointer");
    return vpce_bwd(T, V, logits, ld, targets, vocab_start, gmax, gsum, DLoss{dloss, 0, 1.0f / (float)T}, grad, ld_grad, io_dtype,
                    grad_dtype, stream);
}

static int vpce_bwd(int64_t T, int64_t V, const void* logits, int64_t ld, const int64_t* targets, int64_t vocab_start,
                    const float* gmax, const float* gsum, const DLoss& dloss, void* grad, int64_t ld_grad, int io_dtype,
                    int grad_dtype, void* stream) {
    if (T < 0 || V <= 0) return fail(CW_ERR_INVALID, "cw_vpce_bwd: bad shape T=%lld V=%lld", (long long)T, (long long)V);
    if (io_dtype != CW_BF16 && io_dtype != CW_F32 && io_dtype != CW_F16)
        return fail(CW_ERR_INVALID, "cw_vpce_bwd: bad io_dtype %d", io_dtype);
    if (grad_dtype != CW_BF16 && grad_dtype != CW_F32 && grad_dtype != CW_F16)
        return fail(CW_ERR_INVALID, "cw_vpce_bwd: bad grad_dtype %d", grad_dtype);
    if (grad_dtype != CW_F32 && grad_dtype != io_dtype)
        return fail(CW_ERR_UNSUPPORTED, "cw_vpce_bwd: the gradient is fp32 or of the logits' type");
    if (T == 0) return CW_OK;
    if (logits == nullptr || targets == nullptr || gmax == nullptr || gsum == nullptr || grad == nullptr || ld < V ||
        ld_grad < V)
        return fail(CW_ERR_INVALID, "cw_vpce_bwd: null pointer or leading dimension < V");
    if (const int drc = require_gfx950("cw_vpce_bwd"); drc != CW_OK) return drc;
    hipStream_t s = (hipStream_t)stream;
    if (io_dtype == CW_F16 && grad_dtype == CW_F16)
        return bwd_impl<f16_t, f16_t>(T, V, logits, ld, targets, vocab_start, gmax, gsum, dloss, grad, ld_grad, s);
    if (io_dtype == CW_F16)
        return bwd_impl<f16_t, float>(T, V, logits, ld, targets, vocab_start, gmax, gsum, dloss, grad, ld_grad, s);
    if (io_dtype == CW_BF16 && grad_dtype == CW_BF16)
        return bwd_impl<bf16_t, bf16_t>(T, V, logits, ld, targets, vocab_start, gmax, gsum, dloss, grad, ld_grad, s);
    if (io_dtype == CW_BF16)
        return bwd_impl<bf16_t, float>(T, V, logits, ld, targets, vocab_start, gmax, gsum, dloss, grad, ld_grad, s);
    return bwd_impl<float, float>(T, V, logits, ld, targets, vocab_start, gmax, gsum, dloss, grad, ld_grad, s);
}
