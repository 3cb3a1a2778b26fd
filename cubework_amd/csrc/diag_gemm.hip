// Measurement aid (libcubework_diag.so, loaded by bench.py only): the block GEMM's launch for the headline shape, and a
// 256 x 256 tile kernel with one part taken out, so that the part's share of a launch - in time and, through the socket's
// energy counter, in joules - can be read as a difference against the same kernel whole:
//   part 0  the library's launch for this shape (gemm_wide.h; part 4 for K = 128 in one step, which that kernel does not take)
//   part 4  the kernel of 4 wavefronts and 32x32x16 matrix instructions that the library launched before, whole; of it
//   part 1  the k loop issues no operand loads: the four LDS stages are filled once and re-used
//   part 2  no epilogue: no bias / activation arithmetic, nothing stored
//   part 3  the k loop reads no fragments from LDS: the first tile's stay in the registers
// NN layout, bf16, bias + GeLU(tanh) epilogue, tile-aligned shapes with at least 128 tiles, 1 to 4 k-steps:
// the headline shape of the benchmark. Results of parts 1 to 3 are meaningless as numbers.
#include "gemm_wide.h"

namespace cw {
namespace {

using namespace gemm_tile;

constexpr int kMaxSteps = 4;
constexpr int TM = 4, TN = 4, NS = 4;  // MFMA tiles of a wavefront, LDS stages of 32 k

// 256 x 256 tiles on 4 wavefronts, from the loaders, LDS images and epilogue of gemm_tile.h: one barrier per k tile of 32 in the middle of
// its MFMAs, fragments read one k step ahead (a whole trip ahead would not leave registers for 4 x 4 accumulators), operands two to
// three k tiles ahead. Whole aligned tiles, one per block. What the library launched for such shapes before gemm_wide.h:
// 8192 x 2048 x 2048 62 us (53 there).
// ABL: 0 the whole kernel; 1 the k loop issues no operand loads (the stages are filled once and re-used); 2 no epilogue (nothing is
// stored); 3 the k loop reads no fragments from LDS (the first trip's stay in the registers).
template <int ABL>
__global__ __launch_bounds__(kThreads, 1) void ring_kernel(const TileArgs args) {
    constexpr int BM = 64 * TM, BN = 64 * TN;
    using LA = Loader<false, TM, 1>;
    using LB = Loader<true, TN, 1>;
    constexpr int kStage = LA::kBytes + LB::kBytes, kPer = TM + TN;  // bytes of a stage, load instructions per wavefront and k tile
    extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
    lds_char* lds_base = (lds_char*)lds;
    const uint32_t lds_addr0 = (uint32_t)(uintptr_t)lds_base;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int K = args.K, kps = K / kBK, KT = kps * args.n_steps;
    const int full_grid = (args.full + 7) & ~7;
    const int tile = (blockIdx.x & 7) * (full_grid >> 3) + (blockIdx.x >> 3);
    if (tile >= args.full) return;
    const int kt_beg = (int)(((int64_t)KT * (blockIdx.x & 7)) >> 3);  // the XCDs start at different k (gemm_wide.h)
    int tm, tn;
    tile_origin(tile, args.M / BM, args.N / BN, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;

    LA la;
    LB lb;
    la.init(lane, wave, args.lda, m0, args.M);
    lb.init(lane, wave, args.ldb, n0, args.N);
    Frags<false, TM, 1> fa;
    Frags<true, TN, 1> fb;
    fa.init(lane, wm * 32 * TM);
    fb.init(lane, wn * 32 * TN);
    const int64_t a_org = (int64_t)m0 * args.lda * 2, a_adv = 2 * kBK, b_org = (int64_t)n0 * 2, b_adv = args.ldb * (2 * kBK);
    f32x16_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
    const uint32_t bias_bits = reinterpret_cast<const uint16_t*>(args.bias)[n0 + tid];

    // the k tile whose loads are issued next; past the last one the instructions fetch nothing (is_rem 0)
    int is_left = KT, is_step = kt_beg / kps, is_stage = 0;
    int is_k = (kt_beg - is_step * kps) * kBK;
    const char* is_a = step_ptr(kTabA, is_step) + a_org + (is_k / kBK) * a_adv;
    const char* is_b = step_ptr(kTabB, is_step) + b_org + (is_k / kBK) * b_adv;
    int is_rem = K - is_k;
    auto issue_one = [&](auto op) {
        const uint32_t st = lds_addr0 + is_stage * kStage;
        if constexpr (op.value < TM) la.template issue<op.value>(is_a, 0, is_rem, st, wave);
        else lb.template issue<op.value - TM>(is_b, 0, is_rem, st + LA::kBytes, wave);
    };
    auto issue_advance = [&]() {
        is_stage = (is_stage + 1 == NS) ? 0 : is_stage + 1;
        --is_left;
        is_a += a_adv;
        is_b += b_adv;
        is_rem -= kBK;
        if (is_rem <= 0) {
            is_rem = 0;
            if (is_left > 0) {
                is_step = is_step + 1 == args.n_steps ? 0 : is_step + 1;
                is_a = step_ptr(kTabA, is_step) + a_org;
                is_b = step_ptr(kTabB, is_step) + b_org;
                is_rem = K;
            }
        }
        if (is_left <= 0) is_rem = 0;
    };
    auto publish = [&]() {
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    lds_char* rd = lds_base;  // stage read next
    int rd_stage = 0;
    auto read_advance = [&]() {
        rd_stage = (rd_stage + 1 == NS) ? 0 : rd_stage + 1;
        rd = lds_base + rd_stage * kStage;
    };
    // prologue: trips 0 .. NS-3 requested and the A part of trip NS-2
    for (int p = 0; p < (ABL == 1 ? NS : NS - 2); ++p) {
        static_for<kPer>([&](auto o) { issue_one(o); });
        issue_advance();
    }
    if constexpr (ABL == 1) {
        dma_wait<0>();
    } else {
        static_for<TM>([&](auto o) { issue_one(o); });
        dma_wait<kPer*(NS - 3) + TM>();
    }
    publish();
    bf16x8_t af[2][TM], bfr[2][TN];
    static_for<TM>([&](auto t) { af[0][t.value] = fa.template read<t.value, 0>(rd); });
    static_for<TN>([&](auto t) { bfr[0][t.value] = fb.template read<t.value, 0>(rd + LA::kBytes); });
    if constexpr (ABL == 3) {
        static_for<TM>([&](auto t) { af[1][t.value] = fa.template read<t.value, 1>(rd); });
        static_for<TN>([&](auto t) { bfr[1][t.value] = fb.template read<t.value, 1>(rd + LA::kBytes); });
    }
    constexpr int kMfma = TM * TN;
    for (int kt = 0; kt < KT; ++kt) {
        __builtin_amdgcn_sched_barrier(0);
        // k step 0; reads of k step 1; the B part of the trip whose A part went out in the previous one
        static_for<kMfma>([&](auto q) {
            constexpr int I = q.value / TN, J = q.value % TN, JS = (I & 1) ? TN - 1 - J : J;
            acc[I][JS] = gemm_bf16::mfma_32x32x16<bf16_t>(bfr[0][JS], af[0][I], acc[I][JS]);
            // fragment reads behind the first half of the MFMAs (their latency passes under the second), loads behind it
            if constexpr (q.value < TM + TN) {
                if constexpr (ABL != 3) {
                    if constexpr (q.value < TM) af[1][q.value] = fa.template read<q.value, 1>(rd);
                    else bfr[1][q.value - TM] = fb.template read<q.value - TM, 1>(rd + LA::kBytes);
                }
            } else if constexpr ((q.value - TM) % 2 == 0 && ABL != 1) {
                issue_one(std::integral_constant<int, TM + (q.value - TM - TN) / 2>{});
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        issue_advance();
        read_advance();
        // trip kt+1 complete for everybody, the stage of trip kt-1 free
        dma_wait<kPer*(NS - 3)>();
        publish();
        __builtin_amdgcn_sched_barrier(0);
        static_for<kMfma>([&](auto q) {
            constexpr int I = q.value / TN, J = q.value % TN, JS = (I & 1) ? TN - 1 - J : J;
            acc[I][JS] = gemm_bf16::mfma_32x32x16<bf16_t>(bfr[1][JS], af[1][I], acc[I][JS]);
            if constexpr (q.value < TM + TN) {
                if constexpr (ABL != 3) {
                    if constexpr (q.value < TM) af[0][q.value] = fa.template read<q.value, 0>(rd);
                    else bfr[0][q.value - TM] = fb.template read<q.value - TM, 0>(rd + LA::kBytes);
                }
            } else if constexpr ((q.value - TM) % 2 == 0 && ABL != 1) {
                issue_one(std::integral_constant<int, (q.value - TM - TN) / 2>{});
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    }
    dma_wait<0>();
    __syncthreads();
    if (ABL == 2 && args.n_steps >= 0) return;  // always taken, and keeps the products alive
    using Epi = Epilogue<TM, TN, CW_EPI_BIAS_GELU_TANH, bf16_t>;
    lds[2 * Epi::BUF + tid] = (uint16_t)bias_bits;
    __syncthreads();
    typename Epi::Bias bias;
    Epi::load_bias(lds + 2 * Epi::BUF, bias, wn, lane);
    int buf = 0;
    static_for<TM>([&](auto i) { Epi::slab_out(acc[i.value], i.value, args, true, lds, bias, buf, m0, n0, wm, wn, lane, tid); });
}

template <int ABL>
int launch_part(const TileArgs& args, hipStream_t s) {
    auto kern = ring_kernel<ABL>;
    constexpr size_t lds = kLdsBytes<TM, TN, 1, NS>;
    if (const int lrc = ensure_dynamic_lds((const void*)kern, (int)lds, "gemm ring (measurement library)"); lrc != CW_OK) return lrc;
    hipLaunchKernelGGL(kern, dim3((args.full + 7) / 8 * 8), dim3(kThreads), lds, s, args);
    return check_launch("ring_kernel");
}

}  // namespace
}  // namespace cw

using namespace cw;

extern "C" int cw_diag_gemm_part(int part, int64_t M, int64_t N, int64_t K, int n_steps, const void* const* A_steps,
                                 int64_t lda, const void* const* B_steps, int64_t ldb, const void* bias, void* C,
                                 int64_t ldc, void* stream) {
    if (part < 0 || part > 4) return fail(CW_ERR_INVALID, "cw_diag_gemm_part: part %d outside [0, 4]", part);
    if (n_steps < 1 || n_steps > kMaxSteps || A_steps == nullptr || B_steps == nullptr || bias == nullptr || C == nullptr)
        return fail(CW_ERR_INVALID, "cw_diag_gemm_part: 1 to %d k-steps, operands, bias and C are needed", kMaxSteps);
    if (M < 256 || N < 256 || K < 128 || (M % 256) != 0 || (N % 256) != 0 || (K % 64) != 0 || (M / 256) * (N / 256) < 128 ||
        M > (1 << 24) || N > (1 << 24) || K > (1 << 24))
        return fail(CW_ERR_UNSUPPORTED, "cw_diag_gemm_part: tile-aligned shapes with at least 128 tiles of 256 x 256 only");
    if (lda < K || ldb < N || ldc < N || (lda % 8) != 0 || (ldb % 8) != 0 || (ldc % 8) != 0)
        return fail(CW_ERR_ALIGNMENT, "cw_diag_gemm_part: leading dimensions must cover the rows and be multiples of 8");
    for (int i = 0; i < n_steps; ++i)
        if (A_steps[i] == nullptr || B_steps[i] == nullptr || !aligned16(A_steps[i]) || !aligned16(B_steps[i]))
            return fail(CW_ERR_ALIGNMENT, "cw_diag_gemm_part: step operands must be 16-byte aligned");
    if (!aligned16(C) || !aligned16(bias)) return fail(CW_ERR_ALIGNMENT, "cw_diag_gemm_part: C and bias must be 16-byte aligned");
    if (const int drc = require_gfx950("cw_diag_gemm_part"); drc != CW_OK) return drc;
    TileArgs args = {};
    for (int i = 0; i < n_steps; ++i) {
        args.A[i] = A_steps[i];
        args.B[i] = B_steps[i];
    }
    args.bias = bias;
    args.C = C;
    args.lda = lda;
    args.ldb = ldb;
    args.ldc = ldc;
    args.M = (int)M;
    args.N = (int)N;
    args.K = (int)K;
    args.n_steps = n_steps;
    args.vec_out = 1;
    args.full = (int)((M / 256) * (N / 256));
    args.slices = 1;
    args.rotate = 1;
    hipStream_t s = (hipStream_t)stream;
    if (part == 0 && !wide_takes(K, n_steps)) part = 4;
    switch (part) {
        case 0: return gemm_wide::launch_rows<false, true, 8, 4, 1, CW_EPI_BIAS_GELU_TANH, bf16_t>(args, s);
        case 1: return launch_part<1>(args, s);
        case 2: return launch_part<2>(args, s);
        case 3: return launch_part<3>(args, s);
        default: return launch_part<0>(args, s);
    }
}
