// 16-bit block GEMM for any shape (gfx950): ragged M, N and K, outputs with few tiles, partial last rounds.
//
//   - BM x BN tile of C per 256-thread block (4 wavefronts, 2x2; a wavefront owns TM x TN MFMA tiles of 32x32, BM = 64 TM,
//     BN = 64 TN); trips of KB k tiles of 32 in a ring of NS LDS stages filled by the load unit, one barrier per trip, fragments read a
//     whole trip ahead: a wavefront arrives at the barrier with the next products' operands in registers, and neither the barrier
//     nor the LDS latency is exposed.
//   - Operands are fetched with buffer_load_dwordx4 ... lds. The lane's byte offset goes through the buffer's range
//     check, and a lane whose 16-byte chunk lies outside the operand (row >= M or N, k >= K) is handed an offset
//     beyond the range: the load unit writes zeros for it. So edges cost no branch, no second kernel and no memory
//     traffic, and 128 x 128 tiles serve an M of 1 as well. A k-contiguous operand whose K is not a multiple of 8
//     has one chunk per row that straddles K: its tail is zeroed in LDS before the tile is published.
//   - The launch's work is `full` whole tiles followed by the remaining tiles cut into `slices` k ranges each
//     (partial sums through scratch in accumulator order, finished by tile_reduce_kernel): the last, partly empty
//     round of tiles, or a problem with few tiles and a long reduction, is spread over the whole chip.
//
// LDS images per stage: k-contiguous operand [BM rows][32 k], chunk c of row r at c ^ ((r >> 2) & 3), or, where a trip is 64 k,
// [BM rows][64 k], chunk c of row r at c ^ ((r >> 1) & 7); k-slow operand [32 k][BM rows], chunk c of k row k at c ^ ((k & 3) << 2),
// one image per 32 k. All read conflict free.
// Rows of 64 k are whole 128-byte lines: a load instruction of 8 of them takes the load unit 17 cycles, one of 16 pieces of 64 bytes
// (two images of 32 k a trip, as before) 35, and that bounded the small tiles: 16 such instructions a trip of a 64 x 64 NT tile.
#pragma once
#include <cstddef>

#include "gemm_bf16_kernel.h"

namespace cw {

// Argument block of the kernel and of its reduction. The pointer tables are read from the kernel argument segment with
// a uniform index where one is needed (step_ptr): held in scalar registers they would be spilled for the whole k loop.
struct TileArgs {
    const void* A[CW_MAX_KSTEPS];
    const void* B[CW_MAX_KSTEPS];
    const void* addend[CW_MAX_ADDENDS];
    const void* bias;
    void* C;
    void* preact;
    int64_t lda, ldb, ldc, ldp, ldadd;
    int M, N, K, n_steps, n_addends;
    int vec_out;    // C and preact allow 16-byte accesses at every tile column
    int full;       // tiles computed whole
    int slices;     // k slices of each of the other tiles
    int rotate;     // the XCDs start a whole tile's reduction at different k (gemm_wide.h)
    float* partial; // slices x (tiles - full) tiles of BM x BN fp32 partial sums
};

namespace gemm_tile {

using gemm_bf16::bf16x8_t;
using gemm_bf16::f32x16_t;
using gemm_bf16::static_for;
using gemm_bf16::u32x2_t;
using gemm_bf16::u32x4_t;
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef short s16x8_t __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) char lds_char;
typedef __attribute__((address_space(3))) uint16_t lds_u16;

constexpr int kBK = 32;
constexpr int kThreads = 256;
constexpr uint32_t kRange = kDmaRange;  // bytes a lane offset may reach; an offset of kRange itself is out of range

constexpr int kTabA = 0, kTabB = CW_MAX_KSTEPS, kTabAddend = 2 * CW_MAX_KSTEPS;  // entries before each table
static_assert(offsetof(TileArgs, A) == 0 && offsetof(TileArgs, B) == 8 * kTabB && offsetof(TileArgs, addend) == 8 * kTabAddend,
              "pointer tables lead the argument block, which is the kernels' only argument");
__device__ __forceinline__ const char* step_ptr(int table, int idx) {
    const auto* tab = (const __attribute__((address_space(4))) uint64_t*)__builtin_amdgcn_kernarg_segment_ptr();
    return reinterpret_cast<const char*>(tab[table + __builtin_amdgcn_readfirstlane(idx)]);
}

// 64-byte units by which row k of a k-slow image is rotated (xor): the four k rows that a transposing read touches
// together fall into different banks. Rows of 64 elements (W = 1) are 128 bytes, so two of them share the 64 banks.
template <int W>
__device__ __forceinline__ int kslow_swizzle(int k) {
    return W == 1 ? (k >> 1) & 1 : k & 3;
}

// Loader of one operand: W MFMA tiles per wavefront, 64 W rows per block, W load instructions per wavefront and 32 k of a trip of KB.
template <bool TRANS, int W, int KB>
struct Loader {
    static constexpr int kRows = 64 * W;
    static constexpr int kImage = kRows * kBK * 2, kBytes = KB * kImage;  // of 32 k, of a trip
    static constexpr int kKPer = 1024 / (kRows * 2);  // TRANS: k rows per instruction
    static constexpr bool kLines = !TRANS && KB == 2;  // rows of 64 k
    static constexpr int kOffsets = kLines ? 2 * W : W;
    static_assert(KB == 1 || KB == 2, "");
    uint32_t voff[kOffsets];
    int klane;  // !TRANS: first k of the lane's chunk (of instruction 0); TRANS: the lane's k row in instruction 0
    // row0: first operand row of the block; rmax: rows of the operand
    __device__ __forceinline__ void init(int lane, int wave, int64_t ld, int row0, int rmax) {
        if constexpr (kLines) {
            const int r = wave * 16 * W + (lane >> 3), c = (lane & 7) ^ (lane >> 4);
            klane = c * 8;
#pragma unroll
            for (int i = 0; i < kOffsets; ++i)
                voff[i] = row0 + r + 8 * i < rmax ? (uint32_t)(((int64_t)(r + 8 * i) * ld + (c ^ (i & 1) * 4) * 8) * 2) : kRange;
        } else if constexpr (!TRANS) {
            const int r = wave * 16 * W + (lane >> 2), c = (lane & 3) ^ (lane >> 4);
            klane = c * 8;
#pragma unroll
            for (int i = 0; i < W; ++i)
                voff[i] = row0 + r + 16 * i < rmax ? (uint32_t)(((int64_t)(r + 16 * i) * ld + c * 8) * 2) : kRange;
        } else {
            constexpr int LPR = 64 / kKPer;  // lanes per k row
            klane = wave * 8 + lane / LPR;
#pragma unroll
            for (int i = 0; i < W; ++i) {
                const int k = klane + i * kKPer;
                const int c = (lane % LPR) ^ (kslow_swizzle<W>(k) << 2);
                voff[i] = row0 + c * 8 < rmax ? (uint32_t)(((int64_t)k * ld + c * 8) * 2) : kRange;
            }
        }
    }
    // base: the block's first row at the trip's first k, adv: bytes from there to the next 32 k; k_rem: k values left from base on
    // (<= 0: nothing is fetched)
    template <int I>
    __device__ __forceinline__ void issue(const char* base, int64_t adv, int k_rem, uint32_t lds_oper, int wave) const {
        constexpr int H = I / W, O = I % W;  // the 32 k of the trip and the instruction there, of images of 32 k
        if constexpr (kLines) dma16_buffer(base, (klane ^ (I & 1) * 32) < k_rem ? voff[I] : kRange, lds_oper + (wave * 2 * W + I) * 1024);
        else if constexpr (!TRANS) dma16_buffer(base, klane < k_rem ? voff[I] : kRange, lds_oper + (wave * 16 * W + I * 16) * 64);
        else
            dma16_buffer(base + H * adv, klane + O * kKPer < k_rem - H * kBK ? voff[O] : kRange,
                         lds_oper + H * kImage + (wave * 8 + O * kKPer) * (kRows * 2));
    }
    // !TRANS: zero what lies past k_rem in the chunks that straddle it, in the rows this wavefront loaded (W * 16)
    __device__ __forceinline__ void fix_tail(lds_char* oper, int k_rem, int lane, int wave) const {
        if constexpr (!TRANS) {
            const int c = k_rem >> 3;
            if (lane < 16 * W) {
                const int r = wave * 16 * W + lane;
                lds_u16* p = (lds_u16*)(oper + (kLines ? r * 128 + ((c ^ ((r >> 1) & 7)) << 4) : r * 64 + ((c ^ ((r >> 2) & 3)) << 4)));
                for (int e = k_rem & 7; e < 8; ++e) p[e] = 0;
            }
        }
    }
};

template <bool TRANS, int W, int KB>
struct Frags {
    static constexpr int kRows = 64 * W;
    static constexpr bool kLines = Loader<TRANS, W, KB>::kLines;
    uint32_t off[TRANS ? W : 2 * KB];
    __device__ __forceinline__ void init(int lane, int wrow) {
        if constexpr (!TRANS) {
            const int r = lane & 31, g = lane >> 5, swz = kLines ? (r >> 1) & 7 : (r >> 2) & 3;
#pragma unroll
            for (int ks = 0; ks < 2 * KB; ++ks) off[ks] = (uint32_t)((wrow + r) * (kLines ? 128 : 64) + (((2 * ks + g) ^ swz) << 4));
        } else {
            const int i = lane & 15, grp = lane >> 4, g = grp >> 1, kk = (i >> 2) & 3;
            const int lane_const = (8 * g + (i >> 2)) * (kRows * 2) + ((2 * (grp & 1) + ((i & 3) >> 1)) << 4) + 8 * (i & 1);
#pragma unroll
            for (int t = 0; t < W; ++t) off[t] = (uint32_t)(lane_const + 64 * (((wrow >> 5) + t) ^ kslow_swizzle<W>(kk)));
        }
    }
    template <int T, int KS>
    __device__ __forceinline__ bf16x8_t read(lds_char* oper) const {
        if constexpr (!TRANS) {
            return *(__attribute__((address_space(3))) const bf16x8_t*)(oper + off[KS] + T * 32 * (kLines ? 128 : 64));
        } else {
            lds_char* p = oper + off[T] + KS * 16 * (kRows * 2);  // the next 32 k's image follows: 32 rows further
            const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)p);
            const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(p + 4 * (kRows * 2)));
            const s16x8_t v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            return __builtin_bit_cast(bf16x8_t, v);
        }
    }
};

// Tile `tile` of the tiles_m x tiles_n grid, in groups of 8 tile rows (consecutive ids share operand panels).
__device__ __forceinline__ void tile_origin(int tile, int tiles_m, int tiles_n, int& tm, int& tn) {
    constexpr int GROUP_M = 8;
    const int group = tile / (GROUP_M * tiles_n);
    const int first_m = group * GROUP_M;
    const int gsz = (tiles_m - first_m) < GROUP_M ? (tiles_m - first_m) : GROUP_M;
    const int in_group = tile - group * GROUP_M * tiles_n;
    tm = first_m + in_group % gsz;
    tn = in_group / gsz;
}

// gelu(x) = x/2 erfc(-x / sqrt 2) without branches (erff has some, and see Epilogue::stage). erfc(z) = t exp(-z^2 + q(t)),
// t = 1 / (1 + z/2), z >= 0, is the form that "Numerical Recipes" gives for erfc; q here is a least-squares fit of degree 9 of
// its own, in Chebyshev points of log(erfc(z) e^(z^2) / t). In float32 against float64: relative error 5e-7 for |x| < 1
// (x/2 (1 + erf) has 2e-7 there), 1.3e-6 for -3 < x < -1, 2e-6 for -4 < x < -3 and, growing with the exponent's rounding,
// 3e-6, 7e-6 and 2e-5 down to x = -5.5, -8 and -13 (x/2 (1 + erf) cancels there: 5e-4 at -4, all digits below -5.5). The
// result is rounded to 2^-9 or 2^-12. The register-staged kernel and the backward use erff.
__device__ __forceinline__ float gelu_erf_smooth(float x) {
    const float z = fabsf(x) * 0.7071067811865476f;
    const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(0.5f, z, 1.0f));
    float q = 0.17841362f;
    q = __builtin_fmaf(q, t, -0.858497037f);
    q = __builtin_fmaf(q, t, 1.56252653f);
    q = __builtin_fmaf(q, t, -1.2180208f);
    q = __builtin_fmaf(q, t, 0.334326584f);
    q = __builtin_fmaf(q, t, -0.208975052f);
    q = __builtin_fmaf(q, t, 0.102332011f);
    q = __builtin_fmaf(q, t, 0.373333673f);
    q = __builtin_fmaf(q, t, 1.00007393f);
    q = __builtin_fmaf(q, t, -1.26551338f);
    const float c = t * __builtin_amdgcn_exp2f(__builtin_fmaf(-z, z, q) * kLog2e);
    const float cdf2 = x > 0.0f ? 2.0f - c : c;
    return 0.5f * x * cdf2;
}
template <int EPI>
__device__ __forceinline__ float tile_act(float x) {
    if constexpr (EPI == CW_EPI_BIAS_GELU_ERF) return gelu_erf_smooth(x);
    else return gemm_bf16::epi_act<EPI>(x);
}

// Slab I of a tile (accumulator rows I of both wavefront rows: 2 x 32 rows x BN columns): value = acc + addends + bias,
// optional pre-activation store, activation, rounding, staged through one of two LDS buffers and stored as rows.
// Stores of unaligned rows are 16 bytes at their element's address (global accesses need no alignment), single
// elements only where a row ends.
template <int TM, int TN, int EPI, typename E>
struct Epilogue {
    static constexpr int BN = 64 * TN;
    static constexpr int CP = BN + 8;
    static constexpr int BUF = 64 * CP;  // elements per staging buffer

    // The lane's bias values (zeros without a bias) from the tile's in LDS, read once for all slabs: per use, behind the
    // staging writes, each read would expose its latency (64 reads a tile, 2.7 us).
    using Bias = u32x2_t[TN][4];
    static __device__ __forceinline__ void load_bias(const uint16_t* tile_bias, Bias& bias, int wn, int lane) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                bias[j][g] = *reinterpret_cast<const u32x2_t*>(tile_bias + wn * 32 * TN + 4 * (lane >> 5) + j * 32 + 8 * g);
    }
    // One path for whole and edge tiles, without branches around the sums (across branches the compiler moves the
    // accumulators' reads together and spills them): what lies outside M x N is computed from clamped addend positions and
    // not stored.
    template <bool ACT>
    static __device__ __forceinline__ void stage(const f32x16_t (&acc)[TN], int slab, const TileArgs& a, uint16_t* buf, const Bias& bias,
                                                 int m0, int n0, int wm, int wn, int lane) {
        const int mrow = m0 + (wm * TM + slab) * 32 + (lane & 31);
        const int col_l = wn * 32 * TN + 4 * (lane >> 5);
        uint16_t* dst = buf + (wm * 32 + (lane & 31)) * CP + col_l;
        const int64_t add_row = (int64_t)(mrow < a.M ? mrow : a.M - 1) * a.ldadd;
        const int last_col = (a.N - 1) & ~3;
        // An addend's pieces of a column block are requested together, ahead of the arithmetic. Addend rows are 16-byte
        // aligned (the host copies others), so the last group of four is whole memory.
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            float add[4][4];
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int e = 0; e < 4; ++e) add[g][e] = 0.0f;
#pragma unroll 1
            for (int k = 0; k < a.n_addends; ++k) {
                const uint16_t* ap = reinterpret_cast<const uint16_t*>(step_ptr(kTabAddend, k)) + add_row;
                u32x2_t raw[4];
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int col = n0 + col_l + j * 32 + 8 * g;
                    raw[g] = *reinterpret_cast<const u32x2_t*>(ap + (col < last_col ? col : last_col));
                }
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    add[g][0] += half_conv<E>::lo(raw[g].x);
                    add[g][1] += half_conv<E>::hi(raw[g].x);
                    add[g][2] += half_conv<E>::lo(raw[g].y);
                    add[g][3] += half_conv<E>::hi(raw[g].y);
                }
            }
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                // opaque: the sums are formed here and not, once for both stagings, in front of them, where all would be live at once
                u32x2_t b = bias[j][g];
                asm volatile("" : "+v"(b));
                float v[4];
                v[0] = acc[j][4 * g] + half_conv<E>::lo(b.x) + add[g][0];
                v[1] = acc[j][4 * g + 1] + half_conv<E>::hi(b.x) + add[g][1];
                v[2] = acc[j][4 * g + 2] + half_conv<E>::lo(b.y) + add[g][2];
                v[3] = acc[j][4 * g + 3] + half_conv<E>::hi(b.y) + add[g][3];
                if constexpr (ACT) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = tile_act<EPI>(v[e]);
                }
                u32x2_t p;
                p.x = half_conv<E>::pack2(v[0], v[1]);
                p.y = half_conv<E>::pack2(v[2], v[3]);
                *reinterpret_cast<u32x2_t*>(dst + j * 32 + 8 * g) = p;
            }
        }
    }
    template <bool FAST>
    static __device__ __forceinline__ void store(const uint16_t* buf, int slab, uint16_t* out, int64_t ld, const TileArgs& a, int m0,
                                                 int n0, int tid) {
        constexpr int CH = BN / 8, RPP = kThreads / CH;
        const int r = tid / CH, cq = tid % CH;
        const uint16_t* src = buf + r * CP + cq * 8;
#pragma unroll
        for (int pass = 0; pass < 64 / RPP; ++pass) {
            const int lr = r + RPP * pass;
            const int grow = m0 + (lr >= 32 ? 32 * TM : 0) + slab * 32 + (lr & 31);
            const u32x4_t v = *reinterpret_cast<const u32x4_t*>(src + pass * RPP * CP);
            uint16_t* dst = out + (int64_t)grow * ld + n0 + cq * 8;
            if constexpr (FAST) {
                *reinterpret_cast<u32x4_t*>(dst) = v;
            } else if (grow < a.M) {
                const int left = a.N - (n0 + cq * 8);
                if (left >= 8) {
                    __builtin_memcpy(dst, &v, 16);
                } else {
#pragma unroll
                    for (int i = 0; i < 7; ++i)
                        if (i < left) dst[i] = (uint16_t)(v[i >> 1] >> ((i & 1) * 16));
                }
            }
        }
    }
    static __device__ __forceinline__ void slab_out(const f32x16_t (&acc)[TN], int slab, const TileArgs& a, bool whole, uint16_t* lds,
                                                    const Bias& bias, int& buf, int m0, int n0, int wm, int wn, int lane, int tid) {
        auto out = [&](void* dst, int64_t ld) {
            __syncthreads();
            if (whole) store<true>(lds + buf * BUF, slab, reinterpret_cast<uint16_t*>(dst), ld, a, m0, n0, tid);
            else store<false>(lds + buf * BUF, slab, reinterpret_cast<uint16_t*>(dst), ld, a, m0, n0, tid);
            buf ^= 1;
        };
        if (a.preact != nullptr) {
            stage<false>(acc, slab, a, lds + buf * BUF, bias, m0, n0, wm, wn, lane);
            out(a.preact, a.ldp);
        }
        stage<true>(acc, slab, a, lds + buf * BUF, bias, m0, n0, wm, wn, lane);
        out(a.C, a.ldc);
    }
};

template <int TN>
constexpr size_t kEpilogueLds = (size_t)4 * 64 * (64 * TN + 8) + kThreads * 2;  // two staging buffers, the bias
template <int TM, int TN, int KB, int NS>
constexpr size_t kLdsBytes = (size_t)NS * KB * 64 * (TM + TN) * kBK * 2 > kEpilogueLds<TN> ? (size_t)NS * KB * 64 * (TM + TN) * kBK * 2
                                                                                          : kEpilogueLds<TN>;
// Resident blocks: two where the ring leaves room (their phases interleave on each SIMD), else one with all registers.
template <int TM, int TN, int KB, int NS>
constexpr int kBlocksPerCU = kLdsBytes<TM, TN, KB, NS> <= 80 * 1024 ? 2 : 1;

// KB: k extent of a trip in units of 32 (one barrier per trip); NS: ring stages of KB k blocks.
template <bool TRANS_A, bool TRANS_B, int TM, int TN, int KB, int NS, int EPI, typename E>
__global__ __launch_bounds__(kThreads, (kBlocksPerCU<TM, TN, KB, NS>)) void gemm_tile_kernel(const TileArgs args) {
    constexpr int BM = 64 * TM, BN = 64 * TN, BK = KB * kBK;
    using LA = Loader<TRANS_A, TM, KB>;
    using LB = Loader<TRANS_B, TN, KB>;
    constexpr int kStage = LA::kBytes + LB::kBytes;  // of a trip: A, B
    constexpr int kPer = KB * (TM + TN);             // load instructions per wavefront and trip
    extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
    lds_char* lds_base = (lds_char*)lds;
    const uint32_t lds_addr0 = (uint32_t)(uintptr_t)lds_base;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int M = args.M, N = args.N, K = args.K;
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    const int kps = (K + BK - 1) / BK;  // trips per step
    // workgroup ids are dealt round-robin to the 8 XCDs: each gets a contiguous range of the whole tiles, then a
    // contiguous range of the (slice, tile) units, whose tiles share operand panels in its L2
    int tile, kt_beg = 0, KT = kps * args.n_steps, unit = -1;
    {
        const int full_grid = (args.full + 7) & ~7;
        const int pid = blockIdx.x;
        if (pid < full_grid) {
            tile = (pid & 7) * (full_grid >> 3) + (pid >> 3);
            if (tile >= args.full) return;
        } else {
            const int rest = tiles_m * tiles_n - args.full, units = rest * args.slices;
            const int p = pid - full_grid;
            unit = (p & 7) * ((units + 7) >> 3) + (p >> 3);
            if (unit >= units) return;
            const int z = unit / rest;
            tile = args.full + unit - z * rest;
            const int total = KT;
            kt_beg = (int)((int64_t)total * z / args.slices);
            KT = (int)((int64_t)total * (z + 1) / args.slices) - kt_beg;
        }
    }
    int tm, tn;
    tile_origin(tile, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;

    LA la;
    LB lb;
    la.init(lane, wave, args.lda, m0, M);
    lb.init(lane, wave, args.ldb, n0, N);
    Frags<TRANS_A, TM, KB> fa;
    Frags<TRANS_B, TN, KB> fb;
    fa.init(lane, wm * 32 * TM);
    fb.init(lane, wn * 32 * TN);
    // byte distance of the block's origin and of one k block
    const int64_t a_org = TRANS_A ? (int64_t)m0 * 2 : (int64_t)m0 * args.lda * 2, a_adv = TRANS_A ? args.lda * (2 * kBK) : 2 * kBK;
    const int64_t b_org = TRANS_B ? (int64_t)n0 * 2 : (int64_t)n0 * args.ldb * 2, b_adv = TRANS_B ? args.ldb * (2 * kBK) : 2 * kBK;

    f32x16_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    // the block's bias, one value a thread, fetched ahead of the operands and put into LDS by the epilogue
    uint32_t bias_bits = 0;
    if (args.bias != nullptr && tid < BN && n0 + tid < N) bias_bits = reinterpret_cast<const uint16_t*>(args.bias)[n0 + tid];

    // the trip whose loads are issued next; past the last one nothing is left (is_rem 0: the instructions fetch
    // nothing and fill a free stage with zeros), which keeps the load counting the same in every trip
    int is_left = KT, is_step = kt_beg / kps, is_stage = 0;
    int is_k = (kt_beg - is_step * kps) * BK;
    const char* is_a = step_ptr(kTabA, is_step) + a_org + (is_k / kBK) * a_adv;
    const char* is_b = step_ptr(kTabB, is_step) + b_org + (is_k / kBK) * b_adv;
    int is_rem = is_left > 0 ? K - is_k : 0;
    auto issue_one = [&](auto op) {  // instruction `op` of the trip's kPer
        const uint32_t st = lds_addr0 + is_stage * kStage;
        if constexpr (op.value < KB * TM) la.template issue<op.value>(is_a, a_adv, is_rem, st, wave);
        else lb.template issue<op.value - KB * TM>(is_b, b_adv, is_rem, st + LA::kBytes, wave);
    };
    auto issue_advance = [&]() {
        is_stage = (is_stage + 1 == NS) ? 0 : is_stage + 1;
        --is_left;
        is_a += KB * a_adv;
        is_b += KB * b_adv;
        is_rem -= BK;
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
    // k values of the trip to be published next (only a step's last trip has fewer than BK)
    int pub_rem = K - is_k, pub_stage = 0;
    const bool odd_tail = (!TRANS_A || !TRANS_B) && (K & 7) != 0;
    auto publish = [&]() {
        if (odd_tail && pub_rem < BK) {
            lds_char* st = lds_base + pub_stage * kStage;
            la.fix_tail(st, pub_rem, lane, wave);
            lb.fix_tail(st + LA::kBytes, pub_rem, lane, wave);
        }
        pub_rem -= BK;
        if (pub_rem <= 0) pub_rem = K;
        pub_stage = (pub_stage + 1 == NS) ? 0 : pub_stage + 1;
        // this wavefront's fragment reads (of a stage that is about to be refilled) and tail writes are done
        asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    lds_char* rd = lds_base;  // stage read next
    int rd_stage = 0;
    auto read_advance = [&]() {
        rd_stage = (rd_stage + 1 == NS) ? 0 : rd_stage + 1;
        rd = lds_base + rd_stage * kStage;
    };
    bf16x8_t af[2][2 * KB][TM], bfr[2][2 * KB][TN];
    auto read_one = [&](auto set, auto op) {  // fragment `op` of a trip: [k step][A fragments, B fragments]
        constexpr int KS = op.value / (TM + TN), O = op.value % (TM + TN);
        if constexpr (O < TM) af[set.value][KS][O] = fa.template read<O, KS>(rd);
        else bfr[set.value][KS][O - TM] = fb.template read<O - TM, KS>(rd + LA::kBytes);
    };
    // prologue: trips 0 .. NS-1 requested, trip 0 published and its fragments on the way
    for (int p = 0; p < NS; ++p) {
        static_for<kPer>([&](auto o) { issue_one(o); });
        issue_advance();
    }
    dma_wait<kPer*(NS - 1)>();
    publish();
    static_for<2 * KB * (TM + TN)>([&](auto o) { read_one(std::integral_constant<int, 0>{}, o); });
    read_advance();
    // Trip kt: barrier (trip kt+1 complete in LDS for everybody, the stage of trip kt free: its fragments are in
    // registers); then the MFMAs of kt with the fragment reads of kt+1 and the loads of kt+NS placed between them.
    constexpr int kMfma = 2 * KB * TM * TN, kReads = 2 * KB * (TM + TN), kOps = kReads + kPer;
    auto trip = [&](auto set) {
        constexpr int S = set.value;
        dma_wait<kPer*(NS - 2)>();
        publish();
        __builtin_amdgcn_sched_barrier(0);
        static_for<kMfma>([&](auto q) {
            constexpr int KS = q.value / (TM * TN), R = q.value % (TM * TN), I = R / TN, J = R % TN, JS = (I & 1) ? TN - 1 - J : J;
            acc[I][JS] = gemm_bf16::mfma_32x32x16<E>(bfr[S][KS][JS], af[S][KS][I], acc[I][JS]);
            constexpr int O0 = q.value * kOps / kMfma, O1 = (q.value + 1) * kOps / kMfma;
            static_for<O1 - O0>([&](auto o) {
                constexpr int OP = O0 + o.value;
                if constexpr (OP < kReads) read_one(std::integral_constant<int, 1 - S>{}, std::integral_constant<int, OP>{});
                else issue_one(std::integral_constant<int, OP - kReads>{});
            });
            __builtin_amdgcn_sched_barrier(0);
        });
        read_advance();
        issue_advance();
    };
    for (int kt = 0;;) {
        trip(std::integral_constant<int, 0>{});
        if (++kt >= KT) break;
        trip(std::integral_constant<int, 1>{});
        if (++kt >= KT) break;
    }
    dma_wait<0>();
    __syncthreads();
    if (unit >= 0) {
        // accumulator order: [TM][TN][4][256 threads] x 4 floats
        float* part = args.partial + (int64_t)unit * (BM * BN) + tid * 4;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    raw16_t u;
#pragma unroll
                    for (int e = 0; e < 4; ++e) u[e] = __float_as_uint(acc[i][j][4 * g + e]);
                    *reinterpret_cast<raw16_t*>(part + ((i * TN + j) * 4 + g) * (kThreads * 4)) = u;
                }
        return;
    }
    using Epi = Epilogue<TM, TN, EPI, E>;
    lds[2 * Epi::BUF + tid] = (uint16_t)bias_bits;
    __syncthreads();
    typename Epi::Bias bias;
    Epi::load_bias(lds + 2 * Epi::BUF, bias, wn, lane);
    int buf = 0;
    const bool whole = args.vec_out != 0 && m0 + BM <= M && n0 + BN <= N;
    static_for<TM>([&](auto i) { Epi::slab_out(acc[i.value], i.value, args, whole, lds, bias, buf, m0, n0, wm, wn, lane, tid); });
}

// Finishes the sliced tiles: block (tile, slab) adds the slices' partial sums in slice order and runs the epilogue.
template <int TM, int TN, int EPI, typename E>
__global__ __launch_bounds__(kThreads) void tile_reduce_kernel(const TileArgs args) {
    constexpr int BM = 64 * TM, BN = 64 * TN;
    using Epi = Epilogue<TM, TN, EPI, E>;
    __shared__ __attribute__((aligned(16))) uint16_t lds[kEpilogueLds<TN> / 2];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tiles_m = (args.M + BM - 1) / BM, tiles_n = (args.N + BN - 1) / BN;
    const int rest = tiles_m * tiles_n - args.full;
    const int r = blockIdx.x / TM, slab = blockIdx.x % TM;
    int tm, tn;
    tile_origin(args.full + r, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    const bool has_bias = args.bias != nullptr && tid < BN && n0 + tid < args.N;
    lds[2 * Epi::BUF + tid] = has_bias ? reinterpret_cast<const uint16_t*>(args.bias)[n0 + tid] : (uint16_t)0;
    __syncthreads();
    typename Epi::Bias bias;
    Epi::load_bias(lds + 2 * Epi::BUF, bias, wave & 1, lane);
    f32x16_t acc[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[j][e] = 0.0f;
    const float* part = args.partial + (int64_t)r * (BM * BN) + (int64_t)slab * (TN * 4 * kThreads * 4) + tid * 4;
    // several slices' pieces requested together: a launch of a few tiles waits for memory alone
    constexpr int kAhead = TN == 4 ? 2 : 4;
    const int64_t slice = (int64_t)rest * (BM * BN);
    for (int z = 0; z < args.slices; z += kAhead, part += kAhead * slice) {
        raw16_t u[kAhead][TN * 4];
#pragma unroll
        for (int a = 0; a < kAhead; ++a) {
            const float* p = part + (z + a < args.slices ? a * slice : 0);
#pragma unroll
            for (int i = 0; i < TN * 4; ++i) u[a][i] = load_raw_stream(p + i * (kThreads * 4));
        }
#pragma unroll
        for (int a = 0; a < kAhead; ++a)
            if (z + a < args.slices) {
#pragma unroll
                for (int i = 0; i < TN * 4; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[i / 4][4 * (i % 4) + e] += __uint_as_float(u[a][i][e]);
            }
    }
    int buf = 0;
    const bool whole = args.vec_out != 0 && m0 + BM <= args.M && n0 + BN <= args.N;
    Epi::slab_out(acc, slab, args, whole, lds, bias, buf, m0, n0, wave >> 1, wave & 1, lane, tid);
}

template <bool TA, bool TB, int TM, int TN, int KB, int NS, int EPI, typename E>
int launch_cfg(const TileArgs& args, hipStream_t s) {
    constexpr int BM = 64 * TM, BN = 64 * TN;
    auto kern = gemm_tile_kernel<TA, TB, TM, TN, KB, NS, EPI, E>;
    constexpr size_t lds = kLdsBytes<TM, TN, KB, NS>;
    static_assert(lds <= 160 * 1024, "LDS image does not fit the CU");
    if (const int lrc = ensure_dynamic_lds((const void*)kern, (int)lds, "gemm_tile"); lrc != CW_OK) return lrc;
    const int64_t tiles = (int64_t)((args.M + BM - 1) / BM) * ((args.N + BN - 1) / BN);
    const int64_t rest = tiles - args.full;
    const int64_t grid = ((args.full + 7) & ~7) + ((rest * args.slices + 7) & ~(int64_t)7);
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(kThreads), lds, s, args);
    if (const int rc = check_launch("gemm_tile_kernel"); rc != CW_OK || rest == 0) return rc;
    hipLaunchKernelGGL((tile_reduce_kernel<TM, TN, EPI, E>), dim3((unsigned)(rest * TM)), dim3(kThreads), 0, s, args);
    return check_launch("tile_reduce_kernel");
}

// PLAIN_ONLY: no activations (the weight-gradient orientation, which nothing asks to be activated).
template <bool TA, bool TB, bool PLAIN_ONLY, int TM, int TN, int KB, int NS, typename E>
int launch_epi(const TileArgs& args, int epilogue, hipStream_t s) {
    if constexpr (!PLAIN_ONLY) {
        switch (epilogue) {
            case CW_EPI_BIAS_GELU_TANH: return launch_cfg<TA, TB, TM, TN, KB, NS, CW_EPI_BIAS_GELU_TANH, E>(args, s);
            case CW_EPI_BIAS_GELU_ERF: return launch_cfg<TA, TB, TM, TN, KB, NS, CW_EPI_BIAS_GELU_ERF, E>(args, s);
            case CW_EPI_BIAS_RELU: return launch_cfg<TA, TB, TM, TN, KB, NS, CW_EPI_BIAS_RELU, E>(args, s);
            default: break;
        }
    }
    if (epilogue != CW_EPI_NONE && epilogue != CW_EPI_BIAS) return fail(CW_ERR_INVALID, "cw_gemm_ksteps: bad epilogue %d", epilogue);
    return launch_cfg<TA, TB, TM, TN, KB, NS, CW_EPI_BIAS, E>(args, s);
}

}  // namespace gemm_tile
}  // namespace cw
