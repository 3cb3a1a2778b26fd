// 16-bit block GEMM on tiles of up to 256 x 256 (gfx950): the kernel of every product with enough tiles.
//
//   - One block of 8 wavefronts (2 x 4) per compute unit walks through its tiles (grid: at most the 256 units). A wavefront
//     owns 16 TM x 64 of the tile as TM x 4 accumulators of v_mfma_f32_16x16x32, two wavefronts share a SIMD. The loads run
//     ahead over the seams of steps and of tiles, so that only the first tile of a block waits for memory, and a tile's stores
//     drain under the next tile's products.
//   - Operands go to LDS by buffer_load_dwordx4 ... lds in stages of 64 k, three stages of A and two of B: all 160 KB. Rows of 64
//     k are whole 128-byte lines: with stages of 32 k a load instruction fetched 16 pieces of 64 bytes, and the load unit takes
//     35 cycles for those against 17 (measured from L2, a compute unit: 29 and 61 bytes a cycle, where a tile needs 31).
//   - One barrier per stage, behind the second row of MFMAs of its second k step: there this wavefront's fragments of the stage
//     are all read, which frees the stage's LDS, and the next stage's first fragments are read under the remaining rows. LDS
//     reads and loads stand singly between MFMAs.
//   - 16x16x32 and not 32x32x16: the same FLOP with half of the accumulator traffic. On random operands, where the board's
//     power cap sets the clock, 8192^3 NT took 784 us against 858 with everything else alike, and the same time on zeros. Both
//     instructions give the same bits.
//
// What bounds it: matrix cores and the power cap. 8192 x 8192 x 2048 (M x N x K) in us, random bf16 from HBM, NT / NN / TN:
// 199 / 203 / 206, the kernel of 4 wavefronts and 32x32x16 that it replaced 240 / 241 / 217; 8192 x 2048 x 2048: 53 / 54,
// before 62 / 62 (a launch of one round: 6 of the 53 us are its epilogue, whose stores nothing hides). 128 accumulators, 80 fragment
// registers and the loaders' offsets fill the 256 registers of a wavefront: at 256 rows the compiler spills 11 (NT), 17 (NN) or 24 (TN)
// vector registers a lane (the headline writes 1.5 MiB more than its result a launch), at 224 rows 0 or 2.
//
// Whole 256-row tiles whose rows are mostly beyond M are wasted products: BM is 32 TM, the least of 160, 192, 224 and 256 that
// covers M with as many tiles (gemm_plan.hip).
//
// KG = 2: tiles of 128 x 128 for outputs of about 256 of them (a weight gradient of 2048 x 2048, 4096 tokens by a hidden size of
// 1024). A block of 4 wavefronts leaves one per SIMD, which waits at every barrier and for every fragment, and stages of 32 k
// run the load unit at half rate. Here two groups of 4 wavefronts own the tile together and each takes one 64 k half of a 128 k
// stage: the stage has the bytes of the 256 x 256 tile's, so the ring and its waits are the same. Their sums meet in LDS behind
// the last stage, in one order (a group's sum each, then the two added). us against 128 x 128 tiles of 4 wavefronts, NT / TN
// (M x N x K): 4096 x 1024 x 4096 42 -> 33, 2048 x 2048 x 8192 TN 79 -> 66, 1024 x 4096 x 4096 TN 41 -> 36; below about 1300 of k
// the smaller blocks' epilogue is the cheaper one (4096 x 1024 x 1024: 15 and 14). Bound by L2 -> LDS: 62 bytes a cycle and
// compute unit at the full matrix rate, where the load unit reaches 61; TN by the transposing LDS reads.
//
// TN = 2: tiles of 128 columns by 128, 160 or 192 rows for few rows (an evaluation of 300) and for NN products whose order of sums
// is fixed, which the planner does not slice. 300 rows by 256 columns are 64 tiles for a projection of 16384, and 64 or 128 x 256
// ones on blocks of 4 wavefronts fetch every weight three to five times; here 256 tiles of 160 x 128 take it in one round. The
// stages are half as long, so the loads run three (128 rows: four) ahead instead of two: weights come from HBM once and are waited
// for. us (M x N x K): 300 x 16384 x 4096 66 -> 47, 300 x 12288 x 4096 57 -> 45, 1554 x 2560 x 2560 33 -> 29 (NT 38 -> 29),
// 500 x 8192 x 2048 25 -> 22. LDS-read bound at the full matrix rate (7 fragments for 10 MFMAs), memory-bound below 160 rows.
#pragma once
#include <cstddef>

#include "gemm_plan.h"
#include "gemm_tile.h"

namespace cw {
namespace gemm_wide {

using gemm_bf16::bf16x8_t;
using gemm_bf16::static_for;
using gemm_bf16::u32x4_t;
using gemm_tile::u32x2_t;
using gemm_tile::kRange;
using gemm_tile::kTabA;
using gemm_tile::kTabAddend;
using gemm_tile::kTabB;
using gemm_tile::lds_char;
using gemm_tile::lds_u16;
using gemm_tile::s16x4_t;
using gemm_tile::s16x8_t;
using gemm_tile::step_ptr;

constexpr int kBK = 64;
typedef float f32x4_t __attribute__((ext_vector_type(4)));

template <typename E>
__device__ __forceinline__ f32x4_t mfma_16x16x32(bf16x8_t a, bf16x8_t b, f32x4_t acc) {
    if constexpr (std::is_same<E, f16_t>::value)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(gemm_bf16::f16x8_t, a), __builtin_bit_cast(gemm_bf16::f16x8_t, b), acc, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
}

// 16-byte chunks by which k row k of a k-slow image is rotated (xor)
__device__ __forceinline__ int kslow_swizzle(int k) { return ((k & 3) << 2) ^ (((k >> 3) & 1) << 1); }

// Loader of one operand: ROWS operand rows x KG images of 64 k, 1 KB per load instruction, PER instructions per wavefront and
// stage. k-contiguous image [ROWS][64 k]: chunk c of row r at c ^ ((r >> 1) & 7); k-slow image [64 k][ROWS]: chunk c of k row k
// at c ^ kslow_swizzle(k).
template <bool TRANS, int ROWS, int KG, int NW>
struct Loader {
    static constexpr int kBytes = ROWS * KG * kBK * 2;
    static constexpr int PER = ROWS * KG / 8 / NW;
    static constexpr int CPR = ROWS / 8;  // TRANS: 16-byte chunks per k row
    static_assert(ROWS * KG % (8 * NW) == 0 && ROWS % 16 == 0 && (!TRANS || (ROWS & (ROWS - 1)) == 0), "whole instructions per wavefront");
    uint32_t voff[PER];
    // k position of the lane's chunk in instruction i (k row for TRANS)
    static __device__ __forceinline__ int kpos(int lane, int wave, int i) {
        const int j = wave * PER + i;
        if constexpr (!TRANS) return ((lane & 7) ^ ((4 * j + (lane >> 4)) & 7)) * 8 + 8 * j / ROWS * kBK;
        else return (j * 64 + lane) / CPR;
    }
    __device__ __forceinline__ void init(int lane, int wave, int64_t ld, int row0, int rmax) {
        asm volatile("" : "+v"(lane));  // opaque: nothing of this is kept in registers between tiles
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int j = wave * PER + i, k = kpos(lane, wave, i);
            if constexpr (!TRANS) {
                const int r = 8 * j % ROWS + (lane >> 3);
                voff[i] = row0 + r < rmax ? (uint32_t)(((int64_t)r * ld + k) * 2) : kRange;
            } else {
                const int c = ((j * 64 + lane) % CPR) ^ kslow_swizzle(k);
                voff[i] = row0 + c * 8 < rmax ? (uint32_t)(((int64_t)k * ld + c * 8) * 2) : kRange;
            }
        }
    }
    template <int I>
    __device__ __forceinline__ void issue(const char* base, uint32_t lds_oper) const {
        dma16_buffer(base, voff[I], lds_oper + I * 1024);
    }
    // the lane's chunks at k positions from k_rem on are not fetched (until the next init)
    __device__ __forceinline__ void mask(int lane, int wave, int k_rem) {
        asm volatile("" : "+v"(lane));
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (kpos(lane, wave, i) >= k_rem) voff[i] = kRange;
    }
    // k-contiguous rows whose K is no multiple of 8: what the wavefront's chunks hold behind K, in a stage that has arrived and is
    // not yet published, becomes zeros (`lds_oper` as in issue)
    static __device__ __forceinline__ void zero_tail(int lane, int wave, int k_rem, lds_char* lds_oper) {
        if constexpr (!TRANS) {
            asm volatile("" : "+v"(lane));
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                const int d = k_rem - kpos(lane, wave, i);
                if (d <= 0 || d >= 8) continue;
                volatile lds_u16* chunk = (volatile lds_u16*)(lds_oper + i * 1024 + lane * 16);
                for (int e = d; e < 8; ++e) chunk[e] = 0;
            }
        }
    }
};

// Fragment reads of one operand: W MFMA tiles of 16 rows x 32 k per wavefront from operand row wrow of a 64 k image on, which
// begins `image` bytes behind the operand.
template <bool TRANS, int ROWS, int W>
struct Frags {
    uint32_t off[TRANS ? W : 2];
    __device__ __forceinline__ void init(int lane, int wrow, uint32_t image) {
        const int i = lane & 15, q = lane >> 4;
        if constexpr (!TRANS) {
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) off[ks] = image + (uint32_t)((wrow + i) * 128 + (((4 * ks + q) ^ ((i >> 1) & 7)) << 4));
        } else {
            const int k = 8 * q + (i >> 2);
#pragma unroll
            for (int t = 0; t < W; ++t) off[t] = image + (uint32_t)(k * (ROWS * 2) + (((wrow / 8 + 2 * t + ((i & 3) >> 1)) ^ kslow_swizzle(k)) << 4) + 8 * (i & 1));
        }
    }
    template <int T, int KS>
    __device__ __forceinline__ bf16x8_t read(lds_char* oper) const {
        if constexpr (!TRANS) {
            return *(__attribute__((address_space(3))) const bf16x8_t*)(oper + off[KS] + T * 16 * 128);
        } else {
            lds_char* p = oper + off[T] + KS * 32 * (ROWS * 2);
            const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)p);
            const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(p + 4 * (ROWS * 2)));
            const s16x8_t v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            return __builtin_bit_cast(bf16x8_t, v);
        }
    }
};

// What follows the sums: a wavefront's accumulators go through LDS of its own, one row of TN MFMA tiles (16 x 16 TN)
// at a time, and come back as 8 columns of a row per lane: addends and results move as 16 bytes per lane, 128-byte
// lines per 8 lanes (TN = 2: 64 bytes per 4), edges are a matter of one lane, and no accumulator is copied to another register.
// With addends, and for TN = 2, the sums go through as fp32: chunk c (4 columns) of row r stands at c ^ r. Without addends TN = 4
// applies bias and activation first and sends rounded results, half of the bytes, chunk c (8 columns) of row r at c ^ (r / 2). No load
// runs beside any of this, so its instructions count: rounded results, a pair of them converted at a time and addresses of whole tiles
// as a scalar took 4096 x 3072 x 768 from 27.2 / 26.7 / 28.0 us (NN / NT / TN) to 25.6 / 24.9 / 26.5, 8192 x 10240 x 2560 from 324 / 325 /
// 335 to 322 / 317 / 325, GELU of 4096 x 3072 x 768 from 30.6 to 29.5. TN = 2 gains nothing by it (1554 x 10240 x 2560 NN 97.6 -> 98.6).
template <int TN, int EPI, typename E>
struct Out {
    static constexpr int kPitch = 64 * TN, kPatch = 16 * kPitch;  // bytes of a row, of the wavefront's patch
    static constexpr int LPR = 2 * TN, kHalves = TN / 2, kHalfRows = 64 / LPR;  // lanes of a row, passes, rows of a pass
    static_assert(TN == 2 || TN == 4, "");
    static constexpr int kPitch16 = 128, kPatch16 = 16 * kPitch16;  // the same of rounded results (TN = 4): two patches of a half
    lds_char *wr, *rd;      // the lane's addresses in the wavefront's patch
    lds_char *wr16, *rd16;  // the same of rounded results
    int col4;               // the lane's first column of the accumulators
    int row0, col0;         // of the wavefront
    int row, col, M, N;  // of the lane's piece in half 0 of row 0 of the tiles
    static constexpr int64_t kFastPitch = 1 << 26;  // 16 rows' offset in 32 bits
    bool whole;
    __device__ __forceinline__ Out(const TileArgs& a, lds_char* patch, int row0, int col0, bool whole_tile, int lane) : row0(row0), col0(col0) {
        asm volatile("" : "+v"(lane));  // opaque: nothing of this is kept in registers between tiles
        const int r = lane & 15, q = lane >> 4, rr = lane / LPR, c = lane % LPR, m = 4 * TN - 1;
        wr = patch + r * kPitch + ((q ^ (r & m)) << 4);
        rd = patch + rr * kPitch + (((2 * c) ^ (rr & m)) << 4);
        wr16 = patch + r * kPitch16 + (((q >> 1) ^ (r >> 1)) << 4) + 8 * (q & 1);
        rd16 = patch + rr * kPitch16 + ((c ^ (rr >> 1)) << 4);
        col4 = col0 + 4 * q;
        row = row0 + rr;
        col = col0 + 8 * c;
        M = a.M;
        N = a.N;
        whole = whole_tile;
    }
    static __device__ __forceinline__ lds_char* flip(lds_char* p, uint32_t bits) { return (lds_char*)(uintptr_t)((uint32_t)(uintptr_t)p ^ bits); }
    __device__ __forceinline__ void put(const f32x4_t (&acc)[TN]) const {
#pragma unroll
        for (int j = 0; j < TN; ++j) *(__attribute__((address_space(3))) f32x4_t*)flip(wr, 64 * j) = acc[j];
    }
    // pass H of the row of tiles in the patch (TN = 4: 8 rows each)
    template <int H>
    __device__ __forceinline__ void get(float (&v)[8]) const {
        lds_char* p = flip(rd, H * 128) + H * 2048;
        const f32x4_t lo = *(__attribute__((address_space(3))) const f32x4_t*)p;
        const f32x4_t hi = *(__attribute__((address_space(3))) const f32x4_t*)flip(p, 16);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = lo[e];
            v[4 + e] = hi[e];
        }
    }
    // an addend's piece of row r (16-byte aligned rows: the host copies others, so the last group of eight is whole memory)
    __device__ __forceinline__ u32x4_t addend(const TileArgs& a, int k, int r) const {
        const int last = (N - 1) & ~7;
        const uint16_t* p = reinterpret_cast<const uint16_t*>(step_ptr(kTabAddend, k)) + (int64_t)(r < M ? r : M - 1) * a.ldadd;
        return *reinterpret_cast<const u32x4_t*>(p + (col < last ? col : last));
    }
    static __device__ __forceinline__ void add(float (&v)[8], const u32x4_t& raw) {
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            v[2 * d] += half_conv<E>::lo(raw[d]);
            v[2 * d + 1] += half_conv<E>::hi(raw[d]);
        }
    }
    __device__ __forceinline__ void store(const float (&v)[8], void* dst, int64_t ld, int r) const {
        u32x4_t o;
#pragma unroll
        for (int d = 0; d < 4; ++d) o[d] = half_conv<E>::pack2(v[2 * d], v[2 * d + 1]);
        store_piece(o, dst, ld, r);
    }
    __device__ __forceinline__ void store_piece(u32x4_t o, void* dst, int64_t ld, int r) const {
        uint16_t* out = reinterpret_cast<uint16_t*>(dst) + (int64_t)r * ld + col;
        if (whole) {
            *reinterpret_cast<u32x4_t*>(out) = o;
        } else if (r < M) {
            const int left = N - col;
            if (left >= 8) {
                __builtin_memcpy(out, &o, 16);
            } else {
#pragma unroll
                for (int e = 0; e < 7; ++e)
                    if (e < left) out[e] = (uint16_t)(o[e >> 1] >> ((e & 1) * 16));
            }
        }
    }
    __device__ __forceinline__ void finish(float (&v)[8], const TileArgs& a, int r) const {
        if (a.preact != nullptr) store(v, a.preact, a.ldp, r);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = gemm_tile::tile_act<EPI>(v[e]);
        store(v, a.C, a.ldc, r);
    }
    // of the lane's piece
    __device__ __forceinline__ u32x4_t bias8(const TileArgs& a) const {
        if (a.bias == nullptr) return u32x4_t{0u, 0u, 0u, 0u};
        const uint16_t* b = reinterpret_cast<const uint16_t*>(a.bias) + col;
        if (whole && ((uintptr_t)a.bias & 15) == 0) return *reinterpret_cast<const u32x4_t*>(b);
        uint32_t w[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) w[e] = col + e < N ? b[e] : 0u;
        return u32x4_t{w[0] | w[1] << 16, w[2] | w[3] << 16, w[4] | w[5] << 16, w[6] | w[7] << 16};
    }
    // bias and activation where the sums are: a lane has 4 columns of a row in each MFMA tile
    template <bool ACT, bool BIAS>
    __device__ __forceinline__ void put_rounded(const f32x4_t (&acc)[TN], const u32x2_t (&bias4)[TN], int buf) const {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            f32x4_t v = acc[j];
            if constexpr (BIAS) {
                v[0] += half_conv<E>::lo(bias4[j].x);
                v[1] += half_conv<E>::hi(bias4[j].x);
                v[2] += half_conv<E>::lo(bias4[j].y);
                v[3] += half_conv<E>::hi(bias4[j].y);
            }
            if constexpr (ACT) {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = gemm_tile::tile_act<EPI>(v[e]);
            }
            *(__attribute__((address_space(3))) u32x2_t*)(flip(wr16, 32 * j) + buf * kPatch16) =
                u32x2_t{half_conv<E>::pack2(v[0], v[1]), half_conv<E>::pack2(v[2], v[3])};
        }
    }
    // row I of the tiles; FAST: of a whole tile, whose addresses are a scalar and one offset of the lane
    template <int I, bool FAST>
    __device__ __forceinline__ void store_rounded(int buf, void* dst, int64_t ld, int r) const {
        u32x4_t o[kHalves];
#pragma unroll
        for (int h = 0; h < kHalves; ++h) o[h] = *(__attribute__((address_space(3))) const u32x4_t*)(flip(rd16, 64 * h) + h * 1024 + buf * kPatch16);
#pragma unroll
        for (int h = 0; h < kHalves; ++h) {
            if constexpr (FAST) {
                char* base = reinterpret_cast<char*>(dst) + 2 * ((int64_t)(row0 + 16 * I + kHalfRows * h) * ld + col0);
                *reinterpret_cast<u32x4_t*>(base + 2u * ((uint32_t)(row - row0) * (uint32_t)ld + (uint32_t)(col - col0))) = o[h];
            } else {
                store_piece(o[h], dst, ld, r + kHalfRows * h);
            }
        }
    }
    template <bool FAST, bool BIAS, bool PREACT, int TM>
    __device__ __forceinline__ void walk_rounded(const f32x4_t (&acc)[TM][TN], const u32x2_t (&bias4)[TN], const TileArgs& a) const {
        if constexpr (!PREACT) put_rounded<true, BIAS>(acc[0], bias4, 0);
        static_for<TM>([&](auto i) {
            constexpr int I = i.value;
            int r = row + 16 * I;
            asm volatile("" : "+v"(r));  // opaque: the addresses of a row are formed here and not for all rows at once
            if constexpr (PREACT) {
                put_rounded<false, BIAS>(acc[I], bias4, 0);
                put_rounded<true, BIAS>(acc[I], bias4, 1);
                store_rounded<I, FAST>(0, a.preact, a.ldp, r);
                store_rounded<I, FAST>(1, a.C, a.ldc, r);
            } else {
                if constexpr (I + 1 < TM) put_rounded<true, BIAS>(acc[I + 1], bias4, (I + 1) & 1);
                store_rounded<I, FAST>(I & 1, a.C, a.ldc, r);
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    }
    template <int TM>
    __device__ __forceinline__ void rows_rounded(const f32x4_t (&acc)[TM][TN], const TileArgs& a) const {
        u32x2_t bias4[TN];
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int c = col4 + 16 * j;
            const uint16_t* b = reinterpret_cast<const uint16_t*>(a.bias) + c;
            bias4[j] = u32x2_t{0x80008000u, 0x80008000u};  // no bias: -0, which changes no sum, not even one of -0
            if (a.bias != nullptr) {
                if (whole && ((uintptr_t)a.bias & 7) == 0) {
                    bias4[j] = *reinterpret_cast<const u32x2_t*>(b);
                } else {
                    uint32_t w[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) w[e] = c + e < N ? b[e] : 0u;
                    bias4[j] = u32x2_t{w[0] | w[1] << 16, w[2] | w[3] << 16};
                }
            }
        }
        const bool fast = whole && a.ldc < kFastPitch && (a.preact == nullptr || a.ldp < kFastPitch);
        // whole tiles have walks of their own, edges share one: a -0 as the bias of none costs 1 us a tile where all take it
        if (fast && a.preact == nullptr && a.bias == nullptr) return walk_rounded<true, false, false>(acc, bias4, a);
        if (fast && a.preact == nullptr) return walk_rounded<true, true, false>(acc, bias4, a);
        if constexpr (EPI != CW_EPI_BIAS)
            if (fast) return walk_rounded<true, true, true>(acc, bias4, a);
        if (a.preact == nullptr) walk_rounded<false, true, false>(acc, bias4, a);
        else walk_rounded<false, true, true>(acc, bias4, a);
    }
    template <int TM>
    __device__ __forceinline__ void rows(const f32x4_t (&acc)[TM][TN], const TileArgs& a) const {
        if constexpr (TN == 4) {
            if (a.n_addends == 0) return rows_rounded(acc, a);
        }
        const u32x4_t bias = bias8(a);
        put(acc[0]);
        if (TN == 2 && a.n_addends == 0) {
            static_for<TM>([&](auto i) {
                float v[kHalves][8];
                static_for<kHalves>([&](auto h) { get<h.value>(v[h.value]); });
                if constexpr (i.value + 1 < TM) put(acc[i.value + 1]);
#pragma unroll
                for (int h = 0; h < kHalves; ++h) add(v[h], bias);
                int r = row + 16 * i.value;
                asm volatile("" : "+v"(r));  // opaque: the addresses of a row are formed here and not for all rows at once
#pragma unroll
                for (int h = 0; h < kHalves; ++h) finish(v[h], a, r + kHalfRows * h);
                __builtin_amdgcn_sched_barrier(0);
            });
        } else {
            constexpr int G = TM < 2 ? 1 : 2;  // rows of tiles whose pieces of the first addend are requested together
            u32x4_t raw[G][kHalves];
            static_for<TM>([&](auto i) {
                if constexpr (i.value % G == 0) {
#pragma unroll
                    for (int g = 0; g < G && i.value + g < TM; ++g) {
                        int r = row + 16 * (i.value + g);
                        asm volatile("" : "+v"(r));
#pragma unroll
                        for (int h = 0; h < kHalves; ++h) raw[g][h] = addend(a, 0, r + kHalfRows * h);
                    }
                }
                float v[kHalves][8];
                static_for<kHalves>([&](auto h) { get<h.value>(v[h.value]); });
                if constexpr (i.value + 1 < TM) put(acc[i.value + 1]);
#pragma unroll
                for (int h = 0; h < kHalves; ++h) {
                    int r = row + 16 * i.value + kHalfRows * h;
                    asm volatile("" : "+v"(r));
                    add(v[h], bias);
                    add(v[h], raw[i.value % G][h]);
                    for (int k = 1; k < a.n_addends; ++k) add(v[h], addend(a, k, r));
                    finish(v[h], a, r);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        }
    }
};

constexpr int NW = 8, WM = 2;  // wavefronts of a block, along M
constexpr int kThreads = 64 * NW, kUnits = 256;

// TN = 4, KG = 1: the wavefronts are 2 x 4, each of 16 TM x 64 of the tile. TN = 2: each of 16 TM x 32. KG = 2: two groups of 2 x 2,
// each of which owns the whole tile and takes one half of a stage's 128 k; behind the last stage they exchange halves of their sums.
template <int TM, int TN, int KG>
struct Shape {
    static constexpr int WN = 4 / KG, BM = 16 * WM * TM, BN = 16 * WN * TN, kStage = KG * kBK;
    // rows of the operands' LDS images (of A, BM of them are fetched)
    static constexpr int kRowsA = TN == 4 ? 256 / KG : (BM + 63) / 64 * 64, kRowsB = BN;
    // stages that the loads run ahead: what 160 KB of LDS hold
    static constexpr int kAhead = TN == 4 ? 2 : TM == 4 ? 4 : 3, kStagesA = kAhead + 1, kStagesB = kAhead;
    static constexpr size_t kLdsBytes = (size_t)(kStagesA * kRowsA + kStagesB * kRowsB) * kStage * 2;
    static constexpr int kOutTM = TM / KG;  // rows of MFMA tiles that a wavefront finishes
    static_assert(BM <= kRowsA && TM % KG == 0 && (KG == 1 || TN == 4), "");
    static_assert(kLdsBytes <= 160 * 1024 && kRowsA * kStage * 2 >= NW * 1024 * TN, "one block per compute unit; the epilogue's patches in a free stage of A");
    static __device__ __forceinline__ int group(int wave) { return wave / (WM * WN); }
    static __device__ __forceinline__ int wm(int wave) { return wave / WN % WM; }
    static __device__ __forceinline__ int wn(int wave) { return wave % WN; }
    static __device__ __forceinline__ int out_row(int wave) { return wm(wave) * 16 * TM + group(wave) * 16 * kOutTM; }
    static __device__ __forceinline__ int out_col(int wave) { return wn(wave) * 16 * TN; }
};

template <bool TRANS_A, bool TRANS_B, int TM, int TN, int KG, int EPI, typename E>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_wide_kernel(const TileArgs args) {
    using S = Shape<TM, TN, KG>;
    constexpr int BM = S::BM, BN = S::BN, kStage = S::kStage;
    using LA = Loader<TRANS_A, S::kRowsA, KG, NW>;
    using LB = Loader<TRANS_B, S::kRowsB, KG, NW>;
    using Epi = Out<TN, EPI, E>;
    extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
    lds_char* lds_base = (lds_char*)lds;
    const uint32_t lds_a = (uint32_t)(uintptr_t)lds_base, lds_b = lds_a + S::kStagesA * LA::kBytes;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int M = args.M, N = args.N, K = args.K;
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    const int kps = (K + kStage - 1) / kStage;
    const int total = kps * args.n_steps;  // more than kAhead, as is the length of a slice
    const int full_grid = (args.full + 7) & ~7;
    const int rest = tiles_m * tiles_n - args.full, units = rest * args.slices, per_xcd = (units + 7) >> 3;
    const int pids = full_grid + 8 * per_xcd;

    struct Unit {
        int m0, n0, step, k, len, unit;
    };
    // the first unit at or after pid, which moves behind it; false (and a unit of no length) behind the last
    auto next_unit = [&](int& pid, Unit& u) -> bool {
        for (; pid < pids; pid += gridDim.x) {
            int tile, beg = 0;
            if (pid < full_grid) {
                tile = (pid & 7) * (full_grid >> 3) + (pid >> 3);
                if (tile >= args.full) continue;
                // The XCDs walk the flattened (step, k) range cyclically from starting points an eighth of it apart: walking in step, all
                // blocks would ask memory for the same k slice at the same moment, and where it comes from HBM that concentrates the
                // traffic on a few channels (8192 x 2048 x 2 x 2048 from memory, on the kernel of 4 wavefronts: k loop 95 -> 78 us).
                if (args.rotate) beg = (int)(((unsigned)total * (unsigned)(pid & 7)) >> 3);
                u.len = total;
                u.unit = -1;
            } else {
                const int p = pid - full_grid;
                u.unit = (p & 7) * per_xcd + (p >> 3);
                if (u.unit >= units) continue;
                const int z = (int)((unsigned)u.unit / (unsigned)rest), per = (int)((unsigned)total / (unsigned)args.slices), more = total - per * args.slices;
                tile = args.full + u.unit - z * rest;
                beg = z * per + (z < more ? z : more);
                u.len = per + (z < more ? 1 : 0);
            }
            const unsigned per_group = 8u * (unsigned)tiles_n, group = (unsigned)tile / per_group, in_group = (unsigned)tile - group * per_group;
            const unsigned first_m = group * 8u, gsz = (unsigned)tiles_m - first_m < 8u ? (unsigned)tiles_m - first_m : 8u;
            const unsigned tn = gsz == 8u ? in_group >> 3 : in_group / gsz;
            u.m0 = __builtin_amdgcn_readfirstlane((int)(first_m + in_group - tn * gsz)) * BM;
            u.n0 = __builtin_amdgcn_readfirstlane((int)tn) * BN;
            u.step = beg == 0 ? 0 : __builtin_amdgcn_readfirstlane((int)((unsigned)beg / (unsigned)kps));
            u.k = __builtin_amdgcn_readfirstlane(beg - u.step * kps);
            u.len = __builtin_amdgcn_readfirstlane(u.len);
            u.unit = __builtin_amdgcn_readfirstlane(u.unit);
            pid += gridDim.x;
            return true;
        }
        u.len = 0;
        return false;
    };

    LA la;
    LB lb;
    Frags<TRANS_A, S::kRowsA, TM> fa;
    Frags<TRANS_B, S::kRowsB, TN> fb;
    fa.init(lane, S::wm(wave) * 16 * TM, S::group(wave) * (LA::kBytes / KG));
    fb.init(lane, S::wn(wave) * 16 * TN, S::group(wave) * (LB::kBytes / KG));
    const int64_t a_adv = TRANS_A ? args.lda * (2 * kStage) : 2 * kStage, b_adv = TRANS_B ? args.ldb * (2 * kStage) : 2 * kStage;

    // ---- what is requested next of either operand: `cnt` stages from p on, then `part` (the stage in which a step's K ends
    // inside a stage), then the next of the unit's `left` stages, then the next unit
    struct Walk {
        const char* p;
        int cnt, part, left, step, m0;
    };
    Unit cur, nxt;
    Walk wa, wb;
    auto walk_step = [&](Walk& w, auto is_a, int k) {
        const int64_t org = is_a.value ? (TRANS_A ? (int64_t)w.m0 * 2 : (int64_t)w.m0 * args.lda * 2) : (TRANS_B ? (int64_t)w.m0 * 2 : (int64_t)w.m0 * args.ldb * 2);
        w.p = step_ptr(is_a.value ? kTabA : kTabB, w.step) + org + k * (is_a.value ? a_adv : b_adv);
        const int take = kps - k < w.left ? kps - k : w.left;
        w.part = (K % kStage) != 0 && take == kps - k ? 1 : 0;
        w.cnt = take - w.part;
        w.left -= take;
        if constexpr (is_a.value) la.init(lane, wave, args.lda, w.m0, w.m0 + BM < M ? w.m0 + BM : M);
        else lb.init(lane, wave, args.ldb, w.m0, N);
    };
    auto walk_unit = [&](Walk& w, auto is_a, const Unit& u) {
        w.m0 = is_a.value ? u.m0 : u.n0;
        w.left = u.len;
        w.step = u.step;
        walk_step(w, is_a, u.k);
    };
    auto walk_event = [&](Walk& w, auto is_a) {  // cnt is 0
        if (w.part == 0) {
            if (w.left > 0) {
                w.step = w.step + 1 == args.n_steps ? 0 : w.step + 1;
                walk_step(w, is_a, 0);
            } else if (nxt.len > 0) {
                walk_unit(w, is_a, nxt);
            } else {  // nothing is left: the instructions go on and fetch nothing
                w.cnt = INT32_MAX;
                if constexpr (is_a.value) la.mask(lane, wave, -1);
                else lb.mask(lane, wave, -1);
            }
        }
        if (w.cnt == 0) {
            w.part = 0;
            w.cnt = 1;
            if constexpr (is_a.value) la.mask(lane, wave, K % kStage);
            else lb.mask(lane, wave, K % kStage);
        }
    };
    auto walk_on = [&](Walk& w, auto is_a) {
        w.p += is_a.value ? a_adv : b_adv;
        if (--w.cnt == 0) walk_event(w, is_a);
    };
    constexpr std::true_type kA{};
    constexpr std::false_type kB{};
    constexpr uint32_t kRingA = S::kStagesA * LA::kBytes, kRingB = S::kStagesB * LB::kBytes;
    const uint32_t lds_wa = lds_a + wave * (LA::PER * 1024), lds_wb = lds_b + wave * (LB::PER * 1024);
    uint32_t wr_a = 0, wr_b = 0;  // ring positions written and read next
    uint32_t rd_a = 0, rd_b = 0;
    auto ring_on = [](uint32_t& pos, uint32_t bytes, uint32_t ring) { pos = pos + bytes == ring ? 0 : pos + bytes; };
    auto issue_a = [&](auto op) { la.template issue<op.value>(wa.p, lds_wa + wr_a); };
    auto issue_b = [&](auto op) { lb.template issue<op.value>(wb.p, lds_wb + wr_b); };

    int pid = blockIdx.x;
    if (!next_unit(pid, cur)) return;
    nxt.len = nxt.k = 0;
    walk_unit(wa, kA, cur);
    walk_unit(wb, kB, cur);
    if (wa.cnt == 0) walk_event(wa, kA);
    if (wb.cnt == 0) walk_event(wb, kB);
    for (int p = 0; p < S::kAhead; ++p) {
        static_for<LA::PER>(issue_a);
        static_for<LB::PER>(issue_b);
        ring_on(wr_a, LA::kBytes, kRingA);
        ring_on(wr_b, LB::kBytes, kRingB);
        walk_on(wa, kA);
        walk_on(wb, kB);
    }
    auto publish = [&]() {
        asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    // K that ends inside a 16-byte piece of k-contiguous rows: what is behind it in a step's last stage is cleared before that stage
    // is published, by the wavefront that fetched it: a uniform branch a stage, nothing where K is a multiple of 8. Such products ran
    // on the kernels of 4 wavefronts before (us, M x N x K): 300 x 16384 x 4092 NT 87 -> 53, 8192 x 2048 x 12565 NN 369 -> 315,
    // 8192 x 8192 x 2044 NT 250 -> 216, 1554 x 2560 x 2556 NT 40 -> 33. pk, pleft: the step's stage that is published next, stages of its unit from it on.
    const bool ragged = (!TRANS_A || !TRANS_B) && K % 8 != 0;
    int pk = cur.k, pleft = cur.len;
    auto zero_tails = [&]() {
        if (pk + 1 == kps) {
            LA::zero_tail(lane, wave, K % kStage, lds_base + wave * (LA::PER * 1024) + rd_a);
            LB::zero_tail(lane, wave, K % kStage, lds_base + kRingA + wave * (LB::PER * 1024) + rd_b);
        }
        ++pk;
        if (--pleft == 0) {
            pk = nxt.k;
            pleft = nxt.len;
        } else if (pk == kps) {
            pk = 0;
        }
    };
    f32x4_t acc[TM][TN];
    bf16x8_t af[TM], bfr[2][TN];
    lds_char *pa = lds_base, *pb = lds_base + kRingA;
    dma_wait<(S::kAhead - 1) * (LA::PER + LB::PER)>();
    if (ragged) zero_tails();
    publish();

    auto read_first = [&]() {
        static_for<TN>([&](auto t) { bfr[0][t.value] = fb.template read<t.value, 0>(pb); });
        static_for<TM>([&](auto t) { af[t.value] = fa.template read<t.value, 0>(pa); });
    };
    read_first();

    constexpr int kStores = S::kOutTM * Epi::kHalves;  // of a wavefront and whole tile: 16 bytes a lane each
    // loads behind the next stage's last one when the barrier is reached
    constexpr int kBehind = (S::kAhead - 1) * LA::PER + (S::kAhead - 2) * LB::PER;
    constexpr int kBarRow = TM > 4 ? 1 : 0;  // the row of k step 1 behind which the barrier stands
    bool stored_fast = false;
    // One k step: TM x TN MFMAs in serpentine order; what else there is to do is dealt out behind single MFMAs, so that no more
    // instructions than fit under an MFMA stand between two.
    auto k_step = [&](auto set, auto zero, auto&& behind) {
        static_for<TM>([&](auto row) {
            static_for<TN>([&](auto jc) {
                constexpr int I = row.value, J = (I & 1) ? TN - 1 - jc.value : jc.value;
                const f32x4_t z = {0.0f, 0.0f, 0.0f, 0.0f};
                acc[I][J] = mfma_16x16x32<E>(bfr[set.value][J], af[I], zero.value ? z : acc[I][J]);
                behind(row, jc);
                __builtin_amdgcn_sched_barrier(0);
            });
        });
    };
    auto stage = [&](auto first) {
        constexpr std::integral_constant<int, 0> k0{};
        constexpr std::integral_constant<int, 1> k1{};
        __builtin_amdgcn_sched_barrier(0);
        k_step(k0, first, [&](auto row, auto jc) {
            constexpr int R = row.value, P = jc.value, NB = TM - 2, H = TN / 2;
            if constexpr (P == 0 && R > 0) af[R - 1] = fa.template read<R - 1, 1>(pa);
            if constexpr (P % H == 1 % H && R < NB) {
                constexpr int T = R * TN / NB + P / H;
                if constexpr (T < (R + 1) * TN / NB) bfr[1][T] = fb.template read<T, 1>(pb);
            }
            static_for<LA::PER>([&](auto d) {
                if constexpr (d.value * TM / LA::PER == R && P == (2 + (d.value & 1) * H * (LA::PER > TM ? 1 : 0)) % TN) issue_a(d);
            });
            if constexpr (R == TM - 1 && P == TN - 1) {
                ring_on(wr_a, LA::kBytes, kRingA);
                walk_on(wa, kA);
            }
        });
        af[TM - 1] = fa.template read<TM - 1, 1>(pa);
        k_step(k1, std::false_type{}, [&](auto row, auto jc) {
            constexpr int R = row.value - kBarRow - 1, P = jc.value, NR = TM - 1 - kBarRow, H = TN / 2;
            if constexpr (R == -1 && P == TN - 1) {
                __builtin_amdgcn_sched_barrier(0);
                if (decltype(first)::value && stored_fast) dma_wait<kBehind + kStores>();
                else dma_wait<kBehind>();
                ring_on(rd_a, LA::kBytes, kRingA);
                ring_on(rd_b, LB::kBytes, kRingB);
                if (ragged) zero_tails();
                publish();
                pa = lds_base + rd_a;
                pb = lds_base + kRingA + rd_b;
            }
            if constexpr (R >= 0) {
                if constexpr ((P == 0 || P == TN - 1)) {
                    constexpr int T = R * (TM - 1) / NR + (P == 0 ? 0 : 1);
                    static_assert(T >= (R + 1) * (TM - 1) / NR || T < row.value, "a fragment is replaced behind its last use");
                    if constexpr (T < (R + 1) * (TM - 1) / NR) af[T] = fa.template read<T, 0>(pa);
                }
                if constexpr (P % H == 1 % H && R < NR - 1) {
                    constexpr int T = R * TN / (NR - 1) + P / H;
                    if constexpr (T < (R + 1) * TN / (NR - 1)) bfr[0][T] = fb.template read<T, 0>(pb);
                }
                static_for<LB::PER>([&](auto d) {
                    constexpr int D = d.value * NR / LB::PER, FIRST = (D * LB::PER + NR - 1) / NR;
                    if constexpr (D == R && P == (2 + (d.value - FIRST) * H) % TN) issue_b(d);
                });
                if constexpr (row.value == TM - 1 && P == TN - 1) {
                    ring_on(wr_b, LB::kBytes, kRingB);
                    walk_on(wb, kB);
                }
            }
        });
        af[TM - 1] = fa.template read<TM - 1, 0>(pa);
    };

    for (;;) {
        const bool more = next_unit(pid, nxt);
        stage(std::true_type{});
        for (int kt = cur.len - 1; kt > 0; --kt) stage(std::false_type{});
        stored_fast = false;
        // the slot of A that is free until the next stage's loads, which wait for the barrier below
        lds_char* patch = lds_base + wr_a;
        auto finish = [&](const auto& sum) {
            if (cur.unit >= 0) {
                // accumulator order: [kOutTM][TN][threads] x 4 floats
                float* part = args.partial + (int64_t)cur.unit * (BM * BN) + tid * 4;
#pragma unroll
                for (int i = 0; i < S::kOutTM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j) *reinterpret_cast<f32x4_t*>(part + (i * TN + j) * (kThreads * 4)) = sum[i][j];
            } else {
                const bool whole = args.vec_out != 0 && cur.m0 + BM <= M && cur.n0 + BN <= N;
                stored_fast = whole && args.preact == nullptr;
                const Epi out(args, patch + wave * Epi::kPatch, cur.m0 + S::out_row(wave), cur.n0 + S::out_col(wave), whole, lane);
                out.rows(sum, args);
            }
        };
        if constexpr (KG == 1) {
            finish(acc);
        } else {
            // group g finishes the g-th half of its wavefronts' rows of tiles; of the others, a row at a time goes to its peer
            const bool second = S::group(wave) != 0;
            f32x4_t sum[S::kOutTM][TN];
#pragma unroll
            for (int i = 0; i < S::kOutTM; ++i) {
                auto slot = [&](int w, int j) { return (__attribute__((address_space(3))) f32x4_t*)(patch + w * Epi::kPatch + j * 1024 + lane * 16); };
#pragma unroll
                for (int j = 0; j < TN; ++j) *slot(wave, j) = second ? acc[i][j] : acc[S::kOutTM + i][j];
                publish();
#pragma unroll
                for (int j = 0; j < TN; ++j) sum[i][j] = (second ? acc[S::kOutTM + i][j] : acc[i][j]) + *slot(wave ^ (NW / 2), j);
                publish();
            }
            finish(sum);
        }
        if (!more) break;
        cur = nxt;
        __builtin_amdgcn_s_barrier();
        // the next stage's first fragments once more: kept through the epilogue, they would be spilled
        asm volatile("" ::: "memory");
        read_first();
    }
    dma_wait<0>();
}

// Finishes the sliced tiles: block (tile, row of MFMA tiles) adds the slices' partial sums in slice order and runs the epilogue.
template <int TM, int TN, int KG, int EPI, typename E>
__global__ __launch_bounds__(kThreads) void wide_reduce_kernel(const TileArgs args) {
    using S = Shape<TM, TN, KG>;
    constexpr int BM = S::BM, BN = S::BN;
    using Epi = Out<TN, EPI, E>;
    __shared__ __attribute__((aligned(1024))) char lds[NW * Epi::kPatch];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tiles_m = (args.M + BM - 1) / BM, tiles_n = (args.N + BN - 1) / BN;
    const int rest = tiles_m * tiles_n - args.full;
    const int r = blockIdx.x / S::kOutTM, i = blockIdx.x % S::kOutTM;
    int tm, tn;
    gemm_tile::tile_origin(args.full + r, tiles_m, tiles_n, tm, tn);
    f32x4_t acc[1][TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[0][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    const float* part = args.partial + (int64_t)r * (BM * BN) + i * (TN * kThreads * 4) + tid * 4;
    // four slices' pieces requested together: a launch of a few tiles waits for memory alone
    constexpr int kAhead = 4;
    for (int z = 0; z < args.slices; z += kAhead, part += (int64_t)rest * (kAhead * BM * BN)) {
        raw16_t u[kAhead][TN];
#pragma unroll
        for (int a = 0; a < kAhead; ++a) {
            const float* p = part + (z + a < args.slices ? a : 0) * ((int64_t)rest * (BM * BN));
#pragma unroll
            for (int j = 0; j < TN; ++j) u[a][j] = load_raw_stream(p + j * (kThreads * 4));
        }
#pragma unroll
        for (int a = 0; a < kAhead; ++a)
            if (z + a < args.slices) {
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[0][j][e] += __uint_as_float(u[a][j][e]);
            }
    }
    const int m0 = tm * BM, n0 = tn * BN;
    const bool whole = args.vec_out != 0 && m0 + BM <= args.M && n0 + BN <= args.N;
    const Epi out(args, (lds_char*)lds + wave * Epi::kPatch, m0 + S::out_row(wave) + i * 16, n0 + S::out_col(wave), whole, lane);
    out.rows(acc, args);
}

template <bool TA, bool TB, int TM, int TN, int KG, int EPI, typename E>
int launch_rows(const TileArgs& args, hipStream_t s) {
    using S = Shape<TM, TN, KG>;
    constexpr int BM = S::BM, BN = S::BN;
    const int64_t tiles = (int64_t)((args.M + BM - 1) / BM) * ((args.N + BN - 1) / BN), rest = tiles - args.full;
    const int64_t stages = (int64_t)((args.K + S::kStage - 1) / S::kStage) * args.n_steps;
    if (!wide_units_hold(tiles, args.full, args.slices, args.partial != nullptr, stages, S::kAhead))
        return fail(CW_ERR_INVALID, "gemm_wide: %d whole tiles of %lld, the others in %d slices, of %lld stages", args.full, (long long)tiles,
                    args.slices, (long long)stages);
    auto kern = gemm_wide_kernel<TA, TB, TM, TN, KG, EPI, E>;
    if (const int lrc = ensure_dynamic_lds((const void*)kern, (int)S::kLdsBytes, "gemm_wide"); lrc != CW_OK) return lrc;
    const int64_t pids = ((args.full + 7) & ~7) + ((rest * args.slices + 7) & ~(int64_t)7);
    hipLaunchKernelGGL(kern, dim3((unsigned)(pids < kUnits ? pids : kUnits)), dim3(kThreads), S::kLdsBytes, s, args);
    if (const int rc = check_launch("gemm_wide_kernel"); rc != CW_OK || rest == 0) return rc;
    hipLaunchKernelGGL((wide_reduce_kernel<TM, TN, KG, EPI, E>), dim3((unsigned)(rest * S::kOutTM)), dim3(kThreads), 0, s, args);
    return check_launch("wide_reduce_kernel");
}

// PLAIN_ONLY: no activations (the weight-gradient orientation, which nothing asks to be activated).
template <bool TA, bool TB, bool PLAIN_ONLY, int TM, int TN, int KG, typename E>
int launch_epi(const TileArgs& args, int epilogue, hipStream_t s) {
    if constexpr (!PLAIN_ONLY) {
        switch (epilogue) {
            case CW_EPI_BIAS_GELU_TANH: return launch_rows<TA, TB, TM, TN, KG, CW_EPI_BIAS_GELU_TANH, E>(args, s);
            case CW_EPI_BIAS_GELU_ERF: return launch_rows<TA, TB, TM, TN, KG, CW_EPI_BIAS_GELU_ERF, E>(args, s);
            case CW_EPI_BIAS_RELU: return launch_rows<TA, TB, TM, TN, KG, CW_EPI_BIAS_RELU, E>(args, s);
            default: break;
        }
    }
    if (epilogue != CW_EPI_NONE && epilogue != CW_EPI_BIAS) return fail(CW_ERR_INVALID, "cw_gemm_ksteps: bad epilogue %d", epilogue);
    return launch_rows<TA, TB, TM, TN, KG, CW_EPI_BIAS, E>(args, s);
}

}  // namespace gemm_wide
}  // namespace cw
