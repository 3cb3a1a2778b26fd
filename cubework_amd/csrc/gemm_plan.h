// Host-side planning of the block GEMM and of the column sums: argument validation, which kernel takes a
// shape, how a product is cut into launches (whole and sliced tiles, a strip of tile rows / columns for the small
// tiles) and how much scratch that needs (partial sums, copies of unaligned operands). Pure integer
// and pointer arithmetic with no HIP call, so that the same functions the entry points run can be driven on a
// machine without a GPU under the address and undefined-behaviour sanitizers (tests/host/plan_harness.hip):
// this is the arithmetic where an off-by-one becomes an out-of-bounds access on the device.
#pragma once

#include "gemm.h"

namespace cw {

// Checks the arguments of cw_gemm_ksteps(_ws) (the reference's assertion on mismatched operand shapes,
// cubework/module/parallel_2d/_operation.py:30, and what a C ABI has to add: null pointers, leading
// dimensions, counts) and fills the kernels' argument block with its alignment flags. Returns CW_OK, or an
// error code with the thread's error text set. *nothing_to_do is set when M or N is zero (CW_OK, no launch).
int gemm_prepare_args(int layout, int64_t M, int64_t N, int64_t K, int n_steps, const void* const* A_steps, int64_t lda,
                      const void* const* B_steps, int64_t ldb, const void* bias, int epilogue, void* C, int64_t ldc,
                      void* preact, int64_t ldp, const void* const* addends, int n_addends, int64_t ldadd, void* workspace,
                      int64_t workspace_bytes, int io_dtype, GemmArgs* out, bool* nothing_to_do);

// Scratch of the split-k launch of a 16-bit product (0: not split). For a large product over a ragged K it is 32 rows of B,
// which no launch reads any more: the size stays for callers that allocate by it.
int64_t gemm_workspace_bytes(int layout, int64_t M, int64_t N, int64_t K, int n_steps, int io_dtype);

enum GemmRoute {
    kRouteSmallRing = 0,      // 128 x 128 tiles
    kRouteRing = 1,           // 256 x 256 tiles
    kRouteRingThenSmall = 2,  // whole rounds of 256 x 256 tiles (head), the mostly empty last round as 128 x 128 tiles (tail)
    kRouteSplitK = 3,         // 256 x 256 tiles over k slices into fp32 partials, then the reduce / epilogue launch
    kRouteOther = 4,          // the best tile_plan for the scratch there is, or the register-staged kernel
};

struct GemmPlan {
    int route;
    GemmArgs head;            // the launch of every route
    GemmArgs tail;            // kRouteRingThenSmall only: the strip
    int slices;               // kRouteSplitK
    bool big;                 // register-staged kernel: 256 x 256 tiles
};

// The plan of a call whose scratch is that of gemm_workspace_bytes, or none (a call with the scratch that tile_plan asks
// for is planned by tile_plan). dma_enabled / strip_enabled: the two CW_GEMM_IMPL switches (staged / onelaunch) as the caller read them.
GemmPlan gemm_half_plan(const GemmArgs& args, int layout, bool dma_enabled, bool strip_enabled);

// ---- tile kernels (gemm_wide.h: configurations 0 and 5 to 7; gemm_tile.h: the others) ---------------------------------------
// Their configurations: block tile 64 tm x 64 tn, k extent of a trip in units of 32, ring stages, resident blocks per compute unit,
// and what a trip costs (us; one block on the unit / two) and a block besides its trips. The costs were a fit to 2000 launches over
// 110 shapes (products of 64 .. 8192 tokens with the model widths 768 .. 4096, in the forward and weight-gradient orientations; rms
// error 11 %). Configurations 0 and 5 to 7, what cutting along k costs them, and where the choice against them lies (1 and 2, the
// factors of TN) were fitted to some 250 later launches of 30 of these shapes; 3 and 4 to 14000 launches of every configuration over
// 1000 shapes (also layers of any width and vocabularies), the others held; the same launches gave the four corrections in tile_plan
// that name their shapes. Over them the error is 14 % rms (3 and 4: 20 to 24), and choosing by the costs costs 1.4 % over the best
// launch of a shape on average. 3 and 4 at 0.440, 0.800, 2.60 and 0.289, 0.460, 2.06 (2.1 %) gave short products 64 x 64 tiles in
// two rounds (us, M x N x K): 2394 x 576 x 1536 NT 15.8 / 12.9 on 64 x 128, 1894 x 1024 x 1024 NT 11.2 / 9.5, 1280 x 1024 x 1024 NT
// 10.5 / 9.1, 473 x 3072 x 768 NN 9.7 / 8.8. (The launches' times are not kept in this tree: a change of the kernels' speed means
// measuring and fitting again.)
struct TileConfig {
    int tm, tn, kb, stages, resident;
    float trip1, trip2, fixed;
};
constexpr TileConfig kTileConfigs[] = {
    {4, 4, 2, 2, 1, 1.43f, 1.43f, 4.00f},    // up to 256 x 256: the least operand traffic per FLOP, one block per compute unit
    {2, 4, 1, 3, 2, 0.480f, 0.897f, 5.00f},  // 128 x 256, two blocks
    {2, 2, 1, 5, 2, 0.285f, 0.546f, 4.50f},  // 128 x 128
    {1, 2, 2, 3, 2, 0.420f, 0.760f, 2.50f},  // 64 x 128
    {1, 1, 2, 4, 2, 0.260f, 0.550f, 2.00f},  // 64 x 64: small outputs spread over the most compute units
    {2, 2, 4, 2, 1, 0.78f, 0.78f, 4.50f},    // 128 x 128, one block of two groups of wavefronts along k (gemm_wide.h)
    {3, 2, 2, 3, 1, 0.62f, 0.62f, 4.00f},    // up to 192 x 128, 8 wavefronts (gemm_wide.h), not for TN
    {2, 2, 2, 4, 1, 0.46f, 0.46f, 4.00f},    // 128 x 128, 8 wavefronts (gemm_wide.h), not for TN
};
constexpr int kTileConfigCount = 8, kPairedConfig = 5, kNarrowConfig = 6;  // kNarrowConfig and the one behind it

// How a product runs on the tile kernels: `full` tiles whole, the others in `slices` k slices through fp32 partial
// sums. An operand whose rows are not 16-byte aligned is copied to rows that are, once per step (pack_a / pack_b).
struct TilePlan {
    int cfg;   // -1: the tile kernels do not take the shape
    int rows;  // tile height: that of the configuration, or less (configuration 0: the least of 160, 192, 224 and 256 that covers
               // M with as many tiles; configuration 6: of 160 and 192)
    int64_t tiles;
    int full, slices;
    bool rotate;
    bool pack_a, pack_b;
    int64_t lda, ldb;             // leading dimensions the kernel sees
    int64_t pack_a_bytes, pack_b_bytes, pack_add_bytes, partial_bytes;
    int64_t scratch() const { return pack_a_bytes + pack_b_bytes + pack_add_bytes + partial_bytes; }
};
// Whether a kernel of gemm_wide.h takes such a product: at least `stages` stages of `stage` k (the loads run ahead by one less).
inline bool wide_takes(int64_t K, int n_steps, int stage = 64, int stages = 3) { return (K + stage - 1) / stage * n_steps >= stages; }
// What a launch of such a kernel rests on: `tiles` tiles of which `full` are whole, the others in slices through partial sums, and every
// unit longer than the `ahead` stages that the loads run ahead (of a shorter one the loads behind its last stage are given up, the next
// unit's with them: wrong sums).
inline bool wide_units_hold(int64_t tiles, int64_t full, int slices, bool has_partial, int64_t stages, int ahead) {
    if (full < 0 || full > tiles || stages <= ahead) return false;
    return full == tiles || (slices >= 2 && has_partial && stages / slices > ahead);
}
int wide_rows(int64_t M);
int narrow_rows(int64_t M);
// max_scratch < 0: the choice with as much scratch as it likes; else the best one that fits. align_a / align_b: every step's
// pointer is 16-byte aligned and the leading dimension a multiple of 8; n_pack_addends: addends of which that is not true.
TilePlan tile_plan(int layout, int64_t M, int64_t N, int64_t K, int n_steps, int64_t lda, int64_t ldb, bool align_a, bool align_b,
                   int n_pack_addends, int64_t max_scratch);

// Row slabs of the column-sum kernels for an [M, N] operand with V elements per 16 bytes: one partial row of N
// sums per slab (vec: the vector kernel takes the shape; else the element-wise kernel).
void colsum_plan(int64_t M, int64_t N, int V, bool vec, int64_t& slabs, int64_t& rows_per_slab);
constexpr int kColWaves = 4;                 // wavefronts per block of the vector kernel, each on its own rows
constexpr int kColUnroll = 4;                // rows in flight per wavefront
constexpr int64_t kColBlocks = 1024;         // blocks aimed at (4 resident per compute unit)
constexpr int64_t kColGenericSlabRows = 64;  // rows per slab of the element-wise kernel
constexpr int64_t kColMaxSlabs = 512;        // the bound cw_colsum_workspace_bytes promises

}  // namespace cw
