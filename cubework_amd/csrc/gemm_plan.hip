// Host-side planning of the block GEMM and the column sums (declared in gemm_plan.h): no HIP call, no kernel.
#include <cstring>

#include "gemm_plan.h"
#include "gemm_bf16_kernel.h"

namespace cw {

int gemm_bf16_split_slices(int64_t M, int64_t N, int64_t K, int n_steps) {
    if (M <= 0 || N <= 0 || K <= 0 || n_steps <= 0 || n_steps > kRingMaxSteps) return 1;
    if ((M % 256) != 0 || (N % 256) != 0 || (K % 64) != 0) return 1;
    const int64_t tiles = (M / 256) * (N / 256);
    if (tiles >= 128 || K * n_steps < 2048) return 1;  // enough tiles already, or a short reduction
    int slices = 8;
    while (slices > 1 && (tiles * slices > 256 || (K % (64 * slices)) != 0 || K / slices < 256)) slices >>= 1;
    return slices;
}

static int64_t ragged_k_bytes(int layout, int64_t M, int64_t N, int64_t K, int n_steps) {
    if (layout == CW_NT || n_steps != 1 || K < 64 || (K % 32) == 0 || (K % 8) != 0) return 0;
    const int64_t tiles = ((M + 255) / 256) * ((N + 255) / 256);
    if (tiles < 128 || M < 256 || N < 256 || (N % 8) != 0) return 0;
    return 32 * N * (int64_t)sizeof(uint16_t);
}

int64_t gemm_workspace_bytes(int layout, int64_t M, int64_t N, int64_t K, int n_steps, int io_dtype) {
    if (layout != CW_NN && layout != CW_NT && layout != CW_TN) return 0;
    if (io_dtype != CW_BF16 && io_dtype != CW_F16) return 0;  // the fp32 GEMM is not split
    if (M <= 0 || N <= 0 || K <= 0 || M > INT32_MAX || N > INT32_MAX || K > INT32_MAX) return 0;
    const int slices = gemm_bf16_split_slices(M, N, K, n_steps);
    if (slices > 1) {
        // shapes the 128 x 128 ring kernel takes in preference to the split (gemm_half_plan) need none
        const int64_t tiles128 = ((M + 127) / 128) * ((N + 127) / 128);
        if (tiles128 >= 192 && K * n_steps < 12288) return 0;
        return (int64_t)slices * M * N * (int64_t)sizeof(float);
    }
    return ragged_k_bytes(layout, M, N, K, n_steps);
}

int gemm_prepare_args(int layout, int64_t M, int64_t N, int64_t K, int n_steps, const void* const* A_steps, int64_t lda,
                      const void* const* B_steps, int64_t ldb, const void* bias, int epilogue, void* C, int64_t ldc,
                      void* preact, int64_t ldp, const void* const* addends, int n_addends, int64_t ldadd, void* workspace,
                      int64_t workspace_bytes, int io_dtype, GemmArgs* out, bool* nothing_to_do) {
    *nothing_to_do = false;
    if (layout != CW_NN && layout != CW_NT && layout != CW_TN)
        return fail(CW_ERR_INVALID, "cw_gemm_ksteps: bad layout %d", layout);
    if (epilogue < CW_EPI_NONE || epilogue > CW_EPI_BIAS_RELU)
        return fail(CW_ERR_INVALID, "cw_gemm_ksteps: bad epilogue %d", epilogue);
    if (io_dtype != CW_BF16 && io_dtype != CW_F32 && io_dtype != CW_F16)
        return fail(CW_ERR_INVALID, "cw_gemm_ksteps: bad io_dtype %d", io_dtype);
    if (M < 0 || N < 0 || K < 0 || M > INT32_MAX || N > INT32_MAX || K > INT32_MAX)
        return fail(CW_ERR_INVALID, "cw_gemm_ksteps: bad shape M=%lld N=%lld K=%lld", (long long)M, (long long)N,
                    (long long)K);
    if (n_steps < 0 || n_steps > CW_MAX_KSTEPS)
        return fail(CW_ERR_INVALID, "cw_gemm_ksteps: n_steps=%d outside [0, %d]", n_steps, CW_MAX_KSTEPS);
    if (n_addends < 0 || n_addends > CW_MAX_ADDENDS)
        return fail(CW_ERR_INVALID, "cw_gemm_ksteps: n_addends=%d outside [0, %d]", n_addends, CW_MAX_ADDENDS);
    if (M == 0 || N == 0) {
        *nothing_to_do = true;
        return CW_OK;
    }
    if (C == nullptr || ldc < N) return fail(CW_ERR_INVALID, "cw_gemm_ksteps: C is NULL or ldc < N");
    if (preact != nullptr && ldp < N) return fail(CW_ERR_INVALID, "cw_gemm_ksteps: ldp < N");
    if (K == 0) n_steps = 0;
    if (n_steps > 0) {
        if (A_steps == nullptr || B_steps == nullptr)
            return fail(CW_ERR_INVALID, "cw_gemm_ksteps: operand pointer tables are NULL");
        const int64_t a_cols = (layout == CW_TN) ? M : K;  // contiguous extent of A's rows
        const int64_t b_cols = (layout == CW_NT) ? K : N;
        if (lda < a_cols || ldb < b_cols)
            return fail(CW_ERR_INVALID, "cw_gemm_ksteps: leading dimension smaller than the row (lda=%lld ldb=%lld)",
                        (long long)lda, (long long)ldb);
    }
    if (n_addends > 0 && (addends == nullptr || ldadd < N))
        return fail(CW_ERR_INVALID, "cw_gemm_ksteps: addends table is NULL or ldadd < N");

    GemmArgs args;
    memset(&args, 0, sizeof(args));
    const int vec = (io_dtype == CW_F32) ? 4 : 8;        // elements per 16 bytes
    const uintptr_t out_mask = 15u;                      // outputs / addends move 16 bytes at a time
    const int out_vec = (io_dtype == CW_F32) ? 4 : 8;    // elements per 16 bytes
    args.vec_a = args.vec_b = 1;
    for (int i = 0; i < n_steps; ++i) {
        if (A_steps[i] == nullptr || B_steps[i] == nullptr)
            return fail(CW_ERR_INVALID, "cw_gemm_ksteps: operand pointer of step %d is NULL", i);
        args.A[i] = A_steps[i];
        args.B[i] = B_steps[i];
        if (!aligned16(A_steps[i])) args.vec_a = 0;
        if (!aligned16(B_steps[i])) args.vec_b = 0;
    }
    if (lda % vec != 0) args.vec_a = 0;
    if (ldb % vec != 0) args.vec_b = 0;
    args.vec_add = 1;
    for (int j = 0; j < n_addends; ++j) {
        if (addends[j] == nullptr) return fail(CW_ERR_INVALID, "cw_gemm_ksteps: addend %d is NULL", j);
        args.addend[j] = addends[j];
        if ((reinterpret_cast<uintptr_t>(addends[j]) & out_mask) != 0) args.vec_add = 0;
    }
    if (ldadd % out_vec != 0) args.vec_add = 0;
    args.bias = bias;
    args.vec_bias = (bias == nullptr || (reinterpret_cast<uintptr_t>(bias) & 7u) == 0) ? 1 : 0;
    args.C = C;
    args.vec_c = ((reinterpret_cast<uintptr_t>(C) & out_mask) == 0 && ldc % out_vec == 0) ? 1 : 0;
    args.preact = preact;
    args.vec_p = (preact == nullptr || ((reinterpret_cast<uintptr_t>(preact) & out_mask) == 0 && ldp % out_vec == 0)) ? 1 : 0;
    args.lda = lda;
    args.ldb = ldb;
    args.ldc = ldc;
    args.ldp = ldp;
    args.ldadd = ldadd;
    args.M = (int)M;
    args.N = (int)N;
    args.K = (int)K;
    args.n_steps = n_steps;
    args.n_addends = n_addends;
    args.workspace = workspace_bytes > 0 ? workspace : nullptr;
    args.workspace_bytes = workspace != nullptr ? workspace_bytes : 0;
    *out = args;
    return CW_OK;
}

GemmPlan gemm_half_plan(const GemmArgs& args, int layout, bool dma_enabled, bool strip_enabled) {
    GemmPlan plan;
    memset(&plan, 0, sizeof(plan));
    plan.head = args;
    plan.tail = args;
    plan.slices = 1;
    // the unguarded kernels address operands with 32-bit byte offsets
    const int64_t max_dim = args.M > args.N ? (args.M > args.K ? args.M : args.K) : (args.N > args.K ? args.N : args.K);
    const bool fits32 = (max_dim + 64) * (args.lda > args.ldb ? args.lda : args.ldb) * 2 < ((int64_t)1 << 32);
    const bool all_vec = fits32 && args.vec_a && args.vec_b && args.vec_c && (args.preact == nullptr || args.vec_p) &&
                         (args.bias == nullptr || args.vec_bias) && (args.n_addends == 0 || args.vec_add);
    const int64_t tiles256 = (int64_t)((args.M + 255) / 256) * ((args.N + 255) / 256);
    const bool big = tiles256 >= 128;
    plan.big = big;
    const bool ring_ok = args.n_steps > 0 && args.n_steps <= kRingMaxSteps && args.n_addends <= kRingMaxAddends && dma_enabled;
    // 256 x 256 tiles also for M and N that are not tile multiples (a vocabulary slice of 12568 columns is 50 tiles instead
    // of 49.1), from one full tile in each direction on.
    const bool edges_ok = args.M >= 256 && args.N >= 256 && (args.N % 8) == 0 && (layout != CW_TN || (args.M % 8) == 0);
    // Fewer than 160 tiles of 256 x 256 (at 128 .. 159 of them the large tiles leave 40 % of the compute units
    // idle, and four times as many small tiles fill them): the ring kernel with 128 x 128 tiles, unless a long
    // reduction over few tiles is better served by splitting k (below; measured on 2048 x 2048 outputs: the
    // small tiles win up to a reduction length of 8192, the split from 16384).
    const int slices = gemm_bf16_split_slices(args.M, args.N, args.K, args.n_steps);
    const bool splits = slices > 1 && args.workspace != nullptr && aligned16(args.workspace) &&
                        args.workspace_bytes >= (int64_t)slices * args.M * args.N * (int64_t)sizeof(float);
    {
        const int64_t tiles128 = (int64_t)((args.M + 127) / 128) * ((args.N + 127) / 128);
        if (tiles256 < 160 && all_vec && ring_ok && args.M >= 128 && args.N >= 128 && (args.N % 8) == 0 &&
            (layout != CW_TN || (args.M % 8) == 0) && args.K >= 64 && (args.K % 64) == 0 &&
            args.lda < ((int64_t)1 << 23) && args.ldb < ((int64_t)1 << 23) &&
            ((tiles128 >= 192 && (int64_t)args.K * args.n_steps < 12288) || !splits)) {
            plan.route = kRouteSmallRing;
            return plan;
        }
    }
    if (big && all_vec && ring_ok && edges_ok && (args.K % gemm_bf16::kBK) == 0) {
        // A last round of 256 x 256 tiles that is mostly empty (a vocabulary slice as N: 8192 x 12568 is 32 x 50 =
        // 1600 tiles, 6.25 rounds of the 256 compute units): when the partial round is whole tile columns (or whole
        // tile rows), at most 3/8 of a round, and that strip is at most one round of 128 x 128 tiles, it goes to the
        // small-tile kernel as a second launch and the rest is whole rounds.
        const int64_t tiles_m = (args.M + 255) / 256, tiles_n = (args.N + 255) / 256;
        const int64_t last_round = (tiles_m * tiles_n) % 256;
        const bool small_ok = (args.K % 64) == 0 && args.lda < ((int64_t)1 << 23) && args.ldb < ((int64_t)1 << 23);
        if (tiles_m * tiles_n > 256 && last_round > 0 && last_round <= 96 && small_ok && strip_enabled) {
            auto shift = [&](const void* p, int64_t elems) -> const void* {
                return p == nullptr ? nullptr : reinterpret_cast<const uint16_t*>(p) + elems;
            };
            GemmArgs& head = plan.head;
            GemmArgs& tail = plan.tail;
            bool split = false;
            if (last_round % tiles_m == 0) {  // whole tile columns
                const int64_t n0 = (tiles_n - last_round / tiles_m) * 256, strip = args.N - n0;
                if (n0 >= 256 && strip >= 128 && ((args.M + 127) / 128) * ((strip + 127) / 128) <= 256) {
                    head.N = (int)n0;
                    tail.N = (int)strip;
                    for (int i = 0; i < args.n_steps; ++i) tail.B[i] = shift(args.B[i], layout == CW_NT ? n0 * args.ldb : n0);
                    for (int k = 0; k < args.n_addends; ++k) tail.addend[k] = shift(args.addend[k], n0);
                    tail.bias = shift(args.bias, n0);
                    tail.C = const_cast<void*>(shift(args.C, n0));
                    tail.preact = const_cast<void*>(shift(args.preact, n0));
                    split = true;
                }
            }
            if (!split && last_round % tiles_n == 0) {  // whole tile rows
                const int64_t m0 = (tiles_m - last_round / tiles_n) * 256, strip = args.M - m0;
                if (m0 >= 256 && strip >= 128 && ((strip + 127) / 128) * ((args.N + 127) / 128) <= 256) {
                    head.M = (int)m0;
                    tail.M = (int)strip;
                    for (int i = 0; i < args.n_steps; ++i) tail.A[i] = shift(args.A[i], layout == CW_TN ? m0 : m0 * args.lda);
                    for (int k = 0; k < args.n_addends; ++k) tail.addend[k] = shift(args.addend[k], m0 * args.ldadd);
                    tail.C = const_cast<void*>(shift(args.C, m0 * args.ldc));
                    tail.preact = const_cast<void*>(shift(args.preact, m0 * args.ldp));
                    split = true;
                }
            }
            if (split) {
                plan.route = kRouteRingThenSmall;
                return plan;
            }
        }
        plan.route = kRouteRing;
        return plan;
    }
    if (splits && all_vec && args.n_addends <= kRingMaxAddends && dma_enabled) {
        plan.slices = slices;
        plan.route = kRouteSplitK;
        return plan;
    }
    plan.route = kRouteOther;
    return plan;
}

namespace {

// Time of `count` blocks of `trips` trips each, in rounds of the chip's resident blocks (us).
double tile_rounds(const TileConfig& c, double count, double trips, double layout_factor) {
    const double cap = 256.0 * c.resident, whole = (double)(int64_t)(count / cap), left = count - whole * cap;
    double t = whole * (trips * c.trip2 * layout_factor + c.fixed);
    if (left > 0) t += trips * (left > 256 ? c.trip2 : c.trip1) * layout_factor + c.fixed;
    return t;
}

// Whole tiles of a launch: 256 work-items each, fewer than 2^32 together (as the reduction's, which are fewer).
constexpr int64_t kTileLaunchMax = ((int64_t)1 << 24) - 8;

}  // namespace

int wide_rows(int64_t M) {
    for (int rows : {160, 192, 224})
        if ((M + rows - 1) / rows == (M + 255) / 256) return rows;
    return 256;
}

int narrow_rows(int64_t M) { return (M + 159) / 160 == (M + 191) / 192 ? 160 : 192; }

TilePlan tile_plan(int layout, int64_t M, int64_t N, int64_t K, int n_steps, int64_t lda, int64_t ldb, bool align_a, bool align_b,
                   int n_pack_addends, int64_t max_scratch) {
    TilePlan best;
    memset(&best, 0, sizeof(best));
    best.cfg = -1;
    const int64_t limit = (int64_t)1 << 30;
    if (M <= 0 || N <= 0 || K <= 0 || M > limit || N > limit || K > limit || n_steps < 1 || n_steps > CW_MAX_KSTEPS) return best;
    TilePlan p = best;
    p.pack_a = !align_a;
    p.pack_b = !align_b;
    p.lda = lda;
    p.ldb = ldb;
    // A copy is one launch of a work-item per 8 elements, and a launch has fewer than 2^32 of them: larger operands are not
    // copied.
    auto copy_ld = [](int64_t cols) { return (cols + 7) / 8 * 8; };
    auto copied = [&](int64_t rows, int64_t cols) { return rows <= (((int64_t)1 << 32) - 256) * 8 / copy_ld(cols); };
    auto copy_bytes = [&](int64_t n, int64_t rows, int64_t cols) { return (n * rows * copy_ld(cols) * 2 + 255) / 256 * 256; };
    const int64_t a_rows = layout == CW_TN ? K : M, a_cols = layout == CW_TN ? M : K, b_rows = layout == CW_NT ? N : K, b_cols = layout == CW_NT ? K : N;
    if ((p.pack_a && !copied(a_rows, a_cols)) || (p.pack_b && !copied(b_rows, b_cols)) || (n_pack_addends > 0 && !copied(M, N))) return best;
    if (p.pack_a) {
        p.lda = copy_ld(a_cols);
        p.pack_a_bytes = copy_bytes(n_steps, a_rows, a_cols);
    }
    if (p.pack_b) {
        p.ldb = copy_ld(b_cols);
        p.pack_b_bytes = copy_bytes(n_steps, b_rows, b_cols);
    }
    if (n_pack_addends > 0) p.pack_add_bytes = copy_bytes(n_pack_addends, M, N);
    // the kernels' lane offsets: 256 rows of either operand (or the k rows of a trip, 128 at most) within 2 GB
    if (p.lda >= ((int64_t)1 << 22) || p.ldb >= ((int64_t)1 << 22)) return best;
    // An NN product (B stored [K, N]) that does not reduce its width, K <= N, sums k in ascending order whatever the tile: the
    // 16-bit results of a row do not depend on how many rows there are, and a ReLU behind the next layer sees the same signs.
    // That is the forward of the 2D and 3D layers' projections in front of an activation; by the same rule the 1D layers' input
    // gradient, which is NN too, while their forward is NT and is cut like any other product. Slicing gains little there
    // anyway (the outputs have tiles enough). One exception, fixed by the shape, where a row's sums are taken in another order
    // than those of a batch off the multiples of 256: whole rounds of 256 x 256 tiles start at an XCD-dependent k (memory
    // channels, gemm_wide.h). (The 16x16x32 instruction of configurations 0, 6 and 7 and the 32x32x16 one of 1 to 4 give the same bits.)
    const bool ordered = layout == CW_NN && K <= N;
    const bool rotated = ordered && M % 256 == 0 && N % 256 == 0 && K % 32 == 0 && (M / 256) * (N / 256) >= 160;
    const double bytes = 2.0 * ((double)M * K * n_steps + (double)K * N * n_steps + (double)M * N);
    const double memory_us = bytes / 4.0e6;
    double best_us = 0;
    auto consider = [&](int cfg, int rows, int64_t tiles, int64_t full, int slices) {
        const TileConfig& c = kTileConfigs[cfg];
        const int64_t rest = tiles - full;
        double trips = (double)((K + 32 * c.kb - 1) / (32 * c.kb)) * n_steps;
        TilePlan q = p;
        q.cfg = cfg;
        q.rows = rows;
        q.tiles = tiles;
        q.full = (int)full;
        q.slices = rest > 0 ? slices : 1;
        q.rotate = cfg == 0 ? !ordered || rotated : cfg >= kPairedConfig && !ordered;
        q.partial_bytes = rest * slices * (int64_t)(4096 * c.tm * c.tn) * 4;
        if (max_scratch >= 0 && q.scratch() > max_scratch) return;
        // TN on the kernels of gemm_tile.h: both operands are k-slow and move as whole lines, where the costs were fitted to k-contiguous ones
        // in pieces of 64 bytes (as 128-column tiles still move them; trips of 64 k move lines). On the paired one: the two groups' transposing
        // reads take more LDS cycles than their products.
        // 64 x 128 tiles of an NT product, at most one a unit: k-contiguous operands as lines against the same fit
        // (us, M x N x K, as chosen before / such tiles: 1554 x 768 x 2304 20.3 / 16.0, 489 x 2560 x 2560 22.5 / 17.4, 2561 x 768 x 3072 25.8 / 21.5). Two a
        // unit, 257 to 512 tiles, are left as fitted: with the factor 150 such products ran 3.6 % faster on average (2091 x 1000 x 1024 15.4 / 13.3),
        // but up to 12 % slower where rows are not whole lines (1124 x 3072 x 1144 18.1 / 20.5, 558 x 4096 x 1176 19.0 / 21.3).
        const double lines_factor = cfg == 3 && layout == CW_NT && full == tiles && tiles <= 256 ? 0.86 : 1.0;
        const double layout_factor = lines_factor * (cfg == 0 || layout != CW_TN ? 1.0 : cfg == kPairedConfig ? 1.15 : cfg == 2 ? 1.0 : 0.9);
        // Rows that are not whole 128-byte lines cost the paired kernel's loads more the longer a block walks along them (us, M x N x K):
        // whole tiles, paired / 256 x 256 in slices: 4096 x 1024 x 4104 NT 41 / 44, 4000 x 1000 x 8200 NT 70 / 81, 4096 x 1024 x 12568 NN
        // 131 / 104; the blocks of a sliced product are short, paired / 128 x 128 of one group: 1023 x 768 x 50257 NN in 5 slices 99 / 111,
        // 251 x 2048 x 50272 NN in 8 64 / 73, 2048 x 1024 x 12568 NN in 2 65 / 72, 1632 x 768 x 12568 NN in 3 45 / 50.
        auto pitch_factor = [&](double block_trips) {
            return cfg == kPairedConfig && block_trips > 80 && (p.lda % 64 != 0 || p.ldb % 64 != 0) ? 1.25 : 1.0;
        };
        // a lower tile's trips are shorter (160 rows are still priced some 15 % above what they take)
        if (rows != 64 * c.tm) trips *= 0.2 + 0.8 * rows / (64 * c.tm);
        // The kernels of gemm_wide.h: 4 us a tile, whose stores drain under the next one's products, and 3 us for the last one's. Their
        // reduction waits about 0.9 us a slice whatever its size, and its bytes come from the cache.
        // The small tiles' waits less for a slice, but priced as if it did not, outputs of few rows were cut into up to 16 of them (us, M x N x K,
        // NT, before / now: 58 x 876 x 3712 13.1 / 10.7, 49 x 896 x 2752 12.1 / 10.1, 185 x 768 x 2304 11.4 / 10.1). Of 2415 shapes of the layers in
        // every configuration this and lines_factor make 109 more than 3 % faster and none slower, all 0.5 % on average. (TN, whose k-slow
        // operands always moved as lines: as fitted.)
        const bool walks = cfg == 0 || cfg >= kPairedConfig;
        double us = tile_rounds(c, (double)full, trips, layout_factor * pitch_factor(trips)) + (walks && full > 0 ? 3.0 : 0.0);
        // All tiles of an output of more than 128 rows and columns sliced: behind the eighth slice the reduction, which requests four together,
        // waits a tenth of that, and up to 32 slices are tried (us, M x N x K, NN, up to 16 / as chosen now): 1023 x 768 x 50257 121 / 90
        // (TN 102 / 86, NT 143 / 103), 1280 x 408 x 50304 94 / 75, 178 x 1536 x 51072 66 / 48, 391 x 2048 x 32000 81 / 66. Of 330 products of
        // a long k and of the 2415 shapes of the layers this and the slower walks below make some thirty more than 3 % faster and none slower. Fewer
        // rows or columns are left to the small tiles: 34 x 3072 x 56535 TN 72 / 87.
        const bool deep = full == 0 && M > 128 && N > 128;
        const double waits = deep && slices > 8 ? 7.2 + 0.1 * (slices - 8) : 0.9 * slices;
        double reduce_us = (walks ? 2.0 + waits : layout != CW_TN ? 3.0 + 0.3 * slices : 5.0) + (walks ? 1.2 : 2.0) * q.partial_bytes / 6.6e6 * q.rows / (64 * c.tm);
        // Slices of the paired kernel slow down from some 50 trips on (NN at any pitch; NT, from 60, off the 128-byte lines; measured / priced without:
        // 1.19 in the median of 40 to 59 trips of NN, 1.28 of 60 to 79; 2048 x 512 x 30001 NT in 4 of 59 trips 94, of 256 x 256 tiles 100).
        auto slice_factor = [&](double block_trips) {
            const double pitch = pitch_factor(block_trips), longer = (block_trips - (layout == CW_NN ? 48.0 : 56.0)) / 15.0;
            const bool slows = layout == CW_NN || (layout == CW_NT && (p.lda % 64 != 0 || p.ldb % 64 != 0));
            if (!deep || cfg != kPairedConfig || !slows || longer <= 0.0) return pitch;
            const double slow = 1.0 + 0.25 * (longer < 1.0 ? longer : 1.0);
            return pitch > slow ? pitch : slow;
        };
        // Weight gradients cut in many slices of 256 x 256 tiles: all blocks write their partial sums at once and have walked little besides
        // (us, M x N x K, TN, on such slices / as chosen now): 768 x 3072 x 4416 42.7 / 35.2, 3072 x 768 x 5295 46.4 / 38.4, 1024 x 3072 x
        // 6080 53.4 / 43.5; from some 11000 of k on both are alike. Not so with k-contiguous A: 660 x 4096 x 12288 NT 71 / 78.
        if (layout == CW_TN && cfg == 0 && full == 0 && slices > 3) reduce_us += 3.0 - 0.48 * (slices < 16 ? slices : 16) + 0.37 * q.partial_bytes / 6.6e6 * q.rows / 256;
        if (rest > 0) us += tile_rounds(c, (double)(rest * slices), trips / slices, layout_factor * slice_factor(trips / slices)) + reduce_us;
        // At most one 128 x 256 tile a unit and a short k: nothing hides a block's first loads and its stores, where 128 x 128 ones share the
        // unit (us, M x N x K, 128 x 256 / 128 x 128): 2820 x 1632 x 166 TN 11.3 / 8.9, 6243 x 832 x 256 NT 12.8 / 10.8; above 576 of k
        // the costs hold as they are.
        if (cfg == 1 && full == tiles && tiles <= 256 && trips < 18) us += 1.5;
        // Weight gradients of so few tokens that a 256 x 256 tile has fewer than 7 stages: its stores do not drain under the next one's products,
        // and where the last round is a quarter full or less the smaller tiles' finer rounds are the faster ones (us, M x N x K, TN, 256 x
        // 256 / 128 x 256): 50257 x 1024 x 166 44.4 / 38.1, 50272 x 2048 x 188 76 / 67; fuller last rounds: 50257 x 2560 x 250 98 / 104.
        if (layout == CW_TN && cfg == 0 && trips < 7 && tiles % 256 > 0 && tiles % 256 <= 64) us += (double)((full + 255) / 256);
        // 128-column tiles of NN products over a long k in more than two and a half rounds: their first rounds are no slower than the costs say,
        // the later ones, under the power cap, are (us, M x N x K, such tiles / 128 x 256 or 256 x 256): 7948 x 2560 x 2560 126 / 109, 2465 x 7680
        // x 2560 121 / 106, 14502 x 2560 x 2560 188 / 169, 5280 x 4096 x 4096 177 / 171.
        if (layout == CW_NN && cfg >= kNarrowConfig && full == tiles && tiles > 640 && K * n_steps >= 2496) us *= 1.07;
        // behind whole tiles: the slices start under the last tile's stores, and nothing hides theirs (146 launches: 3 us too high in the median)
        if (cfg == 0 && rest > 0 && full > 0) us += 1.2 * q.partial_bytes / 6.6e6 - 8.0;
        us = us > memory_us ? us + 0.1 * memory_us : memory_us + 0.1 * us;
        if (best.cfg < 0 || us < best_us) {
            best = q;
            best_us = us;
        }
    };
    auto consider_rows = [&](int cfg, int rows) {
        const TileConfig& c = kTileConfigs[cfg];
        // k ranges of the kernels of gemm_wide.h: more stages than their loads run ahead
        const int least = cfg >= kNarrowConfig ? 5 : 3;
        const int64_t tiles = ((M + 64 * c.tm - 1) / (64 * c.tm)) * ((N + 64 * c.tn - 1) / (64 * c.tn));
        if (tiles > kTileLaunchMax) return;
        if ((cfg == 0 || cfg >= kPairedConfig) && !wide_takes(K, n_steps, 32 * c.kb, least)) return;
        const int64_t trips = ((K + 32 * c.kb - 1) / (32 * c.kb)) * n_steps, cap = 256 * c.resident;
        consider(cfg, rows, tiles, tiles, 1);
        // all tiles sliced, to fill the chip about once; or only those of the partial last round
        if (ordered) return;
        const int64_t last = tiles % cap;
        // more of 256-column tiles and of 128-column ones of 160 or 192 rows, where so many slices of all tiles are one round (consider)
        const int most = (cfg == 0 || cfg == kNarrowConfig) && M > 128 && N > 128 && tiles * 17 <= cap ? 32 : 16;
        for (int slices = 2; slices <= most; ++slices) {
            if (trips / slices < least) break;
            if (tiles * slices <= cap) consider(cfg, rows, tiles, 0, slices);
            else if (tiles > cap && last > 0 && last * slices <= cap) consider(cfg, rows, tiles, tiles - last, slices);
        }
    };
    for (int cfg = 0; cfg < kTileConfigCount; ++cfg) {
        if (cfg == kPairedConfig && ordered) continue;  // it sums k in another order than the other tiles do
        if (cfg >= kNarrowConfig && layout == CW_TN) continue;  // not built
        consider_rows(cfg, cfg == 0 ? wide_rows(M) : cfg == kNarrowConfig ? narrow_rows(M) : 64 * kTileConfigs[cfg].tm);
    }
    return best;
}

void colsum_plan(int64_t M, int64_t N, int V, bool vec, int64_t& slabs, int64_t& rows_per_slab) {
    if (!vec) {
        rows_per_slab = kColGenericSlabRows;
        slabs = (M + rows_per_slab - 1) / rows_per_slab;
        return;
    }
    const int64_t coltiles = (N + 64 * V - 1) / (64 * V);
    slabs = kColBlocks / coltiles;
    const int64_t max_slabs = (M + kColWaves * kColUnroll - 1) / (kColWaves * kColUnroll);
    if (slabs > max_slabs) slabs = max_slabs;
    if (slabs > kColMaxSlabs) slabs = kColMaxSlabs;
    if (slabs < 1) slabs = 1;
    rows_per_slab = (M + slabs - 1) / slabs;
    slabs = (M + rows_per_slab - 1) / rows_per_slab;
}

}  // namespace cw
