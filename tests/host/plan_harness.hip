// Host-only driver of the library's planning and validation code (cubework_amd/csrc/gemm_plan.hip with
// cw_runtime.hip's error text), built with the address and undefined-behaviour sanitizers on the host side
// (tests/test_host_sanitizers.py) and run on a machine without a GPU: no HIP call is made. It sweeps ragged,
// huge, zero and misaligned shapes through the same functions the entry points run and checks, for every plan,
// that the launches it describes stay inside the caller's buffers:
//   * a strip cut off for the small-tile kernel: head + tail cover the output exactly once, every shifted
//     pointer stays inside its operand, the strip fits one round of 128 x 128 tiles;
//   * split k: slices divide K into multiples of 64, the partial sums fit the workspace;
//   * the tile kernels' plans (tile_plan): scratch within its bound, whole and sliced tiles, copies and partial sums that
//     add up, tile heights that are built, units longer than the loads run ahead, one order of sums where it is promised, lane offsets
//     below 2 GiB, launches below 2^32 work-items;
//   * column sums: the slabs cover the rows exactly once and their partial rows fit cw_colsum_workspace_bytes'
//     promise of at most 512 (or ceil(M / 64)) rows.
// Prints "ok <checks> routes <how often each kernel route was planned>" and exits 0, or the first violated invariant and exits 1.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "../../cubework_amd/csrc/gemm_plan.h"

using namespace cw;

namespace {

long g_checked = 0;
long g_routes[5] = {0, 0, 0, 0, 0};
long g_tile_plans[3] = {0, 0, 0};  // whole tiles, every tile sliced, the last round sliced

#define REQUIRE(cond, ...)                                    \
    do {                                                      \
        if (!(cond)) {                                        \
            fprintf(stderr, "violated: %s | ", #cond);       \
            fprintf(stderr, __VA_ARGS__);                     \
            fprintf(stderr, "\n");                            \
            exit(1);                                          \
        }                                                     \
    } while (0)

struct Extent {
    const char* base;
    int64_t bytes;
};

bool inside(const void* p, int64_t need_bytes, const Extent& e) {
    const char* c = reinterpret_cast<const char*>(p);
    return c >= e.base && c + need_bytes <= e.base + e.bytes;
}

// Operands live in one fake address range per tensor (never dereferenced): the checks are on the arithmetic.
struct Problem {
    int layout;
    int64_t M, N, K, lda, ldb, ldc;
    int n_steps, n_addends;
    bool with_bias, with_preact, with_ws;
    int misalign;  // bytes added to A's base (0 = aligned)
};

int64_t a_rows(const Problem& p) { return p.layout == CW_TN ? p.K : p.M; }
int64_t a_cols(const Problem& p) { return p.layout == CW_TN ? p.M : p.K; }
int64_t b_rows(const Problem& p) { return p.layout == CW_NT ? p.N : p.K; }
int64_t b_cols(const Problem& p) { return p.layout == CW_NT ? p.K : p.N; }

void check_launch_extents(const GemmArgs& g, int layout, const Problem& p, const Extent (&A)[CW_MAX_KSTEPS],
                          const Extent (&B)[CW_MAX_KSTEPS], const Extent& C, const Extent& P, const Extent& bias,
                          const Extent (&add)[CW_MAX_ADDENDS], const char* what) {
    // the bytes a launch with these arguments touches: whole rows of its M x N output, its operands' used rows
    const int64_t ar = layout == CW_TN ? g.K : g.M, ac = layout == CW_TN ? g.M : g.K;
    const int64_t br = layout == CW_NT ? g.N : g.K, bc = layout == CW_NT ? g.K : g.N;
    REQUIRE(g.M > 0 && g.N > 0 && g.K >= 0, "%s: M=%d N=%d K=%d", what, g.M, g.N, g.K);
    for (int i = 0; i < g.n_steps; ++i) {
        REQUIRE(inside(g.A[i], ((ar - 1) * g.lda + ac) * 2, A[i]), "%s: A[%d] leaves its operand (M=%lld N=%lld K=%lld layout %d)", what,
                i, (long long)p.M, (long long)p.N, (long long)p.K, layout);
        REQUIRE(inside(g.B[i], ((br - 1) * g.ldb + bc) * 2, B[i]), "%s: B[%d] leaves its operand (M=%lld N=%lld K=%lld layout %d)", what,
                i, (long long)p.M, (long long)p.N, (long long)p.K, layout);
    }
    REQUIRE(inside(g.C, ((int64_t)(g.M - 1) * g.ldc + g.N) * 2, C), "%s: C leaves the output", what);
    if (g.preact != nullptr) REQUIRE(inside(g.preact, ((int64_t)(g.M - 1) * g.ldp + g.N) * 2, P), "%s: preact leaves its buffer", what);
    if (g.bias != nullptr) REQUIRE(inside(g.bias, (int64_t)g.N * 2, bias), "%s: bias leaves its vector", what);
    for (int j = 0; j < g.n_addends; ++j)
        REQUIRE(inside(g.addend[j], ((int64_t)(g.M - 1) * g.ldadd + g.N) * 2, add[j]), "%s: addend %d leaves its buffer", what, j);
}

void run_problem(const Problem& p) {
    // fake, well separated address ranges (1 TiB apart), 256-byte aligned
    auto range = [](int idx, int64_t bytes, int off) { return Extent{reinterpret_cast<const char*>(((int64_t)(idx + 1) << 40) + off), bytes}; };
    Extent A[CW_MAX_KSTEPS] = {}, B[CW_MAX_KSTEPS] = {}, add[CW_MAX_ADDENDS] = {};
    const void* a_tab[CW_MAX_KSTEPS] = {};
    const void* b_tab[CW_MAX_KSTEPS] = {};
    const void* add_tab[CW_MAX_ADDENDS] = {};
    for (int i = 0; i < p.n_steps && i < CW_MAX_KSTEPS; ++i) {
        A[i] = range(i, ((a_rows(p) - 1) * p.lda + a_cols(p)) * 2, p.misalign);
        B[i] = range(16 + i, ((b_rows(p) - 1) * p.ldb + b_cols(p)) * 2, 0);
        a_tab[i] = A[i].base;
        b_tab[i] = B[i].base;
    }
    const Extent C = range(40, ((p.M - 1) * p.ldc + p.N) * 2, 0), P = range(41, ((p.M - 1) * p.ldc + p.N) * 2, 0);
    const Extent bias = range(42, p.N * 2, 0);
    for (int j = 0; j < p.n_addends && j < CW_MAX_ADDENDS; ++j) {
        add[j] = range(48 + j, ((p.M - 1) * p.ldc + p.N) * 2, 0);
        add_tab[j] = add[j].base;
    }
    const int64_t ws_bytes = p.with_ws ? gemm_workspace_bytes(p.layout, p.M, p.N, p.K, p.n_steps, CW_BF16) : 0;
    REQUIRE(ws_bytes >= 0, "negative workspace size");
    const Extent W = range(60, ws_bytes, 0);
    GemmArgs args;
    bool nothing = false;
    const int rc = gemm_prepare_args(p.layout, p.M, p.N, p.K, p.n_steps, a_tab, p.lda, b_tab, p.ldb, p.with_bias ? bias.base : nullptr,
                                     p.with_bias ? CW_EPI_BIAS : CW_EPI_NONE, const_cast<char*>(C.base), p.ldc,
                                     p.with_preact ? const_cast<char*>(P.base) : nullptr, p.ldc, add_tab, p.n_addends, p.ldc,
                                     ws_bytes > 0 ? const_cast<char*>(W.base) : nullptr, ws_bytes, CW_BF16, &args, &nothing);
    ++g_checked;
    if (rc != CW_OK || nothing) return;  // refused (with a message) or empty: nothing is launched
    if (args.n_steps == 0) return;       // epilogue only
    for (int dma = 0; dma < 2; ++dma)
        for (int strip = 0; strip < 2; ++strip) {
            const GemmPlan plan = gemm_half_plan(args, p.layout, dma != 0, strip != 0);
            ++g_checked;
            REQUIRE(plan.route >= kRouteSmallRing && plan.route <= kRouteOther, "route %d", plan.route);
            ++g_routes[plan.route];
            if (!dma) REQUIRE(plan.route == kRouteOther, "CW_GEMM_IMPL=staged must reach no tile route, got route %d", plan.route);
            check_launch_extents(plan.head, p.layout, p, A, B, C, P, bias, add, "head");
            switch (plan.route) {
                case kRouteSmallRing:
                    REQUIRE(args.M >= 128 && args.N >= 128 && args.K % 64 == 0 && args.n_steps <= kRingMaxSteps, "small ring preconditions");
                    break;
                case kRouteRing:
                    REQUIRE(args.M >= 256 && args.N >= 256 && args.K % 32 == 0 && args.n_steps <= kRingMaxSteps && args.N % 8 == 0, "ring preconditions");
                    break;
                case kRouteRingThenSmall: {
                    const GemmArgs &h = plan.head, &t = plan.tail;
                    check_launch_extents(t, p.layout, p, A, B, C, P, bias, add, "tail");
                    REQUIRE((h.M == args.M && h.N + t.N == args.N && t.M == args.M) || (h.N == args.N && h.M + t.M == args.M && t.N == args.N),
                            "head %dx%d + tail %dx%d do not tile %dx%d", h.M, h.N, t.M, t.N, args.M, args.N);
                    REQUIRE(h.M % 256 == 0 || h.M == args.M, "head rows");
                    REQUIRE(h.N % 256 == 0 || h.N == args.N, "head columns");
                    REQUIRE(((int64_t)(t.M + 127) / 128) * ((t.N + 127) / 128) <= 256, "the strip is more than one round of small tiles");
                    REQUIRE(t.M >= 128 && t.N >= 128 && h.M >= 256 && h.N >= 256, "strip or head below one tile");
                    // the strip's output begins exactly where the head's ends
                    const char* c_end = reinterpret_cast<const char*>(h.C) + (h.N < args.N ? (int64_t)h.N * 2 : (int64_t)h.M * h.ldc * 2);
                    REQUIRE(reinterpret_cast<const char*>(t.C) == c_end, "the strip's output does not continue the head's");
                    break;
                }
                case kRouteSplitK:
                    REQUIRE(plan.slices >= 2 && plan.slices <= 8 && args.K % (64 * plan.slices) == 0, "slices %d of K=%d", plan.slices, args.K);
                    REQUIRE((int64_t)plan.slices * args.M * args.N * 4 <= args.workspace_bytes, "partial sums exceed the workspace");
                    REQUIRE(wide_units_hold((int64_t)(args.M / 256) * (args.N / 256), 0, plan.slices, true, (int64_t)(args.K / 64) * args.n_steps, 2), "short slices of K=%d", args.K);
                    REQUIRE((int64_t)(args.M / 256) * (args.N / 256) * plan.slices <= 256 && args.M % 256 == 0 && args.N % 256 == 0, "split grid");
                    break;
                default: break;
            }
        }
}

void sweep_gemm() {
    const int64_t dims[] = {0, 1, 7, 8, 127, 128, 129, 255, 256, 264, 2040, 2048, 2056, 4096, 4352, 8192, 8704, 12568, 16384, 50272, 1 << 20};
    const int64_t ks[] = {0, 1, 8, 24, 32, 56, 64, 88, 2048, 2072, 4096, 8192, 12568, 16384};
    for (int layout = 0; layout < 3; ++layout)
        for (int64_t M : dims)
            for (int64_t N : dims)
                for (int64_t K : ks) {
                    if ((double)M * N > 4e11 || (double)M * K > 4e11 || (double)N * K > 4e11) continue;  // keep extents in int64
                    for (int variant = 0; variant < 6; ++variant) {
                        Problem p = {};
                        p.layout = layout;
                        p.M = M;
                        p.N = N;
                        p.K = K;
                        const int64_t pad = (variant == 1) ? 8 : (variant == 2 ? 3 : 0);
                        p.lda = (layout == CW_TN ? M : K) + pad;
                        p.ldb = (layout == CW_NT ? K : N) + pad;
                        p.ldc = N + pad;
                        p.n_steps = variant == 3 ? 4 : (variant == 4 ? 7 : (variant == 5 ? 2 : 1));
                        p.n_addends = variant == 4 ? 3 : (variant == 5 ? 2 : 0);
                        p.with_bias = variant != 0;
                        p.with_preact = variant == 5;
                        p.with_ws = variant != 2;
                        p.misalign = variant == 2 ? 2 : 0;
                        if (p.lda < 1) p.lda = 1;
                        if (p.ldb < 1) p.ldb = 1;
                        if (p.ldc < 1) p.ldc = 1;
                        run_problem(p);
                    }
                }
}

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// What one plan of the tile kernels promises: it fits the scratch it was given, its tiles, slices and sub-buffers add up
// as the launches use them (gemm_bf16.hip's tile_launch, gemm_tile.h's launch_cfg, gemm_wide.h's launch_rows), and no offset or grid leaves its type.
void check_tile_plan(int layout, int64_t M, int64_t N, int64_t K, int steps, int64_t lda, int64_t ldb, bool al_a, bool al_b, int n_pack,
                     int64_t max_scratch, bool must_plan) {
    const TilePlan p = tile_plan(layout, M, N, K, steps, lda, ldb, al_a, al_b, n_pack, max_scratch);
    ++g_checked;
#define PLAN_REQUIRE(cond)                                                                                                        \
    REQUIRE(cond, "layout %d M=%lld N=%lld K=%lld steps %d lda=%lld ldb=%lld aligned %d %d addends %d scratch %lld: cfg %d full %d slices %d", \
            layout, (long long)M, (long long)N, (long long)K, steps, (long long)lda, (long long)ldb, al_a, al_b, n_pack,         \
            (long long)max_scratch, p.cfg, p.full, p.slices)
    PLAN_REQUIRE(p.cfg >= -1 && p.cfg < kTileConfigCount);
    PLAN_REQUIRE(!must_plan || p.cfg >= 0);
    if (p.cfg < 0) return;
    ++g_tile_plans[p.full == p.tiles ? 0 : (p.full == 0 ? 1 : 2)];
    const TileConfig& c = kTileConfigs[p.cfg];
    const int64_t bm = 64 * c.tm, bn = 64 * c.tn;
    PLAN_REQUIRE(p.tiles == ceil_div(M, bm) * ceil_div(N, bn));
    PLAN_REQUIRE(p.full >= 0 && p.full <= p.tiles && p.slices >= 1 && (p.full < p.tiles || p.slices == 1));
    const int64_t rest = p.tiles - p.full, trips = ceil_div(K, 32 * c.kb) * steps;
    PLAN_REQUIRE(p.slices <= trips);
    // heights that are built, with as many tiles as the configuration's own; the 128-column tiles are not built for TN
    switch (p.cfg) {
        case 0: PLAN_REQUIRE(p.rows == 160 || p.rows == 192 || p.rows == 224 || p.rows == 256); break;
        case kNarrowConfig: PLAN_REQUIRE(p.rows == 160 || p.rows == 192); break;
        default: PLAN_REQUIRE(p.rows == bm); break;
    }
    PLAN_REQUIRE(ceil_div(M, p.rows) == ceil_div(M, bm));
    PLAN_REQUIRE(p.cfg < kNarrowConfig || layout != CW_TN);
    // gemm_wide.h: every unit is longer than the loads run ahead (4 stages at most for 128 columns, 2 for the others)
    const bool walks = p.cfg == 0 || p.cfg >= kPairedConfig;
    if (walks) PLAN_REQUIRE(wide_units_hold(p.tiles, p.full, p.slices, p.partial_bytes > 0, trips, p.cfg >= kNarrowConfig ? 4 : 2));
    // a product whose rows do not depend on their number sums k in one order: not cut, no two sums, rotated on aligned 256 x 256 tiles alone
    if (layout == CW_NN && K <= N) {
        PLAN_REQUIRE(rest == 0 && p.cfg != kPairedConfig);
        PLAN_REQUIRE(!p.rotate || (p.cfg == 0 && M % 256 == 0 && N % 256 == 0));
    }
    PLAN_REQUIRE(!p.rotate || walks);
    // the partial sums of every (tile, slice), behind the copies, all at 16-byte boundaries and within the scratch
    PLAN_REQUIRE(p.partial_bytes == rest * (p.slices > 1 || rest > 0 ? p.slices : 0) * bm * bn * 4);
    PLAN_REQUIRE(p.pack_a_bytes % 16 == 0 && p.pack_b_bytes % 16 == 0 && p.pack_add_bytes % 16 == 0);
    PLAN_REQUIRE(max_scratch < 0 || p.scratch() <= max_scratch);
    // copies: every step's rows at an aligned pitch that holds them; operands that are not copied keep theirs
    const int64_t a_rows = layout == CW_TN ? K : M, a_cols = layout == CW_TN ? M : K, b_rows = layout == CW_NT ? N : K, b_cols = layout == CW_NT ? K : N;
    PLAN_REQUIRE(p.pack_a == !al_a && p.pack_b == !al_b);
    if (p.pack_a) PLAN_REQUIRE(p.lda % 8 == 0 && p.lda >= a_cols && p.pack_a_bytes >= steps * a_rows * p.lda * 2);
    else PLAN_REQUIRE(p.lda == lda && p.pack_a_bytes == 0);
    if (p.pack_b) PLAN_REQUIRE(p.ldb % 8 == 0 && p.ldb >= b_cols && p.pack_b_bytes >= steps * b_rows * p.ldb * 2);
    else PLAN_REQUIRE(p.ldb == ldb && p.pack_b_bytes == 0);
    PLAN_REQUIRE(p.pack_add_bytes >= n_pack * M * ceil_div(N, 8) * 16);
    // a lane's byte offset (the block's rows, or a trip's rows of k) stays inside the buffer's 2 GiB
    const int64_t reach = (int64_t)1 << 31, kt = 32 * c.kb;
    PLAN_REQUIRE((layout == CW_TN ? (kt - 1) * p.lda + bm : (bm - 1) * p.lda + kt) * 2 < reach);
    PLAN_REQUIRE((layout == CW_NT ? (bn - 1) * p.ldb + kt : (kt - 1) * p.ldb + bn) * 2 < reach);
    // every launch is at most 2^32 - 1 work-items: the tiles and slices, their reduction, the copies (16 bytes each)
    const int64_t items = ((int64_t)1 << 32) - 1;
    const int64_t threads = walks ? 512 : 256;  // (gemm_wide.h's launches have 256 blocks at most, their reductions one for 32 rows)
    if (!walks) PLAN_REQUIRE((ceil_div(p.full, 8) + ceil_div(rest * p.slices, 8)) * 8 * threads <= items);
    PLAN_REQUIRE(rest * (walks ? p.rows / 32 : c.tm) * threads <= items);
    for (const int64_t bytes : {p.pack_a_bytes / steps, p.pack_b_bytes / steps, n_pack > 0 ? p.pack_add_bytes / n_pack : 0})
        PLAN_REQUIRE(ceil_div(bytes, 16 * 256) * 256 <= items);
#undef PLAN_REQUIRE
}

void sweep_tile_plan() {
    const int64_t dims[] = {1, 7, 63, 64, 65, 128, 250, 256, 264, 777, 2048, 2056, 4376, 8192, 12568, 50257, 1 << 20, 3 << 20, 1 << 28, 1 << 30};
    const int64_t ks[] = {1, 8, 31, 32, 40, 72, 136, 200, 264, 331, 1003, 2048, 4096, 12568, 50257, 1 << 20, 1 << 30};
    for (int layout = 0; layout < 3; ++layout)
        for (int64_t M : dims)
            for (int64_t N : dims)
                for (int64_t K : ks)
                    for (int variant = 0; variant < 6; ++variant) {
                        const int steps = variant == 3 ? 4 : (variant == 4 ? CW_MAX_KSTEPS : 1), n_pack = variant == 2 ? 1 : (variant == 4 ? CW_MAX_ADDENDS : 0);
                        const int64_t pad = variant == 1 ? 8 : (variant == 5 ? (int64_t)1 << 22 : 0);
                        const int64_t lda = ((layout == CW_TN ? M : K) + 7) / 8 * 8 + pad + (variant == 2 ? 3 : 0);
                        const int64_t ldb = ((layout == CW_NT ? K : N) + 7) / 8 * 8 + pad + (variant == 4 ? 1 : 0);
                        const bool al_a = variant != 2, al_b = variant != 4;
                        // operands and output that a 288 GB device holds, in rows the lane offsets reach: there is a plan
                        const double bytes = 2.0 * ((double)M * K * steps * (al_a ? 1 : 2) + (double)N * K * steps * (al_b ? 1 : 2) + (double)M * N * (1 + 2 * n_pack));
                        const int64_t limit = (int64_t)1 << 22;
                        const bool wide = lda >= limit || ldb >= limit;
                        auto too_big = [](int64_t rows, int64_t cols) { return (double)rows * (double)ceil_div(cols, 8) >= 4294967040.0; };
                        const bool big_copy = (!al_a && (layout == CW_TN ? too_big(K, M) : too_big(M, K))) ||
                                              (!al_b && (layout == CW_NT ? too_big(N, K) : too_big(K, N))) || (n_pack > 0 && too_big(M, N));
                        check_tile_plan(layout, M, N, K, steps, lda, ldb, al_a, al_b, n_pack, -1, bytes < 2.9e11 && !wide && !big_copy);
                        for (const int64_t scratch : {(int64_t)0, (int64_t)4096, (int64_t)1 << 22, (int64_t)1 << 26, (int64_t)1 << 33})
                            check_tile_plan(layout, M, N, K, steps, lda, ldb, al_a, al_b, n_pack, scratch, false);
                    }
    REQUIRE(g_tile_plans[0] > 0 && g_tile_plans[1] > 0 && g_tile_plans[2] > 0, "plans: %ld whole, %ld sliced, %ld with a sliced last round",
            g_tile_plans[0], g_tile_plans[1], g_tile_plans[2]);
    for (int64_t bad : {(int64_t)0, (int64_t)-1, ((int64_t)1 << 30) + 1}) {
        REQUIRE(tile_plan(CW_NN, bad, 8, 8, 1, 8, 8, true, true, 0, -1).cfg == -1 && tile_plan(CW_NN, 8, bad, 8, 1, 8, 8, true, true, 0, -1).cfg == -1 &&
                    tile_plan(CW_NN, 8, 8, bad, 1, 8, 8, true, true, 0, -1).cfg == -1, "a plan for a size of %lld", (long long)bad);
    }
    // the launches of gemm_wide.h refuse a plan for other tiles, partial sums that nothing holds, units as short as the loads run ahead
    REQUIRE(wide_units_hold(10, 10, 1, false, 3, 2) && wide_units_hold(10, 0, 3, true, 9, 2) && wide_units_hold(10, 8, 2, true, 11, 4), "launches that hold");
    REQUIRE(!wide_units_hold(10, 11, 1, true, 9, 2) && !wide_units_hold(10, -1, 2, true, 9, 2), "a plan for other tiles");
    REQUIRE(!wide_units_hold(10, 8, 1, true, 9, 2) && !wide_units_hold(10, 8, 2, false, 9, 2), "partial sums that nothing holds");
    REQUIRE(!wide_units_hold(10, 10, 1, false, 2, 2) && !wide_units_hold(10, 0, 3, true, 8, 2) && !wide_units_hold(10, 8, 2, true, 9, 4), "short units");
    REQUIRE(tile_plan(CW_NN, 8, 8, 8, 0, 8, 8, true, true, 0, -1).cfg == -1 && tile_plan(CW_NN, 8, 8, 8, CW_MAX_KSTEPS + 1, 8, 8, true, true, 0, -1).cfg == -1, "bad step counts");
}

void check_refusals() {
    GemmArgs args;
    bool nothing = false;
    const void* tab[1] = {reinterpret_cast<const void*>(256)};
    void* c = reinterpret_cast<void*>(512);
    auto call = [&](int layout, int64_t M, int64_t N, int64_t K, int steps, const void* const* a, int64_t lda, const void* const* b,
                    int64_t ldb, void* C, int64_t ldc, int epi, int dt, int nadd) {
        return gemm_prepare_args(layout, M, N, K, steps, a, lda, b, ldb, nullptr, epi, C, ldc, nullptr, 0, nullptr, nadd, 0, nullptr, 0, dt,
                                 &args, &nothing);
    };
    REQUIRE(call(9, 8, 8, 8, 1, tab, 8, tab, 8, c, 8, 0, 0, 0) == CW_ERR_INVALID, "bad layout accepted");
    REQUIRE(call(0, 8, 8, 8, 1, tab, 8, tab, 8, c, 8, 9, 0, 0) == CW_ERR_INVALID, "bad epilogue accepted");
    REQUIRE(call(0, 8, 8, 8, 1, tab, 8, tab, 8, c, 8, 0, 7, 0) == CW_ERR_INVALID, "bad dtype accepted");
    REQUIRE(call(0, -1, 8, 8, 1, tab, 8, tab, 8, c, 8, 0, 0, 0) == CW_ERR_INVALID, "negative M accepted");
    REQUIRE(call(0, (int64_t)1 << 31, 8, 8, 1, tab, 8, tab, 8, c, 8, 0, 0, 0) == CW_ERR_INVALID, "M beyond int32 accepted");
    REQUIRE(call(0, 8, 8, 8, 99, tab, 8, tab, 8, c, 8, 0, 0, 0) == CW_ERR_INVALID, "99 steps accepted");
    REQUIRE(call(0, 8, 8, 8, 1, tab, 8, tab, 8, c, 8, 0, 0, 99) == CW_ERR_INVALID, "99 addends accepted");
    REQUIRE(call(0, 8, 8, 8, 1, nullptr, 8, tab, 8, c, 8, 0, 0, 0) == CW_ERR_INVALID, "NULL operand table accepted");
    REQUIRE(call(0, 8, 8, 8, 1, tab, 7, tab, 8, c, 8, 0, 0, 0) == CW_ERR_INVALID, "lda < K accepted");
    REQUIRE(call(0, 8, 8, 8, 1, tab, 8, tab, 8, nullptr, 8, 0, 0, 0) == CW_ERR_INVALID, "NULL C accepted");
    REQUIRE(call(0, 8, 8, 8, 1, tab, 8, tab, 8, c, 7, 0, 0, 0) == CW_ERR_INVALID, "ldc < N accepted");
    REQUIRE(call(0, 0, 8, 8, 1, tab, 8, tab, 8, nullptr, 8, 0, 0, 0) == CW_OK && nothing, "empty output must be a no-op");
    REQUIRE(gemm_workspace_bytes(CW_TN, 2048, 2048, 8192, 2, CW_BF16) == (int64_t)4 * 2048 * 2048 * 4, "split-k scratch of the weight gradient");
    REQUIRE(gemm_workspace_bytes(CW_TN, 2048, 2048, 8192, 2, CW_F32) == 0, "fp32 asks for no scratch");
    REQUIRE(gemm_workspace_bytes(CW_NN, -5, 2048, 8192, 2, CW_BF16) == 0 && gemm_workspace_bytes(7, 8, 8, 8, 1, CW_BF16) == 0, "bad arguments ask for no scratch");
    REQUIRE(gemm_workspace_bytes(CW_NN, (int64_t)1 << 40, (int64_t)1 << 40, 8192, 2, CW_BF16) == 0, "huge shapes ask for no scratch");
    g_checked += 16;
}

void sweep_colsum() {
    const int64_t ms[] = {1, 2, 15, 16, 17, 63, 64, 65, 300, 4095, 4096, 8192, 16384, 1 << 20, (int64_t)1 << 31};
    const int64_t ns[] = {1, 7, 8, 64, 512, 520, 2048, 8192, 8201, 50272, 1 << 20};
    for (int64_t M : ms)
        for (int64_t N : ns)
            for (int V : {4, 8})
                for (int vec = 0; vec < 2; ++vec) {
                    int64_t slabs = -1, rows = -1;
                    colsum_plan(M, N, V, vec != 0, slabs, rows);
                    ++g_checked;
                    REQUIRE(slabs >= 1 && rows >= 1, "colsum_plan(%lld, %lld): slabs %lld rows %lld", (long long)M, (long long)N, (long long)slabs, (long long)rows);
                    REQUIRE((slabs - 1) * rows < M && slabs * rows >= M, "slabs do not cover the rows exactly once (M=%lld N=%lld)", (long long)M, (long long)N);
                    if (vec) REQUIRE(slabs <= kColMaxSlabs, "more partial rows than the workspace bound");
                    else REQUIRE(slabs == (M + kColGenericSlabRows - 1) / kColGenericSlabRows, "generic slabs");
                }
}

}  // namespace

int main() {
    check_refusals();
    sweep_colsum();
    sweep_gemm();
    sweep_tile_plan();
    printf("ok %ld routes small_ring=%ld ring=%ld ring_then_small=%ld split_k=%ld other=%ld\n", g_checked, g_routes[0],
           g_routes[1], g_routes[2], g_routes[3], g_routes[4]);
    return 0;
}
