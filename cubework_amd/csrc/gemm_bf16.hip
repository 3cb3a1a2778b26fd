// bf16 / fp16 block GEMM: choice of kernel and launch (the same for both element types).
//   - the tile kernels (gemm_wide.h, gemm_tile.h) take every shape whose operand rows are 16-byte aligned, and the others after a copy to
//     aligned rows, which the caller's scratch holds. tile_plan (gemm_plan.hip) chooses the tile size and which tiles are
//     cut along k, by a cost model of the launch;
//   - a call with less scratch than that (or none) is planned by gemm_half_plan;
//   - the register-staged kernel (gemm_bf16_kernel.h) takes what is left: unaligned operands without scratch for the copy,
//     and an activation on the weight-gradient orientation.
// CW_GEMM_IMPL=staged in the environment forces the register-staged kernel, CW_GEMM_IMPL=onelaunch one launch per product.
#include <cstdlib>
#include <cstring>

#include "gemm_bf16_kernel.h"
#include "gemm_plan.h"
#include "gemm_tile.h"

namespace cw {

#define CW_TILE_CFGS(e, l) {gemm_tile_##e##_##l##_1, gemm_tile_##e##_##l##_2, gemm_tile_##e##_##l##_3, gemm_tile_##e##_##l##_4}
#define CW_WIDE_ROWS(e, l) {gemm_wide_##e##_##l##_128, gemm_wide_##e##_##l##_160, gemm_wide_##e##_##l##_192, gemm_wide_##e##_##l##_224, gemm_wide_##e##_##l##_256}
#define CW_NARROW_ROWS(e, l) {gemm_wide_##e##_##l##_2128, gemm_wide_##e##_##l##_2160, gemm_wide_##e##_##l##_2192}
#define CW_NARROW_DECL(e, l)                                            \
    int gemm_wide_##e##_##l##_2128(const TileArgs&, int, hipStream_t);  \
    int gemm_wide_##e##_##l##_2160(const TileArgs&, int, hipStream_t);  \
    int gemm_wide_##e##_##l##_2192(const TileArgs&, int, hipStream_t);
#define CW_TILE_DECL(e, l)                                              \
    int gemm_tile_##e##_##l##_1(const TileArgs&, int, hipStream_t);     \
    int gemm_tile_##e##_##l##_2(const TileArgs&, int, hipStream_t);     \
    int gemm_tile_##e##_##l##_3(const TileArgs&, int, hipStream_t);     \
    int gemm_tile_##e##_##l##_4(const TileArgs&, int, hipStream_t);     \
    int gemm_wide_##e##_##l##_128(const TileArgs&, int, hipStream_t);   \
    int gemm_wide_##e##_##l##_160(const TileArgs&, int, hipStream_t);   \
    int gemm_wide_##e##_##l##_192(const TileArgs&, int, hipStream_t);   \
    int gemm_wide_##e##_##l##_224(const TileArgs&, int, hipStream_t);   \
    int gemm_wide_##e##_##l##_256(const TileArgs&, int, hipStream_t);
CW_TILE_DECL(bf16_t, NN)
CW_TILE_DECL(bf16_t, NT)
CW_TILE_DECL(bf16_t, TN)
CW_TILE_DECL(f16_t, NN)
CW_TILE_DECL(f16_t, NT)
CW_TILE_DECL(f16_t, TN)
CW_NARROW_DECL(bf16_t, NN)
CW_NARROW_DECL(bf16_t, NT)
CW_NARROW_DECL(f16_t, NN)
CW_NARROW_DECL(f16_t, NT)

using TileLaunch = int (*)(const TileArgs&, int, hipStream_t);
static constexpr TileLaunch kTileLaunch[2][3][4] = {
    {CW_TILE_CFGS(bf16_t, NN), CW_TILE_CFGS(bf16_t, NT), CW_TILE_CFGS(bf16_t, TN)},
    {CW_TILE_CFGS(f16_t, NN), CW_TILE_CFGS(f16_t, NT), CW_TILE_CFGS(f16_t, TN)},
};
static constexpr TileLaunch kWideLaunch[2][3][5] = {
    {CW_WIDE_ROWS(bf16_t, NN), CW_WIDE_ROWS(bf16_t, NT), CW_WIDE_ROWS(bf16_t, TN)},
    {CW_WIDE_ROWS(f16_t, NN), CW_WIDE_ROWS(f16_t, NT), CW_WIDE_ROWS(f16_t, TN)},
};
static constexpr TileLaunch kNarrowLaunch[2][2][3] = {
    {CW_NARROW_ROWS(bf16_t, NN), CW_NARROW_ROWS(bf16_t, NT)},
    {CW_NARROW_ROWS(f16_t, NN), CW_NARROW_ROWS(f16_t, NT)},
};
static_assert(CW_NN == 0 && CW_NT == 1 && CW_TN == 2, "kTileLaunch is indexed by layout");

// rows x cols elements at `src` (any alignment, row pitch ld) to rows of `out` (pitch ldo, a multiple of 8): one thread per 16
// bytes of output. Memory-bound: one read and one write of the operand (global accesses need no alignment).
__global__ __launch_bounds__(256) void pack_rows_kernel(const uint16_t* __restrict__ src, int64_t ld, int64_t rows, int64_t cols,
                                                        uint16_t* __restrict__ out, int64_t ldo) {
    const int64_t per_row = ldo / 8, idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= rows * per_row) return;
    const int64_t r = idx / per_row, c = (idx - r * per_row) * 8;
    const uint16_t* p = src + r * ld + c;
    raw16_t v = {0u, 0u, 0u, 0u};
    if (c + 8 <= cols) {
        __builtin_memcpy(&v, p, 16);
    } else {
        uint32_t w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int e = 0; e < 7; ++e)
            if (c + e < cols) w[e >> 1] |= (uint32_t)p[e] << ((e & 1) * 16);
        v = raw16_t{w[0], w[1], w[2], w[3]};
    }
    *reinterpret_cast<raw16_t*>(out + r * ldo + c) = v;
}

static int pack_rows(const void* const* src, int n, int64_t ld, int64_t rows, int64_t cols, char* out, int64_t ldo, const void** packed,
                     hipStream_t s) {
    const int64_t chunks = rows * (ldo / 8);  // fewer than 2^32 by plan
    for (int i = 0; i < n; ++i) {
        packed[i] = out + (int64_t)i * rows * ldo * 2;
        hipLaunchKernelGGL(pack_rows_kernel, dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0, s, (const uint16_t*)src[i], ld, rows, cols,
                           (uint16_t*)packed[i], ldo);
        if (const int rc = check_launch("pack_rows_kernel"); rc != CW_OK) return rc;
    }
    return CW_OK;
}

// One instantiation serves CW_EPI_NONE and CW_EPI_BIAS: without an epilogue there is no bias, whatever the caller passes.
static TileArgs to_tile_args(const GemmArgs& g, int epilogue) {
    TileArgs a;
    memcpy(a.A, g.A, sizeof(a.A));
    memcpy(a.B, g.B, sizeof(a.B));
    memcpy(a.addend, g.addend, sizeof(a.addend));
    a.bias = epilogue == CW_EPI_NONE ? nullptr : g.bias;
    a.C = g.C; a.preact = g.preact;
    a.lda = g.lda; a.ldb = g.ldb; a.ldc = g.ldc; a.ldp = g.ldp; a.ldadd = g.ldadd;
    a.M = g.M; a.N = g.N; a.K = g.K; a.n_steps = g.n_steps; a.n_addends = g.n_addends;
    a.vec_out = g.vec_c && (g.preact == nullptr || g.vec_p);
    a.full = 0;
    a.slices = 1;
    a.rotate = 0;
    a.partial = nullptr;
    return a;
}

static int tile_launch(const GemmArgs& g, const TilePlan& plan, int layout, int epilogue, bool f16, hipStream_t s) {
    TileArgs a = to_tile_args(g, epilogue);
    char* ws = reinterpret_cast<char*>(g.workspace);
    if (plan.pack_a) {
        const bool tn = layout == CW_TN;
        if (const int rc = pack_rows(g.A, g.n_steps, g.lda, tn ? g.K : g.M, tn ? g.M : g.K, ws, plan.lda, a.A, s); rc != CW_OK) return rc;
    }
    if (plan.pack_b) {
        const bool nt = layout == CW_NT;
        if (const int rc = pack_rows(g.B, g.n_steps, g.ldb, nt ? g.N : g.K, nt ? g.K : g.N, ws + plan.pack_a_bytes, plan.ldb, a.B, s); rc != CW_OK)
            return rc;
    }
    if (plan.pack_add_bytes > 0) {
        const int64_t ld = ((int64_t)g.N + 7) / 8 * 8;
        if (const int rc = pack_rows(g.addend, g.n_addends, g.ldadd, g.M, g.N, ws + plan.pack_a_bytes + plan.pack_b_bytes, ld, a.addend, s); rc != CW_OK)
            return rc;
        a.ldadd = ld;
    }
    a.lda = plan.lda;
    a.ldb = plan.ldb;
    a.full = plan.full;
    a.slices = plan.slices;
    a.rotate = plan.rotate ? 1 : 0;
    a.partial = reinterpret_cast<float*>(ws + plan.pack_a_bytes + plan.pack_b_bytes + plan.pack_add_bytes);
    if (plan.cfg == 0 || plan.cfg == kPairedConfig) return kWideLaunch[f16 ? 1 : 0][layout][(plan.rows - 128) / 32](a, epilogue, s);
    if (plan.cfg >= kNarrowConfig) return kNarrowLaunch[f16 ? 1 : 0][layout][(plan.rows - 128) / 32](a, epilogue, s);
    return kTileLaunch[f16 ? 1 : 0][layout][plan.cfg - 1](a, epilogue, s);
}

// A plan of one configuration without scratch for operand copies (slices > 1: every tile sliced, partial sums in g.workspace).
static TilePlan tile_plan_of(const GemmArgs& g, int cfg, int slices = 1) {
    TilePlan p = {};
    const int bm = 64 * kTileConfigs[cfg].tm, bn = 64 * kTileConfigs[cfg].tn;
    p.cfg = cfg;
    p.rows = cfg == 0 ? wide_rows(g.M) : bm;
    p.tiles = (int64_t)((g.M + bm - 1) / bm) * ((g.N + bn - 1) / bn);
    p.full = slices > 1 ? 0 : (int)p.tiles;
    p.slices = slices;
    p.rotate = slices == 1 && cfg == 0 && g.M % 256 == 0 && g.N % 256 == 0;
    p.lda = g.lda;
    p.ldb = g.ldb;
    return p;
}

static bool dma_kernel_enabled() {
    static const bool enabled = [] {
        const char* v = std::getenv("CW_GEMM_IMPL");
        return !(v != nullptr && std::strcmp(v, "staged") == 0);
    }();
    return enabled;
}

// CW_GEMM_IMPL=onelaunch keeps a product whose last round of tiles is mostly empty in one launch (A/B measurements).
static bool strip_split_enabled() {
    static const bool enabled = [] {
        const char* v = std::getenv("CW_GEMM_IMPL");
        return !(v != nullptr && std::strcmp(v, "onelaunch") == 0);
    }();
    return enabled;
}

static int staged_launch(const GemmArgs& a, int layout, int epilogue, bool big, bool f16, hipStream_t s) {
    switch (layout) {
        case CW_NN: return f16 ? gemm_f16_launch_nn(a, epilogue, big, s) : gemm_bf16_launch_nn(a, epilogue, big, s);
        case CW_NT: return f16 ? gemm_f16_launch_nt(a, epilogue, big, s) : gemm_bf16_launch_nt(a, epilogue, big, s);
        case CW_TN: return f16 ? gemm_f16_launch_tn(a, epilogue, big, s) : gemm_bf16_launch_tn(a, epilogue, big, s);
        default: return fail(CW_ERR_INVALID, "cw_gemm_ksteps: bad layout %d", layout);
    }
}

// f16: the operands, bias, addends and outputs are IEEE half instead of bfloat16; everything else is shared.
int gemm_half_launch(const GemmArgs& args, int layout, int epilogue, bool f16, hipStream_t s) {
    const bool tiles_ok = dma_kernel_enabled() && args.n_steps > 0 &&
                          (layout != CW_TN || epilogue == CW_EPI_NONE || epilogue == CW_EPI_BIAS);
    const bool one_launch = !strip_split_enabled();
    const int pack_addends = args.vec_add ? 0 : args.n_addends;
    if (tiles_ok) {
        const int64_t scratch = aligned16(args.workspace) ? args.workspace_bytes : 0;
        const TilePlan want = tile_plan(layout, args.M, args.N, args.K, args.n_steps, args.lda, args.ldb, args.vec_a != 0, args.vec_b != 0,
                                        pack_addends, one_launch ? 0 : -1);
        if (want.cfg >= 0 && want.scratch() <= scratch) return tile_launch(args, want, layout, epilogue, f16, s);
    }
    const GemmPlan plan = gemm_half_plan(args, layout, tiles_ok, strip_split_enabled());
    switch (plan.route) {
        case kRouteSmallRing: return tile_launch(args, tile_plan_of(args, 2), layout, epilogue, f16, s);
        case kRouteRing: return tile_launch(args, tile_plan_of(args, wide_takes(args.K, args.n_steps) ? 0 : 1), layout, epilogue, f16, s);
        case kRouteRingThenSmall: {
            const int head = wide_takes(args.K, args.n_steps) ? 0 : 1;
            if (const int rc = tile_launch(plan.head, tile_plan_of(plan.head, head), layout, epilogue, f16, s); rc != CW_OK) return rc;
            return tile_launch(plan.tail, tile_plan_of(plan.tail, 2), layout, epilogue, f16, s);
        }
        case kRouteSplitK: return tile_launch(args, tile_plan_of(args, 0, plan.slices), layout, epilogue, f16, s);
        default: break;
    }
    if (tiles_ok) {
        const TilePlan fits = tile_plan(layout, args.M, args.N, args.K, args.n_steps, args.lda, args.ldb, args.vec_a != 0, args.vec_b != 0,
                                        pack_addends, aligned16(args.workspace) ? args.workspace_bytes : 0);
        if (fits.cfg >= 0) return tile_launch(args, fits, layout, epilogue, f16, s);
    }
    return staged_launch(args, layout, epilogue, plan.big, f16, s);
}

}  // namespace cw
