// 16-bit block GEMM, tile kernels (gemm_tile.h): one object per element type, orientation and configuration 1 to 4 of
// kTileConfigs (gemm_plan.h), compiled from this file with CW_TILE_E (bf16_t, f16_t), CW_TILE_LAYOUT (NN, NT, TN) and
// CW_TILE_CFG (1 .. 4).
#include "gemm_plan.h"
#include "gemm_tile.h"

namespace cw {

#define CW_TILE_CAT_(e, l, c) gemm_tile_##e##_##l##_##c
#define CW_TILE_CAT(e, l, c) CW_TILE_CAT_(e, l, c)
#define CW_TILE_ENUM_(l) CW_##l
#define CW_TILE_ENUM(l) CW_TILE_ENUM_(l)

int CW_TILE_CAT(CW_TILE_E, CW_TILE_LAYOUT, CW_TILE_CFG)(const TileArgs& args, int epilogue, hipStream_t s) {
    constexpr int layout = CW_TILE_ENUM(CW_TILE_LAYOUT);
    constexpr TileConfig c = kTileConfigs[CW_TILE_CFG];
    return gemm_tile::launch_epi<layout == CW_TN, layout != CW_NT, layout == CW_TN, c.tm, c.tn, c.kb, c.stages, CW_TILE_E>(args, epilogue, s);
}

}  // namespace cw
