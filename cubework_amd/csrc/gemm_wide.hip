// 16-bit block GEMM, the kernel of 8 wavefronts (gemm_wide.h): one object per element type, orientation and tile, compiled from
// this file with CW_TILE_E (bf16_t, f16_t), CW_TILE_LAYOUT (NN, NT, TN) and CW_TILE_CFG: 160, 192, 224, 256 (rows; 256 columns), 128
// (128 x 128, two groups of wavefronts along k), 2128, 2160, 2192 (128, 160, 192 rows; 128 columns).
#include "gemm_wide.h"

namespace cw {

#define CW_WIDE_CAT_(e, l, c) gemm_wide_##e##_##l##_##c
#define CW_WIDE_CAT(e, l, c) CW_WIDE_CAT_(e, l, c)
#define CW_WIDE_ENUM_(l) CW_##l
#define CW_WIDE_ENUM(l) CW_WIDE_ENUM_(l)

int CW_WIDE_CAT(CW_TILE_E, CW_TILE_LAYOUT, CW_TILE_CFG)(const TileArgs& args, int epilogue, hipStream_t s) {
    constexpr int layout = CW_WIDE_ENUM(CW_TILE_LAYOUT);
    constexpr int TM = CW_TILE_CFG % 1000 / 32, TN = CW_TILE_CFG < 2000 ? 4 : 2, KG = CW_TILE_CFG == 128 ? 2 : 1;
    return gemm_wide::launch_epi<layout == CW_TN, layout != CW_NT, layout == CW_TN, TM, TN, KG, CW_TILE_E>(args, epilogue, s);
}

}  // namespace cw
