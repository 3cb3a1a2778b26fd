// 16-bit block GEMM, the kernel of 256-column tiles (gemm_wide.h): one object per element type, orientation and tile height,
// compiled from this file with CW_TILE_E (bf16_t, f16_t), CW_TILE_LAYOUT (NN, NT, TN) and CW_TILE_CFG (160, 192, 224, 256; 128:
// tiles of 128 x 128 with two groups of wavefronts along k).
#include "gemm_wide.h"

namespace cw {

#define CW_WIDE_CAT_(e, l, c) gemm_wide_##e##_##l##_##c
#define CW_WIDE_CAT(e, l, c) CW_WIDE_CAT_(e, l, c)
#define CW_WIDE_ENUM_(l) CW_##l
#define CW_WIDE_ENUM(l) CW_WIDE_ENUM_(l)

int CW_WIDE_CAT(CW_TILE_E, CW_TILE_LAYOUT, CW_TILE_CFG)(const TileArgs& args, int epilogue, hipStream_t s) {
    constexpr int layout = CW_WIDE_ENUM(CW_TILE_LAYOUT);
    return gemm_wide::launch_epi<layout == CW_TN, layout != CW_NT, layout == CW_TN, CW_TILE_CFG / 32, CW_TILE_CFG == 128 ? 2 : 1, CW_TILE_E>(args, epilogue, s);
}

}  // namespace cw
