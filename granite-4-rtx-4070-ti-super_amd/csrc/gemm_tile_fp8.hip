// gemm_tile_fp8.hip - the tile GEMM (gemm_tile.h) for FP8 activations: its
// configurations and the choice between them.
#include "gemm_tile.h"

namespace g4 {
namespace {

// Rows x weight rows of a tile, and the costs fitted to 57 shapes (N x K of
// q|k|v 6144 x 4096, down 4096 x 12800, gate|up 25600 x 4096, 17 to 8192 rows,
// us; the choice by them is within 2 % of the best of these at every one).
// Measured against the 128 x 128 / 128 x 64 kernels of gemm.hip, us: q|k|v 64
// rows 17.4 -> 8.7, 1000 rows 29.8 -> 25.7, 8192 rows 224 -> 164; down 64 rows
// 41.5 -> 18.3, 512 rows 45.3 -> 34.3, 8192 rows 425 -> 320; gate|up 64 rows
// 38.2 -> 24.0, 512 rows 80.6 -> 56.7, 8192 rows 867 -> 667 (2.58 PFLOP/s; a
// library product of 8192^3 on the same card reaches 2.72).
constexpr TileConfig<true, 8, 8, 2, 1, true> k256x256{{34.55f, 20.10f, -11.14f}};
constexpr TileConfig<true, 8, 4, 3, 1, true> k256x128{{20.72f, 9.35f, -2.43f}};
constexpr TileConfig<true, 4, 6, 3, 1, false> k128x192{{16.25f, 12.15f, -7.93f}};
constexpr TileConfig<true, 4, 4, 4, 1, false> k128x128{{12.01f, 6.86f, -1.50f}};
constexpr TileConfig<true, 4, 2, 3, 2, false> k128x64{{8.41f, 5.80f, -2.33f}};
constexpr TileConfig<true, 2, 4, 3, 2, true> k64x128{{9.27f, 5.61f, -1.15f}};
constexpr TileConfig<true, 2, 3, 4, 2, false> k64x96{{7.86f, 4.58f, -1.73f}};
constexpr TileConfig<true, 2, 2, 4, 2, false> k64x64{{6.45f, 3.33f, -0.57f}};
constexpr TileConfig<true, 2, 1, 4, 2, false> k64x32{{4.95f, 1.45f, 1.16f}};

template <int EPI>
unsigned go(const GemmArgs& a) {
  return launch_cheapest<EPI>(a, k256x256, k256x128, k128x192, k128x128, k128x64, k64x128, k64x96, k64x64, k64x32);
}

}  // namespace

unsigned launch_gemm_tile_fp8(int epi, const GemmArgs& a) {
  switch (epi) {
    case kEpiBf16: return go<kEpiBf16>(a);
    case kEpiF32: return go<kEpiF32>(a);
    case kEpiResidual: return go<kEpiResidual>(a);
    default: return launch_cheapest<kEpiSwiglu>(a, k256x256, k256x128, k128x128, k64x128, k64x64);
  }
}

}  // namespace g4
