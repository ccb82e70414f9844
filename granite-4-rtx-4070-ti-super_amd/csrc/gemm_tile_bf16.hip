// gemm_tile_bf16.hip - the tile GEMM (gemm_tile.h) for bf16 activations: its
// configurations and the choice between them.
#include "gemm_tile.h"

namespace g4 {
namespace {

// Rows x weight rows of a tile, and the costs fitted to 76 shapes (N x K of
// q|k|v 6144 x 4096, O 4096 x 4096, down 4096 x 12800, one of gate|up 12800 x
// 4096, 17 to 8192 rows, us, the weights in the cache; the choice by them is
// within 8 %, in the mean 0.3 %, of the best of these). Measured against the 128 x
// 128 kernel of gemm.hip, us, the operands rotated through 700 MB: q|k|v 64 rows
// 54.4 -> 15.5, 512 rows 56.2 -> 33.9, 1000 rows 69.0 -> 49.0, 8192 rows 461 -> 310;
// O 64 rows 55.2 -> 13.3, 512 rows 56.5 -> 29.3, 8192 rows 316 -> 225 (in the cache
// 208: 1.32 PFLOP/s; a library product of 8192^3 on the same card reaches 1.28);
// down 64 rows 160 -> 32.3, 512 rows 165 -> 77.4, 8192 rows 930 -> 622.
// Against the general kernel, at the cheapest tile's shapes, tile / general: 256 x
// 256 in the mean 0.92 (up to 1.05) at K = 384, 0.98 (1.11) at 256; 256 x 128 at once
// 1.00 at 512, 0.97 at 640, in turn 1.05 at 256, 0.98 at 384; 128 x 192 1.20 at 384,
// 0.95 at 512; the smaller ones faster from where they fit (512).
constexpr TileConfig<false, 8, 8, 2, 1, true> k256x256{{75.48f, 24.40f, -18.93f}, {384, 384}};
constexpr TileConfig<false, 8, 4, 3, 1, true> k256x128{{44.77f, 12.50f, -6.99f}, {640, 384}};
constexpr TileConfig<false, 4, 6, 4, 1, true> k128x192{{35.10f, 10.14f, -4.51f}, {512, 512}};
constexpr TileConfig<false, 4, 4, 3, 2, true> k128x128{{22.34f, 11.67f, -7.56f}};
constexpr TileConfig<false, 4, 3, 3, 2, false> k128x96{{19.94f, 7.63f, -2.81f}};
constexpr TileConfig<false, 2, 4, 3, 2, true> k64x128{{15.63f, 7.11f, -4.25f}};
constexpr TileConfig<false, 2, 3, 4, 2, false> k64x96{{13.89f, 4.94f, -1.22f}};
constexpr TileConfig<false, 2, 2, 4, 2, false> k64x64{{11.36f, 3.00f, -0.73f}};
constexpr TileConfig<false, 1, 2, 6, 2, false> k32x64{{8.40f, 2.10f, 0.47f}};
constexpr TileConfig<false, 1, 1, 4, 4, false> k32x32{{6.24f, 1.37f, 1.81f}};

template <int EPI>
unsigned go(const GemmArgs& a) {
  // Tiles of fewer than 128 rows need a K that is a multiple of 256. Without
  // them a small output leaves CUs idle, which a short K does not make up for
  // (tile / general up to one general tile per CU: 1.07 at K = 640, 0.98 at 896).
  if (a.M > kSkinnyMaxM && a.K % 256 != 0 && a.K < 896 && general_tiles(a, false) <= kCUs) return 0;
  return launch_cheapest<EPI>(a, TileCost{}, k256x256, k256x128, k128x192, k128x128, k128x96, k64x128, k64x96, k64x64, k32x64,
                              k32x32);
}

}  // namespace

unsigned launch_gemm_tile_bf16(int epi, const GemmArgs& a) {
  switch (epi) {
    case kEpiBf16: return go<kEpiBf16>(a);
    case kEpiF32: return go<kEpiF32>(a);
    default: return go<kEpiResidual>(a);
  }
}

}  // namespace g4
