// gemm_tile_fp8.hip - the tile GEMM (gemm_tile.h) for FP8 activations: its
// configurations and the choice between them.
#include "gemm_tile.h"

namespace g4 {
namespace {

// Rows x weight rows of a tile, and the costs fitted to 57 shapes (N x K of
// q|k|v 6144 x 4096, down 4096 x 12800, gate|up 25600 x 4096, 17 to 8192 rows,
// us, the weights in the cache; the choice by them is within 2 % of the best of
// these at every one). Measured against the 128 x 128 / 128 x 64 kernels of
// gemm.hip, us, the operands rotated through 700 MB: q|k|v 64 rows 16.3 -> 12.2,
// 1000 rows 39.1 -> 30.3, 8192 rows 231 -> 174; down 64 rows 39.6 -> 28.1, 512 rows
// 49.7 -> 48.6, 1000 rows 94.5 -> 65.4, 8192 rows 436 -> 341; gate|up 64 rows 38.0 ->
// 27.2, 512 rows 79.3 -> 62.0, 8192 rows 890 -> 708 (in the cache 667: 2.58 PFLOP/s;
// a library product of 8192^3 on the same card reaches 2.72).
// Against the general kernels, at the cheapest tile's shapes, tile / general:
// 256 x 256 in the mean 0.93 (up to 1.08) at K = 1024, 0.96 (1.11) at 768; 256 x 128
// at once 1.00-1.06 at 3584, 0.97-1.03 at 4096, in turn 1.00 at 2560, 0.96 at 3072;
// 128 x 192 1.00 at 1792, 0.94 at 2048; 128 x 128 1.07 at 1280, 0.95 at 1536; 64 x 128
// 1.06 at 2048, 0.93 at 2560; the smaller ones faster from where they fit (1024).
// In turns by the times: q|k|v 2561 rows (4 rounds of 128 x 128 against 2 of two a
// CU) 89.6 -> 68.8 us; gate|up 769 to 896 rows (2 rounds of 256 x 256 against 3) 105
// -> 97, 600 rows 78.5 -> 75.4.
constexpr TileConfig<true, 8, 8, 2, 1, true> k256x256{{34.55f, 20.10f, -11.14f}, {1024, 1024, {43.9f, 7.36f, 3.25f}}};
constexpr TileConfig<true, 8, 4, 3, 1, true> k256x128{{20.72f, 9.35f, -2.43f}, {4096, 3072, {25.25f, 5.24f, 2.25f}}};
constexpr TileConfig<true, 4, 6, 3, 1, false> k128x192{{16.25f, 12.15f, -7.93f}, {2048, 2048, {19.48f, 4.67f, 1.76f}}};
constexpr TileConfig<true, 4, 4, 4, 1, false> k128x128{{12.01f, 6.86f, -1.50f}, {1536, 1536, {13.97f, 3.04f, 1.18f}}};
constexpr TileConfig<true, 4, 2, 3, 2, false> k128x64{{8.41f, 5.80f, -2.33f}};
constexpr TileConfig<true, 2, 4, 3, 2, true> k64x128{{9.27f, 5.61f, -1.15f}, {2560, 2560}};
constexpr TileConfig<true, 2, 3, 4, 2, false> k64x96{{7.86f, 4.58f, -1.73f}};
constexpr TileConfig<true, 2, 2, 4, 2, false> k64x64{{6.45f, 3.33f, -0.57f}};
constexpr TileConfig<true, 2, 1, 4, 2, false> k64x32{{4.95f, 1.45f, 1.16f}};
constexpr TileCost kGeneral{29.20f, 3.99f, 0.02f};  // a round of 512 tiles
// SwiGLU, whose general kernel has 128-row tiles of 64 columns only: 256 x 256 0.97
// at 768, 1.03 at 512; the smaller ones faster from where they fit. Gate and up
// rows in pairs need an even FN and whole loads of each: not 192, 96 or 32
// columns; 128 x 64 was not measured for it.
constexpr TileConfig<true, 8, 8, 2, 1, true> kGlu256x256{k256x256.cost, {768, 768, {44.14f, 7.63f, 3.00f}}};
constexpr TileConfig<true, 8, 4, 3, 1, true> kGlu256x128{k256x128.cost, {4096, 3072, {25.38f, 4.54f, 2.40f}}};
constexpr TileConfig<true, 4, 4, 4, 1, false> kGlu128x128{k128x128.cost, {0, 0, {15.84f, 1.68f, 2.69f}}};
constexpr TileConfig<true, 2, 4, 3, 2, true> kGlu64x128{k64x128.cost};
constexpr TileCost kGluGeneral{30.49f, 2.82f, 1.05f};

template <int EPI>
unsigned go(const GemmArgs& a) {
  // Tiles of fewer than 128 rows need a K that is a multiple of 512. Without
  // them, the general kernel's 128 x 64 tiles give a small output more
  // workgroups: one per CU at most, K = 1280 to 4352, tile / general 1.02-1.10 in
  // the mean; two, 1.00 at 1792, 0.97 (up to 1.10) at 2304, 0.91 at 3328.
  const long long wide = general_tiles(a, false), narrow = (a.M + 127) / 128 * ((a.N + 63LL) / 64);
  if (a.M > kSkinnyMaxM && a.K % 512 != 0 && wide < kCUs && (narrow <= kCUs || a.K < 3072)) return 0;
  return launch_cheapest<EPI>(a, kGeneral, k256x256, k256x128, k128x192, k128x128, k128x64, k64x128, k64x96, k64x64,
                              k64x32);
}

}  // namespace

unsigned launch_gemm_tile_fp8(int epi, const GemmArgs& a) {
  switch (epi) {
    case kEpiBf16: return go<kEpiBf16>(a);
    case kEpiF32: return go<kEpiF32>(a);
    case kEpiResidual: return go<kEpiResidual>(a);
    default: return launch_cheapest<kEpiSwiglu>(a, kGluGeneral, kGlu256x256, kGlu256x128, kGlu128x128, kGlu64x128, k64x64);
  }
}

}  // namespace g4
