// gemm_common.h - arguments, epilogue kinds and fragment helpers shared by the
// GEMM kernels (gemm.hip, gemm_tile.h).
#ifndef G4_GEMM_COMMON_H
#define G4_GEMM_COMMON_H

#include "g4_common.h"
#include "g4_hw.h"
#include "g4_math.h"
#include "granite4_layerops.h"

namespace g4 {

enum : int {
  kEpiBf16 = GRANITE4_GEMM_BF16,
  kEpiF32 = GRANITE4_GEMM_F32,
  kEpiResidual = GRANITE4_GEMM_RESIDUAL,
  kEpiSwiglu = 3
};

typedef int v8i __attribute__((ext_vector_type(8)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

struct GemmArgs {
  const uint8_t* A;
  int lda;
  const float* a_scale;  // device: the activation's per-tensor scale
  const uint8_t* W;
  int M, N, K;  // N: weight rows (swiglu: 2I)
  int I;        // swiglu: act columns
  Granite4GemmEpilogue ep;
  float* partials;  // swiglu: [gridDim.x] max |act|
  int mt, nt;       // tile counts along M and N
  bool vec_out;     // 16-byte output rows (pitch and width multiples of 8)
  bool xcd_order;   // tiles renumbered per XCD (xcd_tile0)
  bool n_major;     // tile kernel: consecutive tiles are one row of them, not one column
  // Skinny kBf16 only (gemm_rows_split): when seg_out[0] is set, column n of
  // segment s (ep.seg1 / ep.seg2 bounds) goes to seg_out[s][m * seg_ld[s] +
  // n - start of s] instead of ep.out_bf16.
  uint16_t* seg_out[3];
  int seg_ld[3];
};

// Workgroups are handed to the 8 XCDs round-robin by id (id % 8), each XCD
// with its own L2. The first tile of workgroup b is renumbered so that
// consecutive tile numbers - the M tiles of one weight column, which read the
// same W rows - run on one XCD and share its L2 instead of each XCD fetching
// the column: b -> (b % 8) * (g / 8) + b / 8 over the first 8 * floor(g / 8)
// workgroups (g the grid), the identity on the rest. Tile t + g keeps the
// same XCD as tile t.
__device__ __forceinline__ int xcd_tile0(bool on) {
  const int b = blockIdx.x, g = gridDim.x, full = g & ~7;
  if (!on || b >= full) return b;
  return (b & 7) * (full >> 3) + (b >> 3);
}

// Whether XCD-ordered tiles (xcd_tile0) cut the L2 fills of a launch of g
// workgroups over mt M tiles. Per round each XCD runs g / 8 tiles; the A rows
// and W rows it fetches grow with the block of tiles it covers, bm M tiles x
// bn N tiles, as bm + bn. XCD order gives each XCD whole columns, bm = mt
// (up to g / 8); the plain order gives it every 8th tile: one M tile (mt <= 8)
// or mt / 8 of them, spread over g / 8 or g / mt columns. Measured: T = 512
// gate|up 88 -> 77 us with XCD order (4 x 16 against 1 x 64), T = 8192 the
// plain order's 8 x 8 beats XCD order's 64 x 1 by 14-17 %.
inline bool gemm_xcd_order(int mt, unsigned g) {
  if (g < 16) return false;
  const long long per = g / 8;
  const long long xbm = mt < per ? mt : per, xbn = (per + mt - 1) / mt;
  const long long pbm = mt <= 8 ? 1 : mt / 8, pbn = mt <= 8 ? per : (g + mt - 1) / mt;
  return xbm + xbn < pbm + pbn;
}

// Whether the tile kernel, where gemm_xcd_order keeps the plain order, numbers
// its tiles along N (consecutive tiles share their A rows) and gives each XCD
// consecutive ones. In the plain order an XCD runs every 8th tile of a column of
// mt: mt / 8 M tiles only where 8 divides mt, all of them where mt is odd, as it
// often is with 256-row tiles, and every XCD then reads all of A. Along N it covers
// g / 8 tiles of a row and the next ones. Taken where that block is at most 4/5 of
// the plain order's. FP8, us, the operands from memory: N x K of 1024 x 4096, 6337
// rows 40 -> 29 (general kernel 31), 7936 rows 47 -> 32 (35); 3072 x 4096, 7936 rows
// 129 -> 91 (107); 6144 x 4096, 6200 rows 187 -> 153; bf16 4096 x 12800, 4900 rows 650 ->
// 501. A block nearly as large is no gain: 25600 x 4096 0.99-1.12.
inline bool gemm_n_major(int mt, int nt, unsigned g) {
  if (g < 16) return false;
  const long long per = g / 8, cols = (static_cast<long long>(g) + mt - 1) / mt;
  const long long every = mt % 8 == 0 ? mt / 8 : mt % 4 == 0 ? mt / 4 : mt % 2 == 0 ? mt / 2 : mt;
  const long long plain = (every < per ? every : per) + (cols < per ? cols : per);
  const long long along = (per + nt - 1) / nt + (nt < per ? nt : per);
  return 5 * along <= 4 * plain;
}

__device__ __forceinline__ float epi_scale(const Granite4GemmEpilogue& ep, int n) {
  return n < ep.seg1 ? ep.scale0 : (n < ep.seg2 ? ep.scale1 : ep.scale2);
}

__device__ __forceinline__ v8i frag_of(const v4u& x, const v4u& y) {
  v8i f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[i] = static_cast<int>(x[i]);
    f[i + 4] = static_cast<int>(y[i]);
  }
  return f;
}

// Two bf16 RNE conversions in one v_cvt_pk_bf16_f32 (equal to the integer
// rounding for every non-NaN value).
__device__ __forceinline__ uint32_t pack_bf16_rne(float lo, float hi) { return pack_bf16_hw(lo, hi); }

typedef __bf16 bf16x8_g __attribute__((ext_vector_type(8)));

constexpr int kSkinnyMaxM = 16;  // rows of the skinny kernel at most

// The LDS-staged tile kernels (gemm_tile.h): choose a tile for the shape and
// launch it. epi: one of the kinds above (bf16 A: not kEpiSwiglu). Returns the
// grid (swiglu: the number of partials written), or 0, launching nothing, where
// no tile takes the arguments (K not a multiple of 256 FP8 / 128 bf16 elements,
// pitches beyond 32-bit tile offsets) or, above kSkinnyMaxM rows, the general
// kernels are the faster ones (short K).
unsigned launch_gemm_tile_fp8(int epi, const GemmArgs& a);
unsigned launch_gemm_tile_bf16(int epi, const GemmArgs& a);

}  // namespace g4

#endif  // G4_GEMM_COMMON_H
