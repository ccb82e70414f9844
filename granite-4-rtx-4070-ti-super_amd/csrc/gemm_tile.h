// gemm_tile.h - the LDS-staged GEMM kernel of everything above the skinny form.
//
// A workgroup of KS x 4 waves owns BM rows x BN weight rows, its 4 waves of a
// K group in 2 x 2, each wave (16 FM) x (16 FN) outputs. K advances one step
// of 128 A bytes per row (128 elements FP8, 64 bf16) through a ring of S LDS
// stages filled by direct-to-LDS loads (16-byte chunks XOR-swizzled by row).
// With KS K groups, group g runs steps [g, g + 1) K / KS through a ring of its
// own, and the groups' partial sums meet in LDS at the end.
//
// What bounds a tile is the LDS: a wave reads 16 (FM + FN) rows per step for
// 256 FM FN outputs, 64 x 64 outputs per wave taking as many LDS clocks as
// matrix clocks and 128 x 128 half as many. So the largest tile gives each of
// 4 waves 128 x 128 outputs: 256 accumulators in AGPRs, one wave per SIMD,
// which no other wave covers, so the wave's own reads must run under its own
// MFMAs. Two forms of that:
//
//   quadrants (QUAD): the wave's outputs are four quadrants (A half, W half).
//     The step walks them in an order that snakes through the halves, so that
//     each needs one new operand half, read from LDS under the MFMAs of the
//     quadrant before. One register set per half.
//   flat: a whole step's fragments are read during the step before, into the
//     other of two register sets: for small wave tiles, whose quadrants have
//     too few MFMAs to cover the LDS latency.
//
// One barrier per step: it proves the next stage landed for every wave and
// frees the stage that every wave has read.
//
// With one K group the ring runs on across tiles: the last S steps of a tile
// load the first stages of the workgroup's next tile, so the epilogue (through an LDS region of its own, no
// barrier) has the next tile's loads in flight and no tile but the first
// waits for memory. Measured with a drained ring instead: about 20 us per
// 256 x 256 tile outside the K loop, T=8192 O 225 us, gate|up FP8 666-684 us.
//
// Fragments: the weight row is the MFMA's A operand and the activation its B
// operand, so a lane ends up with four consecutive output columns of one row.
// Lane l holds row l % 16 of each 16-row block, bytes 32 (l / 16) .. + 31 of
// the 128-byte A row: for FP8 the 16x16x128 instruction's operand, for bf16 A
// two 16x16x32 operands (elements 0..7 and 8..15 of the lane's 16), whose
// weights are the 16 bytes at 16 (l / 16) of the 64-byte W row, converted as
// they are used (exact: an e4m3 value has at most four significant bits). Both
// operands take the same k assignment, so each MFMA sums products of equal k.
#ifndef G4_GEMM_TILE_H
#define G4_GEMM_TILE_H

#include "gemm_common.h"

#include <type_traits>

namespace g4 {
namespace {

// Shape of a tile configuration. FM, FN: a wave's 16-row fragments of A and W.
template <bool F8, int FM, int FN, int S, int KS>
struct TileShape {
  static constexpr int kBM = 32 * FM, kBN = 32 * FN;
  static constexpr int kARow = 128;            // A bytes per row and step
  static constexpr int kWRow = F8 ? 128 : 64;  // W bytes per row and step
  static constexpr int kKb = F8 ? 128 : 64;    // k elements per step
  static constexpr int kABytes = kBM * kARow, kWBytes = kBN * kWRow;
  static constexpr int kStage = kABytes + kWBytes;
  static constexpr int kALoads = kABytes / 4096;                                    // per thread and step
  static constexpr int kWLoads = (kWBytes + 4095) / 4096;
  static constexpr int kLoads = kALoads + kWLoads;
  static constexpr int kWv = F8 ? 2 : 1;       // 16-byte reads per weight fragment
  static constexpr bool kRoll = KS == 1;       // the ring runs on across tiles
  static constexpr int kRing = KS * S * kStage;
  // Epilogue staging: 16 rows x the wave's columns in f32 per wave; beside the
  // ring where it rolls on, else in it (after the K groups' hand-over).
  static constexpr int epi_bytes(bool glu) { return KS * 4 * 64 * (glu ? 8 : 16) * FN; }
  static constexpr int swap_bytes() { return (KS - 1) * 4096 * FM * FN; }
  static constexpr int lds_bytes(bool glu) {
    return kRoll ? kRing + epi_bytes(glu)
                 : (kRing > swap_bytes() + epi_bytes(glu) ? kRing : swap_bytes() + epi_bytes(glu));
  }
};

#ifdef __HIP_DEVICE_COMPILE__
typedef __attribute__((address_space(3))) void* tile_lds_ptr;

// LDS byte address of a pointer into the workgroup's LDS.
__device__ __forceinline__ uint32_t tile_lds_addr(const uint8_t* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((tile_lds_ptr)(p)));
}
// 16-byte LDS read issued as assembly: the compiler's own wait would cover
// every direct-to-LDS load in flight. The value is used only after a
// lgkmcnt(0) wait that it then passes through (`landed`), in the same
// iteration of every loop.
__device__ __forceinline__ v4u tile_read16(uint32_t addr, int offset) {
  v4u v;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "i"(offset) : "memory");
  return v;
}
__device__ __forceinline__ void tile_reads_wait() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
template <int N>
__device__ __forceinline__ void tile_vm_wait() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// acc += w . a, in place in the accumulator registers. Written as assembly:
// with the builtin the compiler rotates the 256 accumulators of the largest
// tile through copies and spills.
__device__ __forceinline__ void tile_mfma(v4f& acc, const v8i& w, const v8i& a) {
  asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0" : "+a"(acc) : "v"(w), "v"(a));
}
__device__ __forceinline__ void tile_mfma(v4f& acc, const bf16x8_g& w, const v4u& a) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(w), "v"(a));
}
// An accumulator's value, read where it is used: left to the compiler, all
// of a tile's reads move ahead of the epilogue and spill.
__device__ __forceinline__ float tile_acc(float acc) {
  float v;
  asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(acc));
  return v;
}
__device__ __forceinline__ v4f tile_acc(const v4f& acc) {
  return v4f{tile_acc(acc[0]), tile_acc(acc[1]), tile_acc(acc[2]), tile_acc(acc[3])};
}
// x + y, added where it is used: as a loop invariant, each load's offset would
// be kept in a register of its own, and spill.
__device__ __forceinline__ uint32_t tile_add(uint32_t x, uint32_t y) {
  uint32_t v;
  asm volatile("v_add_u32 %0, %1, %2" : "=v"(v) : "s"(y), "v"(x));
  return v;
}
// The wait states between a conversion and the MFMA that reads its result.
__device__ __forceinline__ void tile_valu_wait(bf16x8_g& x, bf16x8_g& y) {
  asm volatile("s_nop 1" : "+v"(x), "+v"(y));
}
// Eight e4m3 codes -> eight bf16, one conversion per pair.
__device__ __forceinline__ bf16x8_g fp8x8_to_bf16_hw(uint32_t x, uint32_t y) {
  typedef __bf16 bf16x2_g __attribute__((ext_vector_type(2)));
  const auto c = [](bf16x2_g v) { return __builtin_bit_cast(uint32_t, v); };
  const v4u u = {c(__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x, 1.0f, false)),
                 c(__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x, 1.0f, true)),
                 c(__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(y, 1.0f, false)),
                 c(__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(y, 1.0f, true))};
  return __builtin_bit_cast(bf16x8_g, u);
}
// Chunk position of 16-byte chunk c of tile row r is c ^ swz(r): the 16 rows
// that a fragment read touches lie on distinct banks (64 banks of 4 bytes).
__device__ __forceinline__ int tile_swz128(int r) { return (r >> 1) & 7; }
__device__ __forceinline__ int tile_swz64(int r) { return (r >> 2) & 3; }
#endif

// (M tile, N tile) of a tile number.
__device__ __forceinline__ int2 tile_at(const GemmArgs& a, int tile) {
  const int d = a.n_major ? a.nt : a.mt, q = tile / d, r = tile - q * d;
  return a.n_major ? make_int2(q, r) : make_int2(r, q);
}

template <bool F8, int EPI, int FM, int FN, int S, int KS, bool QUAD>
__global__ __launch_bounds__(256 * KS) __attribute__((amdgpu_waves_per_eu(KS, KS))) void gemm_tile_kernel(GemmArgs a) {
#ifdef __HIP_DEVICE_COMPILE__  // the host pass needs the launch stub only
  using T = TileShape<F8, FM, FN, S, KS>;
  constexpr bool kGlu = EPI == kEpiSwiglu;
  static_assert(!kGlu || FN % 2 == 0, "swiglu: gate and up fragments in pairs");
  static_assert(!QUAD || (FM % 2 == 0 && FN % 2 == 0), "quadrants");
  static_assert(S >= 2, "ring depth");
  constexpr int kCols = kGlu ? 8 * FN : 16 * FN;  // a wave's output columns
  static_assert(T::lds_bytes(kGlu) <= 163840, "LDS");
  __shared__ __align__(1024) uint8_t s_mem[T::lds_bytes(kGlu)];
  const int tid = KS == 1 ? threadIdx.x : threadIdx.x & 255;
  const int kg = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);  // K group
  uint8_t* const s_stage = s_mem + kg * (S * T::kStage);
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int fr = lane & 15, fq = lane >> 4;
  const int steps = a.K / T::kKb / KS;  // per K group: even, at least S rounded up to even (tile_fits)
  const size_t apitch = F8 ? static_cast<size_t>(a.lda) : 2 * static_cast<size_t>(a.lda);
  const int ncols = kGlu ? a.I : a.N;
  constexpr int kTileCols = 2 * kCols;
  const float a_scale = F8 ? *a.a_scale : 1.0f;
  const int tiles = a.mt * a.nt;
  float amax = 0.0f;

  // LDS byte addresses of this lane's fragment chunks in stage 0 (a fragment
  // advances 16 rows, which leaves the swizzle unchanged).
  const uint32_t lds0 = tile_lds_addr(s_stage);
  const uint32_t arow = lds0 + static_cast<uint32_t>((wm * 16 * FM + fr) * T::kARow);
  const uint32_t a_c0 = arow + 16u * static_cast<uint32_t>((2 * fq) ^ tile_swz128(fr));
  const uint32_t a_c1 = arow + 16u * static_cast<uint32_t>((2 * fq + 1) ^ tile_swz128(fr));
  const uint32_t wrow = lds0 + T::kABytes + static_cast<uint32_t>((wn * 16 * FN + fr) * T::kWRow);
  const uint32_t w_c0 = F8 ? wrow + 16u * static_cast<uint32_t>((2 * fq) ^ tile_swz128(fr))
                           : wrow + 16u * static_cast<uint32_t>(fq ^ tile_swz64(fr));
  const uint32_t w_c1 = wrow + 16u * static_cast<uint32_t>((2 * fq + 1) ^ tile_swz128(fr));

  // A tile's operands: its first rows, this thread's first chunk as an offset
  // from them, and that of the tile's last valid row: a row past the end reads
  // the last one (its results are not stored).
  struct Source {
    const uint8_t *abase, *wbase;
    uint32_t ao, alast, wo, wlast;
  };
  // Rows (tile rows) covered by one load of all 256 threads.
  constexpr int kARows = 4096 / T::kARow, kWRows = 4096 / T::kWRow;
  const int ar0 = tid >> 3, wr0 = F8 ? tid >> 3 : tid >> 2;
  const uint32_t ac = 16u * static_cast<uint32_t>((tid & 7) ^ tile_swz128(ar0));
  const uint32_t wc = 16u * static_cast<uint32_t>(F8 ? (tid & 7) ^ tile_swz128(wr0) : (tid & 3) ^ tile_swz64(wr0));
  // swiglu: a wave column's tile rows are its gate rows, then the up rows of
  // the same act columns; the column behind tile row r, by parts of r.
  const auto col_of = [&](int r) { return kGlu ? r / (16 * FN) * (8 * FN) + r % (8 * FN) : r; };
  static_assert(!kGlu || (8 * FN) % kWRows == 0 || kWRows % (16 * FN) == 0, "a load's columns follow its rows");
  const auto source = [&](Source& s, int tile) __attribute__((always_inline)) {
    const int2 at = tile_at(a, tile);
    const int m0 = at.x * T::kBM, n0 = at.y * kTileCols;
    s.abase = a.A + static_cast<size_t>(m0) * apitch + static_cast<size_t>(kg * steps) * 128;
    s.wbase = a.W + static_cast<size_t>(n0) * a.K + static_cast<size_t>(kg * steps) * T::kKb;
    s.ao = static_cast<uint32_t>(ar0 * apitch) + ac;
    s.alast = static_cast<uint32_t>(min(T::kBM - 1, a.M - 1 - m0) * apitch) + ac;
    s.wo = static_cast<uint32_t>(col_of(wr0) * static_cast<size_t>(a.K)) + wc;
    s.wlast = static_cast<uint32_t>(min(kTileCols - 1, ncols - 1 - n0) * static_cast<size_t>(a.K)) + wc;
  };
  // Load l of step k into stage st.
  const auto issue = [&](const Source& s, int l, int k, int st) __attribute__((always_inline)) {
    uint8_t* const dst = s_stage + st * T::kStage + wave * 1024;
    if (l < T::kALoads) {
      const uint32_t off = min(tile_add(s.ao, static_cast<uint32_t>(l * kARows * apitch)), s.alast);
      __builtin_amdgcn_global_load_lds(s.abase + static_cast<size_t>(k) * 128 + off,
                                       (tile_lds_ptr)(dst + l * 4096), 16, 0, 0);
    } else {
      const int w = l - T::kALoads;
      // the wave's 1 KB of load w lies in one half (gate or up) of a wave column
      constexpr int kRowsPerKb = 1024 / T::kWRow;
      const int row = w * kWRows + wave * kRowsPerKb;
      if (T::kWBytes % 4096 != 0 && row >= T::kBN) return;
      const uint8_t* p = s.wbase + static_cast<size_t>(k) * T::kKb;
      if (kGlu && row % (16 * FN) >= 8 * FN) p += static_cast<size_t>(a.I) * a.K;
      const uint32_t off =
          min(tile_add(s.wo, static_cast<uint32_t>(col_of(w * kWRows)) * static_cast<uint32_t>(a.K)), s.wlast);
      __builtin_amdgcn_global_load_lds(p + off, (tile_lds_ptr)(dst + T::kABytes + w * 4096), 16, 0, 0);
    }
  };
  static_assert(T::kWBytes % 2048 == 0, "the last load whole, or half of the waves'");
  // Waits until the loads of at most `S - 2` / `S - 1` steps are in flight
  // (where the weights end in half a load, half of the waves issue one fewer).
  const bool w_short = T::kWBytes % 4096 != 0 && wave >= 2;
  const auto vm_wait = [&](auto n_tag) {
    constexpr int n = decltype(n_tag)::value;
    if (w_short) tile_vm_wait<n * (T::kLoads - 1)>();
    else tile_vm_wait<n * T::kLoads>();
  };
  using Ahead1 = std::integral_constant<int, S - 1>;
  using Ahead2 = std::integral_constant<int, S - 2>;

  // Fragment registers: a half per set (quadrants) or a step per set (flat).
  constexpr int kFa = QUAD ? FM / 2 : FM, kFw = QUAD ? FN / 2 : FN;
  v4f acc[FM][FN];
  v4u fa[2][kFa][2], fw[2][kFw][T::kWv];
  bf16x8_g fb[QUAD ? 2 : 1][kFw][2];  // bf16 A: the weight fragments converted
  const auto read_a = [&](int set, int frag0, int n, uint32_t st) __attribute__((always_inline)) {
    const int i = n >> 1;
    fa[set][i][n & 1] = tile_read16((n & 1 ? a_c1 : a_c0) + st, 16 * (frag0 + i) * T::kARow);
  };
  const auto read_w = [&](int set, int frag0, int n, uint32_t st) __attribute__((always_inline)) {
    const int j = F8 ? n >> 1 : n, v = F8 ? n & 1 : 0;
    fw[set][j][v] = tile_read16((v ? w_c1 : w_c0) + st, 16 * (frag0 + j) * T::kWRow);
  };
  const auto landed_a = [&](int set) {
#pragma unroll
    for (int i = 0; i < kFa; ++i) asm volatile("" : "+v"(fa[set][i][0]), "+v"(fa[set][i][1]));
  };
  const auto landed_w = [&](int set) {
#pragma unroll
    for (int j = 0; j < kFw; ++j)
#pragma unroll
      for (int v = 0; v < T::kWv; ++v) asm volatile("" : "+v"(fw[set][j][v]));
  };
  constexpr int kNA = 2 * kFa, kNW = kFw * T::kWv;  // reads per set
  constexpr int kMf = kFa * kFw * (F8 ? 1 : 2);     // MFMAs per quadrant (flat: per step)
  // kMf MFMAs of the A set sa x the W set sw onto the accumulators from (i0,
  // j0), with extra(t) (reads, loads) after MFMA t; fresh: the W set is new
  // (bf16 A converts it, one fragment ahead).
  const auto multiply = [&](int sa, int sw, int i0, int j0, bool fresh, auto extra) __attribute__((always_inline)) {
    const auto convert = [&](int j, int h) {
      fb[QUAD ? sw : 0][j][h] = fp8x8_to_bf16_hw(fw[sw][j][0][2 * h], fw[sw][j][0][2 * h + 1]);
    };
    if (!F8 && fresh) {
      convert(0, 0);
      convert(0, 1);
    }
#pragma unroll
    for (int t = 0; t < kMf; ++t) {
      if constexpr (F8) {
        const int j = t / kFa, i = t % kFa;
        tile_mfma(acc[i0 + i][j0 + j], frag_of(fw[sw][j][0], fw[sw][j][T::kWv - 1]),
                  frag_of(fa[sa][i][0], fa[sa][i][1]));
      } else {
        const int j = t / (2 * kFa), i = (t / 2) % kFa, tj = t % (2 * kFa);
        bf16x8_g* const b = fb[QUAD ? sw : 0][j];
        if (fresh && tj == 0) tile_valu_wait(b[0], b[1]);
        tile_mfma(acc[i0 + i][j0 + j], b[t & 1], fa[sa][i][t & 1]);
        if (fresh && j + 1 < kFw && tj < 2) convert(j + 1, tj);
      }
      extra(t);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Calls f for the items of n that follow MFMA t: one after each MFMA, or
  // more where there are more items than MFMAs.
  const auto each = [&](int t, int n, auto f) __attribute__((always_inline)) {
    if (n <= kMf) {
      if (t < n) f(t);
    } else {
#pragma unroll
      for (int r = t * n / kMf; r < (t + 1) * n / kMf; ++r) f(r);
    }
  };
  // As each, spread evenly over q quarters of kMf MFMAs, MFMA t of them.
  const auto spread = [&](int t, int all, int n, auto f) __attribute__((always_inline)) {
#pragma unroll
    for (int r = t * n / all; r < (t + 1) * n / all; ++r) f(r);
  };

  int st = 0;
  // One step from stage st; loads step `kl` of `src` into it once it is free.
  // Reads its own second halves (quadrants) and the next stage's first ones
  // (flat: all of them), unless it is the tile's last. par: the step's parity.
  const auto step = [&](const Source& src, int kl, auto par, auto last_tag) __attribute__((always_inline)) {
    constexpr int f = decltype(par)::value, g = 1 - f;
    constexpr bool kLast = decltype(last_tag)::value;
    const int nst = st + 1 == S ? 0 : st + 1;
    const uint32_t cur = static_cast<uint32_t>(st * T::kStage), nxt = static_cast<uint32_t>(nst * T::kStage);
    if constexpr (QUAD) {
      // (A0, Wf) (A0, Wg) (A1, Wg) (A1, Wf), f = the W half read last step
      multiply(0, f, 0, f * kFw, true, [&](int t) { each(t, kNW, [&](int n) { read_w(g, g * kFw, n, cur); }); });
      tile_reads_wait();
      landed_w(g);
      multiply(0, g, 0, g * kFw, true, [&](int t) { each(t, kNA, [&](int n) { read_a(1, kFa, n, cur); }); });
      tile_reads_wait();
      landed_a(1);
      vm_wait(Ahead2{});
      __builtin_amdgcn_s_barrier();
      multiply(1, g, kFa, g * kFw, false, [&](int t) {
        if (!kLast) each(t, kNA, [&](int n) { read_a(0, 0, n, nxt); });
        spread(t, 2 * kMf, T::kLoads, [&](int l) { issue(src, l, kl, st); });
      });
      if (!kLast) {
        tile_reads_wait();
        landed_a(0);
      }
      multiply(1, f, kFa, f * kFw, false, [&](int t) {
        if (!kLast) each(t, kNW, [&](int n) { read_w(g, g * kFw, n, nxt); });
        spread(kMf + t, 2 * kMf, T::kLoads, [&](int l) { issue(src, l, kl, st); });
      });
      if (!kLast) {
        tile_reads_wait();
        landed_w(g);
      }
    } else {
      vm_wait(Ahead2{});
      __builtin_amdgcn_s_barrier();
      multiply(f, f, 0, 0, true, [&](int t) {
        if (!kLast) spread(t, kMf, kNA + kNW, [&](int n) {
          if (n < kNW) read_w(g, 0, n, nxt);
          else read_a(g, 0, n - kNW, nxt);
        });
        spread(t, kMf, T::kLoads, [&](int l) { issue(src, l, kl, st); });
      });
      if (!kLast) {
        tile_reads_wait();
        landed_a(g);
        landed_w(g);
      }
    }
    st = nst;
  };
  using Even = std::integral_constant<int, 0>;
  using Odd = std::integral_constant<int, 1>;

  Source src;
  const int tile_first = xcd_tile0(a.xcd_order);
  if (tile_first >= tiles) return;  // never: the grid has at most as many workgroups as tiles
  source(src, tile_first);
  bool fill = true;
  for (int tile = tile_first; tile < tiles; tile += gridDim.x) {
    if (fill) {
      // The ring's first S stages.
      if (!T::kRoll) __syncthreads();  // the previous tile's epilogue is done with the LDS
      st = 0;
#pragma unroll
      for (int s = 0; s < S; ++s)
#pragma unroll
        for (int l = 0; l < T::kLoads; ++l) issue(src, l, s, s);
      vm_wait(Ahead1{});
      __builtin_amdgcn_s_barrier();
      fill = !T::kRoll;
    }
    // The accumulators are cleared before the wait below, which covers the wait
    // states until an MFMA may read them.
#pragma unroll
    for (int q = 0; q < FM * FN; ++q) {
      acc[q / FN][q % FN] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
      asm volatile("" : "+a"(acc[q / FN][q % FN]));
    }
    // The first stage's leading fragments (landed: the barrier above, or the
    // last step's).
#pragma unroll
    for (int n = 0; n < kNW; ++n) read_w(0, 0, n, static_cast<uint32_t>(st * T::kStage));
#pragma unroll
    for (int n = 0; n < kNA; ++n) read_a(0, 0, n, static_cast<uint32_t>(st * T::kStage));
    tile_reads_wait();
    landed_a(0);
    landed_w(0);
    // The last kTail steps load the next tile's first stages (the last tile
    // its own again, never used, so that every step counts the same loads).
    constexpr int kTail = (S + 1) / 2 * 2;
    int k = 0;
    for (; k < steps - kTail; k += 2) {
      step(src, k + S, Even{}, std::false_type{});
      step(src, k + 1 + S, Odd{}, std::false_type{});
    }
    Source nsrc;
    if (T::kRoll) source(nsrc, tile + static_cast<int>(gridDim.x) < tiles ? tile + static_cast<int>(gridDim.x) : tile);
    const Source& after = T::kRoll ? nsrc : src;
    const auto tail = [&](auto j_tag) __attribute__((always_inline)) {
      // step steps - kTail + j loads step steps + S - kTail + j of this tile
      constexpr int j = decltype(j_tag)::value;
      if constexpr (j + S - kTail < 0) step(src, steps + S - kTail + j, Even{}, std::false_type{});
      else step(after, j + S - kTail, Even{}, std::false_type{});
      step(after, j + 1 + S - kTail, Odd{}, std::bool_constant<j + 2 == kTail>{});
    };
    static_assert(kTail <= 6, "tail steps");
    tail(std::integral_constant<int, 0>{});
    if constexpr (kTail > 2) tail(std::integral_constant<int, 2>{});
    if constexpr (kTail > 4) tail(std::integral_constant<int, 4>{});
    // The accumulators become ordinary values again, after the wait states
    // that the last MFMA's results need.
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int q = 0; q < FM * FN; ++q) asm volatile("" : "+a"(acc[q / FN][q % FN]));

    const int2 at = tile_at(a, tile);
    const int m0 = at.x * T::kBM, n0 = at.y * kTileCols;
    constexpr int kSlot = 4 * FM * FN * 64;  // between the K groups' hand-overs
    if constexpr (KS > 1) {
      // The K groups' partial sums meet, in group order: group b % KS finishes
      // the wave's 16-row block b, the others hand it theirs, lane-contiguous.
      tile_vm_wait<0>();
      __syncthreads();  // the rings are free
      v4f* const xs = reinterpret_cast<v4f*>(s_mem) + wave * (FM * FN * 64) + lane;
#pragma unroll
      for (int b = 0; b < FM; ++b)
        if (kg != b % KS) {
          const int from = kg < b % KS ? kg : kg - 1;
#pragma unroll
          for (int j = 0; j < FN; ++j) xs[from * kSlot + (b * FN + j) * 64] = tile_acc(acc[b][j]);
        }
      __syncthreads();
    }
    // Epilogue, 16 rows of the wave at a time through its own LDS region
    // (16-byte columns XOR-swizzled by row), read back row-contiguous.
    float* const se = reinterpret_cast<float*>(s_mem + (T::kRoll ? T::kRing : T::swap_bytes())) +
                      (kg * 4 + wave) * 16 * kCols;
    constexpr int kPow2 = (kCols / 4) & -(kCols / 4);  // the swizzle stays within the row
    constexpr int kSwz = kPow2 < 8 ? kPow2 - 1 : 7;
    const Granite4GemmEpilogue& ep = a.ep;
    const int col0 = n0 + wn * kCols;
    // one weight scale for all of the wave's columns, or one per column
    const float s_first = a_scale * epi_scale(ep, col0);
    const bool one_scale = kGlu || (ep.seg1 <= col0 || ep.seg1 >= col0 + kCols) &&
                                       (ep.seg2 <= col0 || ep.seg2 >= col0 + kCols);
    constexpr int kLanesPerRow = kCols / 8, kRowsPer = 64 / kLanesPerRow;
    constexpr int kIters = (16 + kRowsPer - 1) / kRowsPer;
    // (the lane anew in every tile: what follows from it stays out of the K loop's registers)
    int le = lane;
    asm volatile("" : "+v"(le));
    const int rl = le / kLanesPerRow, ch = le % kLanesPerRow, er = le & 15, eq = le >> 4;
    const int n = col0 + 8 * ch;
    const auto row_of = [&](int it) { return it * kRowsPer + rl; };
    const auto stored = [&](int b, int it) {  // whether this lane stores in iteration it of block b
      const int r = row_of(it);
      return (64 % kLanesPerRow == 0 || le < kRowsPer * kLanesPerRow) && (16 % kRowsPer == 0 || r < 16) &&
             m0 + wm * 16 * FM + 16 * b + r < a.M && n < ncols;
    };
    const auto out_off = [&](int b, int it) {
      return static_cast<size_t>(m0 + wm * 16 * FM + 16 * b + row_of(it)) * ep.ldc + n;
    };
    // The residual of block b, loaded while the block before it is stored
    uint4 res[2][kIters];
    // (where no 16 bytes of it are wanted, 16 bytes of W instead: a load under a
    // condition would keep the registers alive through the K loop).
    const auto load_res = [&](int b) __attribute__((always_inline)) {
#pragma unroll
      for (int it = 0; it < kIters; ++it)
        res[b & 1][it] = *reinterpret_cast<const uint4*>(
            a.vec_out && stored(b, it) ? reinterpret_cast<const uint8_t*>(ep.residual + out_off(b, it)) : a.W);
    };
    if (EPI == kEpiResidual) load_res(0);
#pragma unroll
    for (int b = 0; b < FM; ++b) {
      if (KS > 1 && kg != b % KS) continue;
      __builtin_amdgcn_sched_barrier(0);
      v4f sum[FN];
      if constexpr (KS > 1) {
        const v4f* const xs = reinterpret_cast<const v4f*>(s_mem) + wave * (FM * FN * 64) + lane;
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const v4f mine = tile_acc(acc[b][j]);
          sum[j] = kg == 0 ? mine : xs[(b * FN + j) * 64];
#pragma unroll
          for (int s = 1; s < KS; ++s)
            sum[j] += s == kg ? mine : xs[(s < kg ? s : s - 1) * kSlot + (b * FN + j) * 64];
        }
      }
      const auto column_block = [&](int c, auto one_tag) {
        // lane: row er, columns 16 c + 4 eq ..
        const int cn = 16 * c + 4 * eq;
        v4f y = KS == 1 ? tile_acc(acc[b][c]) : sum[c];
        if constexpr (kGlu) {
          const v4f u = KS == 1 ? tile_acc(acc[b][c + FN / 2]) : sum[c + FN / 2];
#pragma unroll
          for (int r = 0; r < 4; ++r) y[r] = silu_mul(y[r] * (a_scale * ep.scale0), u[r] * (a_scale * ep.scale1));
        } else if constexpr (decltype(one_tag)::value) {
#pragma unroll
          for (int r = 0; r < 4; ++r) y[r] *= s_first;
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) y[r] *= a_scale * epi_scale(ep, col0 + cn + r);
        }
        *reinterpret_cast<v4f*>(se + er * kCols + 4 * ((cn / 4) ^ (er & kSwz))) = y;
      };
      if (one_scale) {
#pragma unroll
        for (int c = 0; c < kCols / 16; ++c) column_block(c, std::true_type{});
      } else {
#pragma unroll
        for (int c = 0; c < kCols / 16; ++c) column_block(c, std::false_type{});
      }
      if (EPI == kEpiResidual && KS > 1 && b > 0) load_res(b);
      if (EPI == kEpiResidual && KS == 1 && b + 1 < FM) load_res(b + 1);
      tile_reads_wait();
#pragma unroll
      for (int it = 0; it < kIters; ++it) {
        if (!stored(b, it)) continue;
        const int r = row_of(it);
        const v4f lo = *reinterpret_cast<const v4f*>(se + r * kCols + 4 * ((2 * ch) ^ (r & kSwz)));
        const v4f hi = *reinterpret_cast<const v4f*>(se + r * kCols + 4 * ((2 * ch + 1) ^ (r & kSwz)));
        const float y[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        const size_t off = out_off(b, it);
        if (!kGlu && !a.vec_out) {
          for (int e = 0; e < 8 && n + e < ncols; ++e) {
            if (EPI == kEpiF32) ep.out_f32[off + e] = y[e];
            else if (EPI == kEpiResidual)
              ep.out_bf16[off + e] =
                  static_cast<uint16_t>(f32_to_bf16(bf16_to_f32(ep.residual[off + e]) + ep.resid_scale * y[e]));
            else ep.out_bf16[off + e] = static_cast<uint16_t>(f32_to_bf16(y[e]));
          }
          continue;
        }
        if (EPI == kEpiF32) {
          *reinterpret_cast<v4f*>(ep.out_f32 + off) = lo;
          *reinterpret_cast<v4f*>(ep.out_f32 + off + 4) = hi;
          continue;
        }
        uint32_t w[4];
        if (EPI == kEpiResidual) {
          const uint4 rv = res[b & 1][it];
          const uint32_t rw[4] = {rv.x, rv.y, rv.z, rv.w};
#pragma unroll
          for (int e = 0; e < 4; ++e)
            w[e] = pack_bf16_rne(lo_bf16(rw[e]) + ep.resid_scale * y[2 * e],
                                 hi_bf16(rw[e]) + ep.resid_scale * y[2 * e + 1]);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) w[e] = pack_bf16_rne(y[2 * e], y[2 * e + 1]);
        }
        if (kGlu) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            amax = fmaxf(amax, fmaxf(lo_bf16(w[e] & 0x7fff7fffu), hi_bf16(w[e] & 0x7fff7fffu)));
        }
        *reinterpret_cast<uint4*>(ep.out_bf16 + off) = make_uint4(w[0], w[1], w[2], w[3]);
      }
      tile_reads_wait();  // the block's reads are done before the next one's writes
    }
    if (T::kRoll) src = nsrc;
    else if (tile + static_cast<int>(gridDim.x) < tiles) source(src, tile + gridDim.x);
  }
  tile_vm_wait<0>();  // the ring's last loads land before the workgroup ends
  if constexpr (kGlu) {
    __shared__ float s_max[4 * KS];
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) amax = fmaxf(amax, __shfl_xor(amax, o));
    if (lane == 0) s_max[kg * 4 + wave] = amax;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
      for (int w = 1; w < 4 * KS; ++w) amax = fmaxf(amax, s_max[w]);
      a.partials[blockIdx.x] = amax;
    }
  }
#endif
}

// A tile configuration with its measured cost: a launch of r rounds of
// workgroups (one per CU, 256) takes about r (per_k K / 4096 + per_round) +
// fixed microseconds.
struct TileCost {
  float per_k, per_round, fixed;
};
// Where the configuration, the cheapest tile at a shape, is faster than the
// general kernels (gemm.hip), measured over 19 K from 128 to 12800, 17 to 8192
// rows and 256 to 25600 columns. Their prologue is shorter: a K of its own is
// needed where their 128-row tiles are all on the chip at once (two per CU),
// and where they take turns. Their rounds are of 512 tiles and not of 256: in
// turns, `in_turn_us` (if set) is compared with theirs. (It is the time of the
// same launch, fitted over K from 1024 on, and the choice between tiles stays
// with `cost`, which is the closer one between them at layer shapes.)
struct TileVsGeneral {
  int at_once_k = 0, in_turn_k = 0;
  TileCost in_turn_us = {};
};

// Tiles of the general kernels: 128 rows x 128 weight rows.
inline long long general_tiles(const GemmArgs& a, bool glu) {
  const long long n = glu ? (a.I + 63) / 64 : (a.N + 127) / 128;
  return (a.M + 127) / 128 * n;
}

template <bool F8, int FM, int FN, int S, int KS, bool QUAD>
struct TileConfig {
  using Shape = TileShape<F8, FM, FN, S, KS>;
  TileCost cost;
  TileVsGeneral vs = {};

  static int cols(bool glu) { return (glu ? 16 : 32) * FN; }
  // Whether the kernel takes these arguments: whole pairs of steps for every
  // K group, at least as many as the ring's tail, and a tile's rows within
  // 32-bit offsets.
  static bool fits(const GemmArgs& a) {
    const int per = Shape::kKb * KS;
    const long long apitch = (F8 ? 1LL : 2LL) * a.lda;
    return a.K % (2 * per) == 0 && a.K / per >= (S + 1) / 2 * 2 && Shape::kBM * apitch < (1LL << 32) &&
           static_cast<long long>(Shape::kBN) * a.K < (1LL << 32);
  }
  static long long tiles(const GemmArgs& a, bool glu) {
    const int n = glu ? a.I : a.N;
    return static_cast<long long>((a.M + Shape::kBM - 1) / Shape::kBM) * ((n + cols(glu) - 1) / cols(glu));
  }
  static float time(const TileCost& c, const GemmArgs& a, bool glu) {
    const long long rounds = (tiles(a, glu) + kCUs - 1) / kCUs;
    return static_cast<float>(rounds) * (c.per_k * (static_cast<float>(a.K) / 4096.0f) + c.per_round) + c.fixed;
  }
  float predicted(const GemmArgs& a, bool glu) const { return time(cost, a, glu); }
  // Whether the general kernels are the faster ones where this is the cheapest
  // tile. general: their cost per round of 2 kCUs tiles.
  bool loses(const GemmArgs& a, bool glu, const TileCost& general) const {
    const long long g = general_tiles(a, glu), at_once = 2 * kCUs;
    if (a.K < (g <= at_once ? vs.at_once_k : vs.in_turn_k)) return true;
    // (SwiGLU 300 rows, I = 9600: 450 general tiles at once 16.2-42.1 us for K of
    // 1536 to 4608, 450 128 x 128 tiles in two rounds 18.7-42.6)
    if (g <= at_once) return glu && tiles(a, glu) > kCUs;
    const long long rounds = (g + at_once - 1) / at_once;
    return vs.in_turn_us.per_k > 0.0f &&
           static_cast<float>(rounds) * (general.per_k * (static_cast<float>(a.K) / 4096.0f) + general.per_round) +
                   general.fixed <
               time(vs.in_turn_us, a, glu);
  }
  template <int EPI>
  static unsigned launch(GemmArgs a) {
    constexpr bool kGlu = EPI == kEpiSwiglu;
    const long long t = tiles(a, kGlu);
    if (t > INT_MAX) return 0;
    a.mt = (a.M + Shape::kBM - 1) / Shape::kBM;
    a.nt = ((kGlu ? a.I : a.N) + cols(kGlu) - 1) / cols(kGlu);
    const unsigned grid = static_cast<unsigned>(t < kCUs ? t : kCUs);
    a.xcd_order = gemm_xcd_order(a.mt, grid);
    a.n_major = !a.xcd_order && gemm_n_major(a.mt, a.nt, grid);
    a.xcd_order = a.xcd_order || a.n_major;
    hipLaunchKernelGGL((gemm_tile_kernel<F8, EPI, FM, FN, S, KS, QUAD>), grid, 256 * KS, 0, stream(), a);
    return grid;
  }
};

// Launches the configuration with the least predicted time of those that fit;
// returns its grid, or 0 (nothing is launched) where none fits or, above
// kSkinnyMaxM rows, the general kernels are the faster ones.
template <int EPI, class... C>
unsigned launch_cheapest(const GemmArgs& a, const TileCost& general, const C&... configs) {
  constexpr bool kGlu = EPI == kEpiSwiglu;
  float best = 0.0f;
  int pick = -1, i = 0;
  const auto look = [&](const auto& c) {
    if (c.fits(a)) {
      const float t = c.predicted(a, kGlu);
      if (pick < 0 || t < best) best = t, pick = i;
    }
    ++i;
  };
  (look(configs), ...);
  unsigned grid = 0;
  i = 0;
  const auto go = [&](const auto& c) {
    if (i++ == pick && (a.M <= kSkinnyMaxM || !c.loses(a, kGlu, general))) grid = c.template launch<EPI>(a);
  };
  (go(configs), ...);
  return grid;
}

}  // namespace
}  // namespace g4

#endif  // G4_GEMM_TILE_H
