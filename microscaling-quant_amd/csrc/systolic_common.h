// What the systolic kernels share: the launch arguments, the fast datapath's per-lane constants, the caller's
// hints and epilogue.
#pragma once

#include "mxq_common.h"
#include "mxq_numerics.h"
#include "reducer_common.h"

namespace mxq_sys {

using namespace mxq_red;

constexpr int kMaxLanes = 64;
constexpr uint32_t kFastAMaxBits = 0x71800000u;   // 2^100: A's rows are staged times up to 2^15

struct SysArgs {
  Operand A, XA, B, XB;   // A: K x M, XA: nb x M, B: K x N, XB: nb x N
  float* C;
  int64_t ldc, batch_c;   // C: M x N
  uint32_t* flags;        // one per fast tile per problem (1: the general kernel computes it)
  int64_t tiles_x, tiles_y;
  int fbm, fbn;           // the fast kernel's tile height and width
  int64_t K, M, N;
  int size, block_size;
  mxq_arith_spec ar;
  int8_t lane_e[kMaxLanes];
  int8_t lane_m[kMaxLanes];
  float fast_prod_max;    // the fast kernel's bound on max|a| * max|b| (see fast_prod_bound)
  // the caller's hints (mxq_systolic_hints), NULL when absent
  const uint8_t* skip;    // per problem, 32-row group and 32-column group of C: nonzero = not needed
  int64_t skip_rows, skip_cols;
  const int32_t* k_end;   // per problem and 64-column group of A: rows at and past it hold only +-0 codes
  int64_t kend_groups;    // ceil(M / 64): 64-column groups of A, 64-row groups of C
  const int32_t* c_end;   // per problem and 64-row group of C: skipped tiles from this column on are not stored
  // dispatch position (blockIdx.x + tiles_x * (blockIdx.y + tiles_y * blockIdx.z)) -> fast tile
  // (z * tiles_y + ty) * tiles_x + tx, by descending work (k_tile_order); NULL: the grid's own tile
  const uint32_t* order;
  // with an order and skip: bit 31 of an order entry set when its tile is skipped (tile_skipped at the fast tile
  // size, as k_tile_bucket found it), so the fast kernels read no skip bytes; the tile is the low 31 bits
  int order_skip;
  // with k_end: per problem, 32-row stage and 32-column group of A (suf_a) and of B (suf_b), nonzero when rows
  // of that stage may not be skipped (k_suffix_flags)
  const uint8_t* suf_a;
  const uint8_t* suf_b;
  const uint8_t* a_live;      // the caller's suffix bytes of A (mxq_systolic_hints), NULL when absent
  int64_t stages;
  int epi_on;                 // apply `epi` to every output as it is stored
  mxq_systolic_epilogue epi;
};

// The caller's epilogue, per output row: the mask row of output row r of problem z (NULL without a mask), then
// R(R(v * scale) + row[c]) per output, R = bf16 RNE or identity.  Rows, m, z_per_b and z0 + z fit 31 bits
// (M / 32 <= 65535; the launch checks the rest), so both divisions are 32-bit: as 64-bit divisions on the scalar
// unit they were some hundred instructions in every workgroup's stores.
__device__ __forceinline__ const float* epi_mask(const SysArgs& a, int64_t z) {   // problem z's mask rows
  const mxq_systolic_epilogue& e = a.epi;
  if (!e.mask) return nullptr;
  const uint32_t zb = (uint32_t)e.z_per_b;
  const int64_t b = (int64_t)((uint32_t)(e.z0 + z) / zb) - (int64_t)((uint32_t)e.z0 / zb);
  return e.mask + b * e.mask_b_stride;
}
__device__ __forceinline__ uint32_t epi_rm(const SysArgs& a, int64_t r) {             // r % m
  return (uint32_t)r % (uint32_t)a.epi.m;
}
__device__ __forceinline__ const float* epi_row(const SysArgs& a, int64_t z, int64_t r) {
  const float* mz = epi_mask(a, z);
  return mz ? mz + (int64_t)epi_rm(a, r) * a.epi.mask_row_stride : nullptr;
}

__device__ __forceinline__ float epi_apply(const SysArgs& a, const float* row, int64_t c, float v) {
  const mxq_systolic_epilogue& e = a.epi;
  v = v * e.scale;
  if (e.bf16) v = bf16_rne(v);
  if (row) {
    v = v + row[c];
    if (e.bf16) v = bf16_rne(v);
  }
  return v;
}

// ---------------------------------------------------------------------------------- fast datapath
// qtorch's grid (float_em ties_away) for values its saturation is never reached by: the bits rounded half away at m
// fraction bits, and below the least value 2^-L to 0 up to its half, to itself above.  A float below 2^-L plus and
// minus 1.5 * 2^(23 - L) is rounded to a multiple of 2^-L, a tie (half of 2^-L) to the even one, 0.
struct Qtorch {
  uint32_t half, keep;   // half the step of m fraction bits, and the mask of the bits kept
  float magic, least;    // 1.5 * 2^(23 - L), 2^-L
};
constexpr Qtorch qtorch_of(int e, int m) {
  Qtorch q{};
  q.half = 1u << (22 - m);
  q.keep = ~((1u << (23 - m)) - 1u);
  const int L = (1 << (e - 1)) - 1;
  double p = 1.0;
  for (int i = 0; i < L; ++i) p *= 0.5;
  q.least = e == 8 ? 0.0f : (float)p;               // float32's own exponents: nothing is below the least value
  q.magic = e == 8 ? 0.0f : (float)(1.5 * 8388608.0 * p);
  return q;
}
template <bool UNDER>
__device__ __forceinline__ float qtorch_fast(float x, const Qtorch& q) {
#pragma clang fp contract(off)
  const float r = u2f((f2u(x) + q.half) & q.keep);
  if constexpr (!UNDER) return r;
  const float h = (r + q.magic) - q.magic;
  return __builtin_fabsf(r) < q.least ? h : r;
}

// Per-lane constants of the fast kernel, built on the host from the schedule (see make_fast_lanes).
struct FastLanes {
  int32_t a_exp[32];     // A's rows of lane i are staged times 2^a_exp[i]: 6 + m_i (e4 lanes), 0 (bf16 lane)
  float rescale[32];     // before e4 lane i the scaled sum is multiplied by 2^(m_i - m_{i-1}) (1: unchanged)
  float split[32];       // 2^(23 - m_i) + 1: split_rne's constant for RNE at m_i fraction bits
  float magic[32];       // 1.5 * 2^(17 - m_i): (p + magic) - magic rounds p to a multiple of 2^-(6 + m_i)
  float out_scale;       // scaled sum -> sum after the last e4 lane: 2^-(6 + m_last)
  uint32_t pmask;        // product truncation to prod_m fraction bits
  float flush_thr;       // bf16 lane: |product| below this becomes zero
  uint32_t xs_lo, xs_hi; // scale magnitudes (bit patterns) that allow the short tile add
  float pw[32], low[32]; // P = 2^(23 - m_i) and 1 - P: fma_rne's constants (kWide's lanes only)
  // MXQUANT's grids (Qtorch): the product's and the lanes'
  Qtorch prod, lane[32];
};

// The fast datapaths, by Arithmetic and ladder:
//   kE4Final  MXGEMMINI, HW_FINAL (constants are literals)
//   kE4       MXGEMMINI, e4 lanes of non-decreasing m, optionally a last bf16 lane
//   kWide     MXGEMMINI, lanes of e >= 5 and m <= 10 (bf16 among them), neither ever falling, on whose grids every
//             kept product lies (the flush threshold times 2^-prod_m is a multiple of each lane's subnormal step)
//   kMxqFinal MXQUANT, HW_FINAL
//   kMxq      MXQUANT, any lanes
//   kMxqHigh  MXQUANT, lanes no nonzero sum of products falls below (their least value is at most the product
//             grid's last bit at its least value)
enum LaneKind { kE4Final, kE4, kWide, kMxqFinal, kMxq, kMxqHigh };
constexpr bool kind_mxq(int kind) { return kind >= kMxqFinal; }

// RNE of a float32 bit pattern at 7 fraction bits (bf16).  Finite values, infinities and the quiet NaNs the
// ALU makes (0x7FC00000, 0xFFC00000) map as bf16_rne does; a NaN whose low 16 bits would carry is never
// present (the workgroup's codes and scales are finite whenever its results are kept; every NaN is made by
// the ALU).
__device__ __forceinline__ float bf16_bits(float x) {
  const uint32_t u = f2u(x);
  return u2f((u + 0x7FFFu + ((u >> 16) & 1u)) & 0xFFFF0000u);
}

// HW_FINAL's ladder (mxq/schedule.py:21): lanes 0-7 e4m4, 8-9 e4m5, 10-14 e4m6, lane 15 bf16.
constexpr int hw_final_m(int i) { return i < 8 ? 4 : (i < 10 ? 5 : 6); }

// The per-lane constants of the fast datapath: compile-time immediates for HW_FINAL (HWF), else the host-built
// table.  i is a compile-time constant at every use (the lane loop is unrolled).
template <bool HWF>
struct LaneConsts {
  const FastLanes& fl;
  // RNE of an e4 sum at lane i's m: two operations where the constants are literals, else the three-operation split
  __device__ __forceinline__ float rne(float y, int i) const {
    if constexpr (HWF) return fma_rne(y, (float)(1u << (23 - hw_final_m(i))));
    else return split_rne(y, fl.split[i]);
  }
  // before lane i the scaled sum is multiplied by rescale(i) when the lane's m steps up
  __device__ __forceinline__ bool steps_up(int i) const {
    if constexpr (HWF) return i == 8 || i == 10;
    else return fl.rescale[i] != 1.0f;
  }
  __device__ __forceinline__ float rescale(int i) const {
    if constexpr (HWF) return 2.0f;
    else return fl.rescale[i];
  }
  __device__ __forceinline__ float out_scale() const {
    if constexpr (HWF) return 0x1p-12f;                      // 2^-(6 + m of lane 14)
    else return fl.out_scale;
  }
  // 1.5 * 2^(17 - m_i): adding and subtracting it rounds a product in value units to the lane's subnormal step
  __device__ __forceinline__ float magic(int i) const {
    if constexpr (HWF) return 1.5f * (float)(1u << (17 - hw_final_m(i)));
    else return fl.magic[i];
  }
};

// Scales a thread's staged A rows by 2^a_exp[lane of the row] on the way to LDS.  A thread always stages the
// same rows of a stage (stages start at multiples of 32 and SIZE | 32), so the exponents are fixed per thread.
template <int W, int NT, int SIZE>
struct ScaledRows {
  static constexpr int PER = KT * W / NT;
  int ex[PER];
  __device__ __forceinline__ void init(const FastLanes& fl, bool vec) {
    const int t = threadIdx.x;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int e = vec ? (t + (j / 4) * NT) * 4 + (j % 4) : t + j * NT;
      ex[j] = fl.a_exp[(e / W) % SIZE];
    }
  }
  __device__ __forceinline__ void apply(float (&v)[PER]) const {
#pragma unroll
    for (int j = 0; j < PER; ++j) v[j] = ldexpf(v[j], ex[j]);
  }
};

// A thread's TM x TN outputs of problem z into C (inside C only).
template <int TM, int TN>
__device__ __forceinline__ void write_tile(const SysArgs& a, int64_t z, int64_t mr, int64_t nc,
                                           const float (&C)[TM][TN]) {
  float* Cz = a.C + z * a.batch_c;
  // the epilogue's mask rows: problem z's base once, then (mr + x) % m stepped row by row (below m, so one
  // subtraction wraps it)
  const float* mz = a.epi_on ? epi_mask(a, z) : nullptr;
  uint32_t rm = mz ? epi_rm(a, mr) : 0u;
#pragma unroll
  for (int x = 0; x < TM; ++x) {
    if (x > 0) {
      rm += 1u;
      rm = rm >= (uint32_t)a.epi.m ? rm - (uint32_t)a.epi.m : rm;
    }
    if (mr + x >= a.M) continue;
    if (a.epi_on) {
      const float* row = mz ? mz + (int64_t)rm * a.epi.mask_row_stride : nullptr;
#pragma unroll
      for (int y = 0; y < TN; ++y)
        if (nc + y < a.N) Cz[(mr + x) * a.ldc + nc + y] = epi_apply(a, row, nc + y, C[x][y]);
    } else {
#pragma unroll
      for (int y = 0; y < TN; ++y)
        if (nc + y < a.N) Cz[(mr + x) * a.ldc + nc + y] = C[x][y];
    }
  }
}

// Whether every 32 x 32 group of the bm x bn tile (bm, bn in {32, 64}) at (m0, n0) of problem z is marked in
// the caller's skip map.  The four candidate bytes are loaded together, unconditionally (indices clamped into
// the map, the unwanted bytes ignored), rather than one after another.
__device__ __forceinline__ void skip_bytes(const SysArgs& a, int64_t z, int64_t m0, int64_t n0, uint32_t (&v)[4]) {
  const uint8_t* sk = a.skip + z * a.skip_rows * a.skip_cols;
  const int64_t r0 = m0 / 32, c0 = n0 / 32;   // inside the map: m0 < M, n0 < N
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int64_t r = r0 + (k >> 1) < a.skip_rows ? r0 + (k >> 1) : a.skip_rows - 1;
    const int64_t c = c0 + (k & 1) < a.skip_cols ? c0 + (k & 1) : a.skip_cols - 1;
    v[k] = sk[r * a.skip_cols + c];
  }
}

__device__ __forceinline__ bool skip_all(const SysArgs& a, int64_t m0, int64_t n0, int bm, int bn,
                                         const uint32_t (&v)[4]) {
  const int64_t r0 = m0 / 32, c0 = n0 / 32;
  bool all = true;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const bool in = 32 * (k >> 1) < bm && 32 * (k & 1) < bn && r0 + (k >> 1) < a.skip_rows &&
                    c0 + (k & 1) < a.skip_cols;
    all &= !in || v[k] != 0u;
  }
  return all;
}

__device__ __forceinline__ bool tile_skipped(const SysArgs& a, int64_t z, int64_t m0, int64_t n0, int bm, int bn) {
  uint32_t v[4];
  skip_bytes(a, z, m0, n0, v);
  return skip_all(a, m0, n0, bm, bn, v);
}

// Where the reduction of the tile whose rows start at m0 stops under the caller's k_end: at K without one, else
// k_end rounded up to a whole stage.
__device__ __forceinline__ int64_t tile_kstop(const SysArgs& a, int64_t z, int64_t m0) {
  if (!a.k_end) return a.K;
  const int64_t ke = a.k_end[z * a.kend_groups + m0 / 64];
  const int64_t ks = ke <= 0 ? 0 : (ke + KT - 1) / KT * KT;
  return ks > a.K ? a.K : ks;
}

// One reduction's steps in value units, by datapath.
template <int KIND, int SIZE, bool BF16_LAST>
struct Datapath {
  static_assert((KIND != kE4Final && KIND != kMxqFinal) || (SIZE == 16 && BF16_LAST), "HW_FINAL has 16 lanes, the last bf16");
  const FastLanes& fl;

  // The sum after lane i (a compile-time constant at every use): S before it, q = a * b.  For MXGEMMINI the product
  // is q with the bits past prod_m masked off.
  //   e4 lanes: rounded to the lane's subnormal step 2^-(6+m) by adding and subtracting 1.5 * 2^(17-m) (exact:
  //     |p| < 2^(16-m) whenever the tile's results are kept; the flush below 2^prod_floor is under half a step),
  //     added exactly, RNE at m.
  //   wide lanes and the bf16 lane: flushed below the threshold, one float32 add (24 >= 2 * (m + 1) + 1 bits, so the
  //     rounding to float32 before the one to m <= 10 bits is harmless), RNE at m.
  // The first lane's sum is its product: prod_m <= m, so the lane's RNE keeps it.
  __device__ __forceinline__ float step(float S, float q, int i) const {
#pragma clang fp contract(off)
    if constexpr (kind_mxq(KIND)) {
      if constexpr (KIND == kMxqFinal) {
        const float p = qtorch_fast<true>(q, fl.prod);
        if (i == SIZE - 1) return qtorch_fast<false>(S + p, qtorch_of(8, 7));
        return qtorch_fast<true>(i == 0 ? p : S + p, qtorch_of(4, hw_final_m(i)));
      } else {
        const float p = qtorch_fast<true>(q, fl.prod);
        return qtorch_fast<KIND == kMxq>(i == 0 ? p : S + p, fl.lane[i]);
      }
    } else {
      float t = u2f(f2u(q) & fl.pmask);
      if (KIND == kWide || (BF16_LAST && i == SIZE - 1)) {
        t = __builtin_fabsf(t) < fl.flush_thr ? 0.0f : t;
        if (KIND == kWide && i == 0) return t;
        if constexpr (KIND == kWide) return fma_rne(S + t, fl.pw[i], fl.low[i]);
        return fma_rne(S + t, 65536.0f);
      }
      const LaneConsts<KIND == kE4Final> lc{fl};
      const float mg = lc.magic(i);
      const float p = (t + mg) - mg;
      return i == 0 ? p : lc.rne(S + p, i);
    }
  }
  // The tile of a finished sum: bf16(S * scale) for MXGEMMINI (exact, S of at most 8 significant bits, or rounded
  // where nothing is subnormal, when the block's scales allow the short form), the float32 product for MXQUANT.
  __device__ __forceinline__ float tile(float S, float scale, bool short_add) const {
#pragma clang fp contract(off)
    const float t = S * scale;
    if constexpr (kind_mxq(KIND)) return t;
    if (!short_add) return bf16_bits(t);
    return KIND == kWide ? fma_rne(t, 65536.0f) : t;
  }
  // C after the tile of a block whose scales allow the short form: MXGEMMINI's exact product joins the sum in one fma.
  __device__ __forceinline__ float tile_add(float C, float S, float scale) const {
    if constexpr (kind_mxq(KIND) || KIND == kWide) return add(C, tile(S, scale, true), false);
    return fma_rne(__builtin_fmaf(S, scale, C), 65536.0f);
  }
  // C after the tile: one rounding to bf16 (two operations while no scale has been large), or the float32 sum.
  __device__ __forceinline__ float add(float C, float t, bool large) const {
#pragma clang fp contract(off)
    if constexpr (kind_mxq(KIND)) return C + t;
    return large ? bf16_bits(C + t) : fma_rne(C + t, 65536.0f);
  }
};

// The kernels' launches, a translation unit for each family of datapaths.
void launch_tile_e4(int kind, bool bf16_last, dim3 grid, const SysArgs& a, const FastLanes& fl, hipStream_t st);
void launch_tile_wide(dim3 grid, const SysArgs& a, const FastLanes& fl, hipStream_t st);
void launch_tile_mxquant(int kind, dim3 grid, const SysArgs& a, const FastLanes& fl, hipStream_t st);

// k_systolic_small's tile: rows x 2^log_cw outputs a workgroup of `waves` waves.
struct SmallTile {
  int rows, log_cw, waves;
};
void launch_small_e4(int kind, bool bf16_last, const SysArgs& a, const FastLanes& fl, const SmallTile& t, int64_t count,
                     hipStream_t st);
void launch_small_wide(const SysArgs& a, const FastLanes& fl, const SmallTile& t, int64_t count, hipStream_t st);
void launch_small_mxquant(int kind, const SysArgs& a, const FastLanes& fl, const SmallTile& t, int64_t count,
                          hipStream_t st);

}  // namespace mxq_sys
