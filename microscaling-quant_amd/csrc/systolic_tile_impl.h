// The systolic product on tiles of 64 x 64 or 32 x 32 outputs: k_systolic_tile, eight or four waves a workgroup, 4 x 2
// or 2 x 2 outputs a thread, every datapath of Datapath, blocks of 32.
//
// Stages of 64 rows (32 on the small tile) move straight from global memory into LDS (global_load_lds: no registers, no
// LDS stores) while the stage before is reduced, one barrier a stage; the operands' maxima are read back from LDS once
// a stage.  Rows of whole fours of columns, 16-byte aligned, move 16 bytes a lane, others 4; a tile past the last
// column reads that column again (its outputs are not stored), and a stage past K's end is filled by the threads,
// zeros below.  The workgroup's verdict and flag are k_systolic_fast's, and so are the caller's hints (dispatch order,
// skipped tiles, the reduction's stop under k_end and the check of the rows past it) and the epilogue.
//
// Bound by VALU issue: 7 instructions a MAC under HW_FINAL, all full rate.  512 x 4096 outputs, K = 4096: 0.94 ms
// (1.07 with three-operation roundings), 512 x 4095: 0.98 (1.14 on k_systolic_fast, which took ragged operands before);
// K = 2048, 333 x 5632: 0.52 on small tiles (0.73 on large ones, whose second round is nearly empty, 0.54 on 32 x 64,
// which were nowhere the fastest), MXGEMMINI e4m4 lanes 512 x 4096: 0.65, e5m6: 0.69, MXQUANT(4, 3): 1.15.
// 4 x 2 outputs a thread (four waves a SIMD): with 4 x 4 (172 VGPRs, two waves a SIMD) 512 x 4096 took 5 % longer,
// with 4 x 1 (sixteen waves, one workgroup a CU) 17 %.
#pragma once

#include "systolic_common.h"

namespace mxq_sys {

// One wave's share of a stage of an operand of W columns, ROWS rows from row r0, straight into LDS.  q: the lane's own
// first element; vec: 16 bytes a lane, 256 / W rows an instruction, else 4 bytes, 64 / W rows.
template <int W, int ROWS, int KS>
__device__ __forceinline__ void load_rows(const float* q, int64_t ld, bool vec, int r0, float (&dst)[KS][W]) {
  typedef __attribute__((address_space(3))) void* lds_t;
  constexpr int RV = 256 / W, RD = 64 / W;
  static_assert(ROWS % RV == 0 && ROWS % RD == 0, "whole instructions");
  if (vec) {
#pragma unroll
    for (int j = 0; j < ROWS; j += RV) __builtin_amdgcn_global_load_lds(q + j * ld, (lds_t)&dst[r0 + j][0], 16, 0, 0);
  } else {
#pragma unroll 1
    for (int j = 0; j < ROWS; j += RD) __builtin_amdgcn_global_load_lds(q + j * ld, (lds_t)&dst[r0 + j][0], 4, 0, 0);
  }
}

// A thread's TM rows of one k, adjacent in LDS.
template <int TM>
__device__ __forceinline__ void lds_row(const float* src, float (&v)[TM]) {
  if constexpr (TM == 4) {
    const float4 q = *reinterpret_cast<const float4*>(src);
    v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
  } else {
    const float2 q = *reinterpret_cast<const float2*>(src);
    v[0] = q.x; v[1] = q.y;
  }
}

// WHOLE: every tile lies inside C and the operands' rows are whole fours of columns, 16-byte aligned (HW_FINAL's own
// instances, which leave the choice a stage out: 512 x 4096 outputs, K = 4096: 0.942 ms, 0.970 without them).  The
// others take a last block that is alone in its stage of two by itself (2048 x 4096 outputs: K = 32 76 -> 45 us, K = 96
// 135 -> 102; ladder e4m4, 1024 x 2048, K = 200: 89 -> 81); in WHOLE's instance that code cost 2 % of the time above.
template <int KIND, int SIZE, bool BF16_LAST, int BM, bool WHOLE>
__global__ void __launch_bounds__(BM * 8, 4) k_systolic_tile(const SysArgs args, const FastLanes fl) {
  static_assert(BM == 64 || BM == 32, "64 x 64 or 32 x 32 tiles");
  constexpr int BN = BM, TM = BM == 32 ? 2 : 4, TN = 2, KS = BM, NBS = KS / KT;   // a stage has as many rows as a tile
  constexpr int NT = (BM / TM) * (BN / TN), NWV = NT / 64;   // threads, waves
  constexpr bool HALF = NBS > 1 && !WHOLE;
  const Datapath<KIND, SIZE, BF16_LAST> dp{fl};
  // the two stage buffers are distinct arrays, each named where it is used: the compiler can then tell the
  // direct-to-LDS loads into one from the reads of the other, and does not wait for the loads before them
  __shared__ __align__(16) float sa0[KS][BM], sa1[KS][BM];
  __shared__ __align__(16) float sb0[KS][BN], sb1[KS][BN];
  __shared__ __align__(16) float xs_a[2][NBS][BM];
  __shared__ __align__(16) float xs_b[2][NBS][BN];
  __shared__ uint32_t denies_w[2][NBS][NWV];        // per buffer, block and wave: scale_denies of its scales
  __shared__ uint32_t red[4][NWV];
  const int tn = threadIdx.x % (BN / TN), tm = threadIdx.x / (BN / TN);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  // the tile: from the caller's dispatch order (k_tile_order: heaviest first) when there is one, else the grid's
  int64_t z, ty, tx;
  bool marked = false;                              // skipped, as the order entry says (order_skip)
  if (args.order) {
    uint32_t t = args.order[blockIdx.x + args.tiles_x * (blockIdx.y + args.tiles_y * (int64_t)blockIdx.z)];
    if (args.order_skip) {
      marked = (t >> 31) != 0u;
      t &= 0x7FFFFFFFu;
    }
    const uint32_t zy = t / (uint32_t)args.tiles_x;
    tx = t - zy * (uint32_t)args.tiles_x;
    z = zy / (uint32_t)args.tiles_y;
    ty = zy - (uint32_t)z * (uint32_t)args.tiles_y;
  } else {
    z = blockIdx.z;
    ty = blockIdx.y;
    tx = blockIdx.x;
  }
  const int64_t m0 = ty * BM, n0 = tx * BN;
  const float* A = args.A.p + z * args.A.batch + m0;
  const float* B = args.B.p + z * args.B.batch + n0;
  const float* XA = args.XA.p + z * args.XA.batch + m0;
  const float* XB = args.XB.p + z * args.XB.batch + n0;
  const int64_t K = args.K, M = args.M, N = args.N;
  // the reduction stops past the caller's k_end for these columns of A (a multiple of 32 below K): nothing of A or its
  // scales is read from there on, and those rows are checked below
  const int64_t stop = tile_kstop(args, z, m0), nb = (stop + KT - 1) / KT;
  // Lanes past an operand's columns read its last ones.
  constexpr int ROWS = KS / NWV;                    // rows of each operand a wave moves
  const int last_a = !WHOLE && M - m0 < BM ? (int)(M - m0) - 1 : BM - 1;
  const int last_b = !WHOLE && N - n0 < BN ? (int)(N - n0) - 1 : BN - 1;
  const bool va = WHOLE || (vec_ok(args.A, A) && M % 4 == 0), vb = WHOLE || (vec_ok(args.B, B) && N % 4 == 0);
  const int swave = __builtin_amdgcn_readfirstlane(wave);
  auto lane_at = [&](const float* p, bool vec, int w, int last, int64_t ld) {
    const int per = vec ? w / 4 : w, c = (vec ? 4 : 1) * (lane % per), most = vec ? last - 3 : last;
    return p + (swave * ROWS + lane / per) * ld + (c < most ? c : most);
  };
  const float* qa = lane_at(A, va, BM, last_a, args.A.ld);
  const float* qb = lane_at(B, vb, BN, last_b, args.B.ld);
  const int64_t xcol = threadIdx.x < BM ? (threadIdx.x < last_a ? threadIdx.x : last_a)
                                        : ((int)threadIdx.x - BM < last_b ? (int)threadIdx.x - BM : last_b);
  float xv[NBS];
  // the scales' loads go first: a wait the compiler places before rewriting their registers then does not
  // wait for the stage's direct-to-LDS loads too
  auto load_stage = [&](int64_t k, float (&da)[KS][BM], float (&db)[KS][BN]) __attribute__((always_inline)) {
    const int t = threadIdx.x;
#pragma unroll
    for (int q = 0; q < NBS; ++q) {
      const int64_t g = k / KT + q;
      xv[q] = 0.0f;
      if (t < BM + BN && g < nb) xv[q] = t < BM ? XA[g * args.XA.ld + xcol] : XB[g * args.XB.ld + xcol];
    }
    if (k + KS <= stop) {
      load_rows<BM, ROWS>(qa + k * args.A.ld, args.A.ld, va, swave * ROWS, da);
      load_rows<BN, ROWS>(qb + k * args.B.ld, args.B.ld, vb, swave * ROWS, db);
    } else if (HALF && k + KT == stop) {         // the last block, alone in its stage: the waves of its rows load it
      if (swave * ROWS < KT) {
        load_rows<BM, ROWS>(qa + k * args.A.ld, args.A.ld, va, swave * ROWS, da);
        load_rows<BN, ROWS>(qb + k * args.B.ld, args.B.ld, vb, swave * ROWS, db);
      }
    } else {                                        // the end is inside a block: through registers, zeros past it
#pragma unroll 1
      for (int e = threadIdx.x; e < KS * BM; e += NT) {
        const int r = e / BM, c = e % BM;
        da[r][c] = k + r < stop ? A[(k + r) * args.A.ld + (c < last_a ? c : last_a)] : 0.0f;
      }
#pragma unroll 1
      for (int e = threadIdx.x; e < KS * BN; e += NT) {
        const int r = e / BN, c = e % BN;
        db[r][c] = k + r < stop ? B[(k + r) * args.B.ld + (c < last_b ? c : last_b)] : 0.0f;
      }
    }
  };
  uint32_t max_a = 0u, max_b = 0u, max_x = 0u;
  // the stage's scales into LDS with their short-add verdicts, then the barrier once this wave's loads landed
  auto finish_stage = [&](int buf) __attribute__((always_inline)) {
    const int t = threadIdx.x;
#pragma unroll
    for (int q = 0; q < NBS; ++q) {
      uint32_t denies = 0u;
      if (t < BM + BN) {
        max_x = umax(max_x, f2u(xv[q]) & 0x7FFFFFFFu);
        denies = scale_denies(xv[q], fl.xs_lo, fl.xs_hi);
        if (t < BM) xs_a[buf][q][t] = xv[q];
        else xs_b[buf][q][t - BM] = xv[q];
      }
      const uint32_t dw = (__any((denies & 1u) != 0u) ? 1u : 0u) | (__any((denies & 2u) != 0u) ? 2u : 0u);
      if (lane == 0) denies_w[buf][q][wave] = dw;
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);             // vmcnt(0): the direct-to-LDS loads of this wave landed
    __syncthreads();
  };

  float C[TM][TN];
#pragma unroll
  for (int x = 0; x < TM; ++x)
#pragma unroll
    for (int y = 0; y < TN; ++y) C[x][y] = 0.0f;

  bool large = false;                               // some scale so far was above xs_hi
  // a stage of `blocks` blocks: their operand maxima read back from LDS, then the blocks reduced into C
  static_assert(KT % ROWS == 0 && KT * BN / 4 == NT, "a block is whole waves' rows and a float4 a thread");
  auto reduce_stage = [&](auto blocks, const float (&ca)[KS][BM], const float (&cb)[KS][BN], int buf)
                          __attribute__((always_inline)) {
    constexpr int BLOCKS = decltype(blocks)::value;
#pragma unroll
    for (int j = 0; j < BLOCKS; ++j) {
      const float4 qa = reinterpret_cast<const float4*>(&ca[0][0])[threadIdx.x + NT * j];
      const float4 qb = reinterpret_cast<const float4*>(&cb[0][0])[threadIdx.x + NT * j];
      max_a = umax(max_a, umax(umax(f2u(qa.x) & 0x7FFFFFFFu, f2u(qa.y) & 0x7FFFFFFFu),
                               umax(f2u(qa.z) & 0x7FFFFFFFu, f2u(qa.w) & 0x7FFFFFFFu)));
      max_b = umax(max_b, umax(umax(f2u(qb.x) & 0x7FFFFFFFu, f2u(qb.y) & 0x7FFFFFFFu),
                               umax(f2u(qb.z) & 0x7FFFFFFFu, f2u(qb.w) & 0x7FFFFFFFu)));
    }
    constexpr int BLOCKS_AT_ONCE = KIND == kE4Final || KIND == kE4 ? BLOCKS : 1;   // the others' code is long
#pragma unroll BLOCKS_AT_ONCE
    for (int q = 0; q < BLOCKS; ++q) {
      uint32_t denies = 0u;
#pragma unroll
      for (int v = 0; v < NWV; ++v) denies |= denies_w[buf][q][v];
      large = large || (denies & 2u) != 0u;
      const bool short_add = denies == 0u && !large;
      float scale[TM][TN];
      {
        float fa[TM];
        lds_row<TM>(&xs_a[buf][q][tm * TM], fa);
        float fb[TN];
        const float2 xb = *reinterpret_cast<const float2*>(&xs_b[buf][q][tn * TN]);
        fb[0] = xb.x; fb[1] = xb.y;
#pragma unroll
        for (int x = 0; x < TM; ++x)
#pragma unroll
          for (int y = 0; y < TN; ++y) scale[x][y] = fa[x] * fb[y];
      }
#pragma unroll
      for (int r0 = KT * q; r0 < KT * q + KT; r0 += SIZE) {
        float S[TM][TN];
#pragma unroll
        for (int i = 0; i < SIZE; ++i) {
          float a[TM];
          lds_row<TM>(&ca[r0 + i][tm * TM], a);
          const float2 b2 = *reinterpret_cast<const float2*>(&cb[r0 + i][tn * TN]);
          const float b[TN] = {b2.x, b2.y};
#pragma unroll
          for (int x = 0; x < TM; ++x)
#pragma unroll
            for (int y = 0; y < TN; ++y) S[x][y] = dp.step(S[x][y], a[x] * b[y], i);
        }
        // The sums stand here for every ladder but HW_FINAL's: the compiler sinks theirs into the tile add's branches,
        // with every operand kept in registers until there, and spills.
        if constexpr (KIND != kE4Final) {
#pragma unroll
          for (int x = 0; x < TM; ++x)
#pragma unroll
            for (int y = 0; y < TN; ++y) asm volatile("" : "+v"(S[x][y]));
        }
        if (short_add) {
#pragma unroll
          for (int x = 0; x < TM; ++x)
#pragma unroll
            for (int y = 0; y < TN; ++y) C[x][y] = dp.tile_add(C[x][y], S[x][y], scale[x][y]);
        } else {
#pragma unroll
          for (int x = 0; x < TM; ++x)
#pragma unroll
            for (int y = 0; y < TN; ++y) C[x][y] = dp.add(C[x][y], dp.tile(S[x][y], scale[x][y], false), true);
        }
      }
    }
  };

  // a tile made only of groups the caller does not need is written as +0 (through the epilogue), uncomputed
  if (args.skip && (args.order_skip ? marked : tile_skipped(args, z, m0, n0, BM, BN))) {
    if (threadIdx.x == 0) args.flags[(z * args.tiles_y + ty) * args.tiles_x + tx] = 0u;
    if (!args.c_end || n0 < args.c_end[z * args.kend_groups + m0 / 64])
      write_tile<TM, TN>(args, z, m0 + tm * TM, n0 + tn * TN, C);
    return;
  }
  // stages of NBS blocks up to `whole`, rows past `stop` zeros in the last of them; with HALF one block may be left
  const int64_t kst = (nb + NBS - 1) / NBS * KS, whole = HALF ? nb / NBS * KS : kst;
  constexpr std::integral_constant<int, NBS> kWholeStage{};
  if (kst > 0) {
    load_stage(0, sa0, sb0);
    finish_stage(0);
  }
  for (int64_t k0 = 0; k0 < whole; k0 += 2 * KS) {
    // even stage: buffer 0 reduced while stage k0 + KS lands in buffer 1; odd stage: the other way round
    const bool more1 = k0 + KS < kst;
    if (more1) load_stage(k0 + KS, sa1, sb1);
    reduce_stage(kWholeStage, sa0, sb0, 0);
    if (!more1) break;
    finish_stage(1);
    if (HALF && k0 + KS >= whole) break;         // the block left over
    const bool more2 = k0 + 2 * KS < kst;
    if (more2) load_stage(k0 + 2 * KS, sa0, sb0);
    reduce_stage(kWholeStage, sa1, sb1, 1);
    if (more2) finish_stage(0);
  }
  if (HALF && whole < kst) {
    const bool odd = (nb / NBS & 1) != 0;
    const float (&ha)[KS][BM] = odd ? sa1 : sa0;
    const float (&hb)[KS][BN] = odd ? sb1 : sb0;
    reduce_stage(std::integral_constant<int, 1>{}, ha, hb, odd ? 1 : 0);
  }

  // rows from `stop` on: exact only if A holds +-0 there and B and every remaining block scale are finite
  // (k_suffix_flags' bytes, as k_systolic_fast reads them); bit j for the tile's 32-column group j of A, then B
  constexpr int GT = BM / 32 + BN / 32;
  uint32_t bad = 0u;
  if (stop < K) {
    const int64_t s0 = stop / KT, ga = (M + 31) / 32, gb = (N + 31) / 32;
    for (int64_t i = threadIdx.x; i < (args.stages - s0) * GT; i += NT) {
      const int64_t st = s0 + i / GT;
      const int j = (int)(i % GT);
      bool b;
      if (j < BM / 32) {
        const int64_t g = m0 / 32 + j;
        b = g < ga && args.suf_a[(z * args.stages + st) * ga + g];
      } else {
        const int64_t g = n0 / 32 + (j - BM / 32);
        b = g < gb && args.suf_b[(z * args.stages + st) * gb + g];
      }
      bad |= b ? 1u << j : 0u;
    }
  }

  for (int off = 32; off > 0; off >>= 1) {
    max_a = umax(max_a, (uint32_t)__shfl_xor((int)max_a, off, 64));
    max_b = umax(max_b, (uint32_t)__shfl_xor((int)max_b, off, 64));
    max_x = umax(max_x, (uint32_t)__shfl_xor((int)max_x, off, 64));
    bad |= (uint32_t)__shfl_xor((int)bad, off, 64);
  }
  if (lane == 0) {
    red[0][wave] = max_a;
    red[1][wave] = max_b;
    red[2][wave] = max_x;
    red[3][wave] = bad;
  }
  __syncthreads();
  uint32_t wa = 0u, wb = 0u, wx = 0u, wbad = 0u;
#pragma unroll
  for (int v = 0; v < NWV; ++v) {
    wa = umax(wa, red[0][v]);
    wb = umax(wb, red[1][v]);
    wx = umax(wx, red[2][v]);
    wbad |= red[3][v];
  }
  const bool ok = wbad == 0u && wa < kFastAMaxBits && wb < 0x7F800000u && wx < 0x7F800000u &&
                  u2f(wa) * u2f(wb) <= args.fast_prod_max;
  // the flag: bit 0, the general kernel computes the tile; bits 1..GT, which groups' left-out rows failed their
  // check (piece_kstop)
  if (threadIdx.x == 0) args.flags[(z * args.tiles_y + ty) * args.tiles_x + tx] = ok ? 0u : 1u | (wbad << 1);
  if (!ok) return;
  write_tile<TM, TN>(args, z, m0 + tm * TM, n0 + tn * TN, C);
}

// The launch of a grid of a.fbm x a.fbm tiles.
template <int KIND, int SIZE, bool BF16_LAST, bool WHOLE>
void launch_tile_shape(dim3 grid, const SysArgs& a, const FastLanes& fl, hipStream_t st) {
  if (a.fbm == 64) k_systolic_tile<KIND, SIZE, BF16_LAST, 64, WHOLE><<<grid, 512, 0, st>>>(a, fl);
  else k_systolic_tile<KIND, SIZE, BF16_LAST, 32, WHOLE><<<grid, 256, 0, st>>>(a, fl);
}
template <int KIND, int SIZE, bool BF16_LAST>
void launch_tile_ladder(dim3 grid, const SysArgs& a, const FastLanes& fl, hipStream_t st) {
  if constexpr (KIND == kE4Final) {
    auto aligned = [](const Operand& o) {
      return o.ld % 4 == 0 && o.batch % 4 == 0 && reinterpret_cast<uintptr_t>(o.p) % 16 == 0;
    };
    // a half-full last stage of 64 rows is more than the instance saves (3 %) below 1024 rows
    const bool half = a.fbm == 64 && a.K % 64 > 0 && a.K % 64 <= 32 && a.K < 1024;
    if (a.M % a.fbm == 0 && a.N % a.fbm == 0 && !half && aligned(a.A) && aligned(a.B))
      return launch_tile_shape<KIND, SIZE, BF16_LAST, true>(grid, a, fl, st);
  }
  launch_tile_shape<KIND, SIZE, BF16_LAST, false>(grid, a, fl, st);
}
template <int KIND, bool BF16_LAST>
void launch_tile_size(dim3 grid, const SysArgs& a, const FastLanes& fl, hipStream_t st) {
  switch (a.size) {
    case 4: launch_tile_ladder<KIND, 4, BF16_LAST>(grid, a, fl, st); break;
    case 8: launch_tile_ladder<KIND, 8, BF16_LAST>(grid, a, fl, st); break;
    case 16: launch_tile_ladder<KIND, 16, BF16_LAST>(grid, a, fl, st); break;
    default: launch_tile_ladder<KIND, 32, BF16_LAST>(grid, a, fl, st); break;
  }
}

}  // namespace mxq_sys
