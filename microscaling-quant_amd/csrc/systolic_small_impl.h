// Systolic products of few outputs (a token or some tens of them, one attention step): k_systolic_small.
//
// An output's chain is sequential over K only in its tile adds: every reduction of `size` rows starts from S = 0, so
// the reductions' sums do not depend on one another.  With few outputs the tile kernels leave most of the chip idle
// and each thread walks all of K; here the waves of a workgroup share K between them instead.  A workgroup holds TM
// rows x CW columns of C (CW = 64, 32 or 16).  In a round its waves compute one reduction a lane (U of them), each
// lane its own column and, when CW < 64, its own reduction of the wave's 64 / CW; the scaled sums (tiles) go to LDS;
// then one thread per output adds the round's tiles in the reference's order.  B is read straight into registers
// (each lane's column, used by its TM rows only), A is staged through LDS, and the next round's operands are loaded
// while this one is computed.
//
// The arithmetic is the tile kernels' fast datapath (Datapath), under the same check of the operands read.  Where it
// fails (after the first round of a long K, or at the end), the workgroup computes its outputs by the general rule itself:
// a call is one launch, without flags.  Operands all past the check (E4M3 codes to 448 under HW_FINAL), a whole call
// against the tile kernel's and the general kernel's after it: 1 x 4096 outputs, K = 4096: 0.22 ms against 7.9; 8 x 4096:
// 1.0 against 10.0; 64 x 4096, K = 2048: 2.0 against 5.1; MXGEMMINI e5m6 lanes 512 x 2048, K = 2048: 13.0 against the
// general kernel's 12.8, MXQUANT(4, 3): 3.2 against 3.0 (36 and 3.7 with each output's K in one thread).
//
// Bound by VALU issue (8.0 to 8.6 instructions a MAC, the datapath's 7 among them) and, for one row, by reading B.
// HW_FINAL, a whole call against the tile kernel's: 1 x 5632 outputs, K = 2048: 23 us against 207 (45 MB of codes);
// 8 x 4096, K = 4096: 45 against 406; 64 x 4096, K = 4096: 199 against 368; 128 x 4096, K = 4096: 337 against 392.
// MXQUANT(4, 3) under HW_FINAL, 512 x 2048, K = 2048: 0.641 ms against the general kernel's 3.07; MXGEMMINI e5m6 lanes
// 0.47 against 12.9.
#pragma once

#include "systolic_common.h"

namespace mxq_sys {

// NW waves a workgroup, U reductions a lane and round.
template <int KIND, int SIZE, bool BF16_LAST, int TM, int U, int NW>
__global__ void __launch_bounds__(64 * NW, 4) k_systolic_small(const SysArgs args, const FastLanes fl, int log_cw,
                                                               const mxq::DivU31 per_block) {
  constexpr int NT = 64 * NW;
  constexpr int MAXSUB = TM == 16 ? 1 : 4;          // reductions side by side in a wave: 64 / CW
  constexpr int SLOTS = NW * MAXSUB * U;            // reductions of a round, at most
  constexpr int APAD = SIZE * TM + 4;               // a reduction's rows of A in LDS, a bank off the next one's
  __shared__ __align__(16) float sa[SLOTS * APAD];
  __shared__ float xs[SLOTS * TM];                  // a reduction's scales of A
  __shared__ float tiles[2][NW * U * 64 * TM];
  __shared__ uint32_t large_w;                      // some scale so far was above xs_hi
  __shared__ uint32_t inexact_w[2];                 // some scale of A in the round denies the short tile (0: none)
  __shared__ uint32_t red[3][NW];
  const Datapath<KIND, SIZE, BF16_LAST> dp{fl};
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cw = 1 << log_cw, subs = 64 >> log_cw;
  const int col = lane & (cw - 1), sub = lane >> log_cw;
  const int64_t z = blockIdx.z, m0 = (int64_t)blockIdx.y * TM, n0 = (int64_t)blockIdx.x << log_cw;
  const float* A = args.A.p + z * args.A.batch + m0;
  const float* B = args.B.p + z * args.B.batch + n0;
  const float* XA = args.XA.p + z * args.XA.batch + m0;
  const float* XB = args.XB.p + z * args.XB.batch + n0;
  const int64_t M = args.M, N = args.N;
  const int K = (int)args.K;                        // below 2^30 (takes_small)
  const int rows_in = M - m0 < TM ? (int)(M - m0) : TM;
  const bool col_in = n0 + col < N;
  const int nred = (K + SIZE - 1) / SIZE;
  const int round = NW * subs * U;                  // reductions a round

  // this thread's output in the tile adds
  const int om = threadIdx.x >> log_cw, oc = threadIdx.x & (cw - 1);
  const bool owner = om < TM;
  float C[TM * 64 > NT ? TM * 64 / NT : 1];         // outputs per thread: rows om, om + NT / CW, ...
  constexpr int PER = TM * 64 > NT ? TM * 64 / NT : 1;
#pragma unroll
  for (int j = 0; j < PER; ++j) C[j] = 0.0f;

  // the caller's skip map: a tile inside marked groups only is +0 through the epilogue
  bool skipped = args.skip != nullptr;
  if (skipped) {
    const uint8_t* sk = args.skip + z * args.skip_rows * args.skip_cols;
    const int64_t c1 = n0 + cw - 1 < N ? n0 + cw - 1 : N - 1;
    skipped = sk[m0 / 32 * args.skip_cols + n0 / 32] != 0 && sk[m0 / 32 * args.skip_cols + c1 / 32] != 0;
  }

  uint32_t max_a = 0u, max_b = 0u, max_x = 0u;
  if (!skipped) {
    if (threadIdx.x < 2) inexact_w[threadIdx.x] = 0u;
    if (threadIdx.x == 0) large_w = 0u;
    // A's part of a round: element (row, column) e = thread + j * NT, so a thread keeps its column and its rows lie
    // NT / TM apart; only the first `round` reductions' rows (a uniform test a step)
    constexpr int A_PER = (SLOTS * SIZE * TM + NT - 1) / NT, X_PER = (SLOTS * TM + NT - 1) / NT, ROWS = NT / TM;
    static_assert(ROWS % SIZE == 0 || SIZE % ROWS == 0, "whole reductions a step");
    float av[A_PER], xv[X_PER], b[U][SIZE], bn[U][SIZE], xb[U], xbn[U];
    const int arow = threadIdx.x / TM, acol = threadIdx.x % TM;
    const bool acol_in = acol < rows_in;
    const uint32_t a_off = (uint32_t)arow * (uint32_t)args.A.ld + (uint32_t)(acol_in ? acol : 0);
    auto load_a = [&](int r0) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < A_PER; ++j) {
        if (j * ROWS >= round * SIZE) break;
        const int k0 = r0 * SIZE + j * ROWS;
        const float* q = A + (int64_t)k0 * args.A.ld;
        float v;
        if (k0 + ROWS <= K) {
          v = q[a_off];
          v = acol_in ? v : 0.0f;
        } else {
          const bool in = acol_in && k0 + arow < K;
          v = A[in ? (int64_t)(k0 + arow) * args.A.ld + acol : 0];
          v = in ? v : 0.0f;
        }
        av[j] = v;
      }
#pragma unroll
      for (int j = 0; j < X_PER; ++j) {
        if (j * NT >= round * TM) break;
        const int s = (threadIdx.x + j * NT) / TM, r = r0 + s;
        const bool in = s < round && r < nred && acol_in;
        const float v = XA[(in ? mxq::divu31(r, per_block) : 0u) * args.XA.ld + (in ? acol : 0)];
        xv[j] = in ? v : 0.0f;
      }
    };
    // a lane's rows: a uniform row address plus a 32-bit offset of its own (below 2^32 bytes: takes_small)
    const uint32_t lane_off = (uint32_t)(sub * SIZE) * (uint32_t)args.B.ld + (uint32_t)col;
    auto load_b = [&](int r0, float (&v)[U][SIZE], float (&x)[U]) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int rw = r0 + (wave * U + u) * subs, r = rw + sub, k = r * SIZE;
        const float* q = B + (int64_t)rw * SIZE * args.B.ld;
        if ((rw + subs) * SIZE <= K && n0 + cw <= N) {
#pragma unroll
          for (int i = 0; i < SIZE; ++i) v[u][i] = (q + i * args.B.ld)[lane_off];
        } else {
#pragma unroll
          for (int i = 0; i < SIZE; ++i) {
            const bool in = col_in && k + i < K;
            const float t = B[(in ? k + i : 0) * args.B.ld + (in ? col : 0)];
            v[u][i] = in ? t : 0.0f;
          }
        }
        const bool in = col_in && r < nred;
        const float t = XB[(in ? mxq::divu31(r, per_block) : 0u) * args.XB.ld + (in ? col : 0)];
        x[u] = in ? t : 0.0f;
      }
    };
    // the workgroup's verdict on what it has read, as the tile kernels'
    auto verdict = [&]() __attribute__((always_inline)) {
      for (int off = 32; off > 0; off >>= 1) {
        max_a = umax(max_a, (uint32_t)__shfl_xor((int)max_a, off, 64));
        max_b = umax(max_b, (uint32_t)__shfl_xor((int)max_b, off, 64));
        max_x = umax(max_x, (uint32_t)__shfl_xor((int)max_x, off, 64));
      }
      if (lane == 0) {
        red[0][wave] = max_a;
        red[1][wave] = max_b;
        red[2][wave] = max_x;
      }
      __syncthreads();
      uint32_t wa = 0u, wb = 0u, wx = 0u;
#pragma unroll
      for (int v = 0; v < NW; ++v) {
        wa = umax(wa, red[0][v]);
        wb = umax(wb, red[1][v]);
        wx = umax(wx, red[2][v]);
      }
      return wa < kFastAMaxBits && wb < 0x7F800000u && wx < 0x7F800000u && u2f(wa) * u2f(wb) <= args.fast_prod_max;
    };
    bool ok = true;
    load_a(0);
    load_b(0, b, xb);
    __syncthreads();                                // large_w cleared
    int buf = 0;
    for (int r0 = 0; r0 < nred; r0 += round) {
      uint32_t denies = 0u;
#pragma unroll
      for (int j = 0; j < A_PER; ++j) {
        if (j * ROWS >= round * SIZE) break;
        const int row = arow + j * ROWS;
        max_a = umax(max_a, f2u(av[j]) & 0x7FFFFFFFu);
        if (row < SLOTS * SIZE) sa[row / SIZE * APAD + row % SIZE * TM + acol] = av[j];
      }
#pragma unroll
      for (int j = 0; j < X_PER; ++j) {
        if (j * NT >= round * TM) break;
        const int e = threadIdx.x + j * NT;
        max_x = umax(max_x, f2u(xv[j]) & 0x7FFFFFFFu);
        denies |= scale_denies(xv[j], fl.xs_lo, fl.xs_hi);
        if (e < SLOTS * TM) xs[e] = xv[j];
      }
      if (denies & 1u) inexact_w[buf] = 1u;         // every writer writes the same word
      __syncthreads();
      const bool a_exact = inexact_w[buf] == 0u;
      if (threadIdx.x == 0) inexact_w[buf ^ 1] = 0u;   // read a barrier ago, written again after the next
      const bool more = r0 + round < nred;
      if (more) {
        load_a(r0 + round);
        load_b(r0 + round, bn, xbn);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int slot = (wave * U + u) * subs + sub;
        const float* as = &sa[slot * APAD];
        float S[TM];
#pragma unroll
        for (int i = 0; i < SIZE; ++i) {
          max_b = umax(max_b, f2u(b[u][i]) & 0x7FFFFFFFu);
          float a[TM];
          if constexpr (TM >= 4) {
#pragma unroll
            for (int q = 0; q < TM / 4; ++q) {
              const float4 t = *reinterpret_cast<const float4*>(as + i * TM + 4 * q);
              a[4 * q] = t.x; a[4 * q + 1] = t.y; a[4 * q + 2] = t.z; a[4 * q + 3] = t.w;
            }
          } else {
#pragma unroll
            for (int x = 0; x < TM; ++x) a[x] = as[i * TM + x];
          }
#pragma unroll
          for (int x = 0; x < TM; ++x) S[x] = dp.step(S[x], a[x] * b[u][i], i);
        }
        // the sums stand here: sunk into the tile's branches they keep every operand in registers until there
#pragma unroll
        for (int x = 0; x < TM; ++x) asm volatile("" : "+v"(S[x]));
        max_x = umax(max_x, f2u(xb[u]) & 0x7FFFFFFFu);
        const uint32_t dn = scale_denies(xb[u], fl.xs_lo, fl.xs_hi);
        denies |= dn;
        const bool short_add = a_exact && __all((dn & 1u) == 0u) != 0;
        float* t = &tiles[buf][slot * TM * cw + col];
        if (short_add) {
#pragma unroll
          for (int x = 0; x < TM; ++x) t[x * cw] = dp.tile(S[x], xs[slot * TM + x] * xb[u], true);
        } else {
#pragma unroll
          for (int x = 0; x < TM; ++x) t[x * cw] = dp.tile(S[x], xs[slot * TM + x] * xb[u], false);
        }
      }
      if (denies & 2u) large_w = 1u;
      __syncthreads();
      // this round's tiles in the reference's order
      const bool large = large_w != 0u;
      const int cnt = nred - r0 < round ? nred - r0 : round;
      if (owner) {
#pragma unroll
        for (int j = 0; j < PER; ++j) {
          const float* t = &tiles[buf][threadIdx.x + j * NT];
          if (large) {
            for (int s = 0; s < cnt; ++s) C[j] = dp.add(C[j], t[s * TM * cw], true);
          } else {
#pragma unroll 8
            for (int s = 0; s < cnt; ++s) C[j] = dp.add(C[j], t[s * TM * cw], false);
          }
        }
      }
      // operands past the datapath are so in their first rows as a rule: the rest of a long K is left to the general rule
      // (not by the four-row tiles, whose loop takes 2 to 4 % longer with it; the others' does not)
      if (TM != 4 && r0 == 0 && nred > 4 * round && !(ok = verdict())) break;
      if (more) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
          for (int i = 0; i < SIZE; ++i) b[u][i] = bn[u][i];
          xb[u] = xbn[u];
        }
      }
      buf ^= 1;                                     // the next round's tiles are written two barriers from here
    }
    if (ok) ok = verdict();
    if (!ok) {
      // Any codes and scales: the general rule, the reductions shared among the waves as above.  B is read again (the
      // next row's value while a row is computed), A through LDS.  Its loads are its own and its rows are taken one after
      // another: with the loads above and the rows interleaved it is 5 to 15 % faster, and the registers that takes cost
      // the datapath above 1 to 5 % (as it is, from -3 to 3 % by ladder, none on average).
#pragma unroll
      for (int j = 0; j < PER; ++j) C[j] = 0.0f;
#pragma unroll 1
      for (int r0 = 0; r0 < nred; r0 += round) {
        __syncthreads();                            // the tiles before are added, A's rows before used
#pragma unroll 1
        for (int e = threadIdx.x; e < round * SIZE * TM; e += NT) {
          const int row = e / TM, x = e % TM;
          const bool in = x < rows_in && r0 * SIZE + row < K;
          const float v = A[in ? (int64_t)(r0 * SIZE + row) * args.A.ld + x : 0];
          sa[row / SIZE * APAD + row % SIZE * TM + x] = in ? v : 0.0f;
        }
#pragma unroll 1
        for (int e = threadIdx.x; e < round * TM; e += NT) {
          const int r = r0 + e / TM, x = e % TM;
          const bool in = x < rows_in && r < nred;
          const float v = XA[(in ? mxq::divu31(r, per_block) : 0u) * args.XA.ld + (in ? x : 0)];
          xs[e] = in ? v : 0.0f;
        }
        __syncthreads();
#pragma unroll 1
        for (int u = 0; u < U; ++u) {
          const int slot = (wave * U + u) * subs + sub, r = r0 + slot, k0 = r * SIZE;
          const float* as = &sa[slot * APAD];
          auto b_at = [&](int k) { return B[(k < K && col_in ? (int64_t)k * args.B.ld + col : 0)]; };
          float S[TM];
#pragma unroll
          for (int x = 0; x < TM; ++x) S[x] = 0.0f;
          float next = b_at(k0);
#pragma unroll 1
          for (int i = 0; i < SIZE; ++i) {
            const float v = next;
            next = b_at(k0 + i + 1);
            if (k0 + i >= K) break;                 // a reduction cut short by K's end ends as it stands
#pragma unroll
            for (int x = 0; x < TM; ++x) {
              asm volatile("" : "+v"(S[x]));        // this row after the one before
              S[x] = gen_acc(S[x], gen_product(as[i * TM + x], v, args.ar), args.lane_e[i], args.lane_m[i], args.ar);
            }
          }
          const bool in = r < nred && col_in;
          const float x_b = XB[(in ? mxq::divu31(r, per_block) : 0u) * args.XB.ld + (in ? col : 0)];
#pragma unroll
          for (int x = 0; x < TM; ++x) tiles[0][slot * TM * cw + col + x * cw] = S[x] * (xs[slot * TM + x] * x_b);
        }
        __syncthreads();
        const int cnt = nred - r0 < round ? nred - r0 : round;
        if (owner) {
#pragma unroll
          for (int j = 0; j < PER; ++j)
#pragma unroll 1
            for (int s = 0; s < cnt; ++s) C[j] = gen_tile(C[j], tiles[0][threadIdx.x + j * NT + s * TM * cw], args.ar);
        }
      }
    }
  }
  if (!owner || n0 + oc >= N) return;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int64_t mm = om + j * (NT >> log_cw);
    if (mm >= rows_in) continue;
    const float* row = args.epi_on ? epi_row(args, z, m0 + mm) : nullptr;
    args.C[z * args.batch_c + (m0 + mm) * args.ldc + n0 + oc] =
        args.epi_on ? epi_apply(args, row, n0 + oc, C[j]) : C[j];
  }
}

template <int KIND, int SIZE, bool BF16_LAST, int TM, int U, int NW>
void launch_small_tile(const SysArgs& a, const FastLanes& fl, const SmallTile& t, int64_t count, hipStream_t st) {
  const dim3 grid((unsigned)((a.N + (1 << t.log_cw) - 1) >> t.log_cw), (unsigned)mxq::ceil_div(a.M, TM), (unsigned)count);
  k_systolic_small<KIND, SIZE, BF16_LAST, TM, U, NW><<<grid, 64 * NW, 0, st>>>(
      a, fl, t.log_cw, mxq::make_divu31((uint32_t)(a.block_size / SIZE)));
}

// HW_FINAL's ladders have every tile; the others two (SmallTile.rows 4 with sixteen waves, 8 with eight).
template <int KIND, int SIZE, bool BF16_LAST>
void launch_small_ladder(const SysArgs& a, const FastLanes& fl, const SmallTile& t, int64_t count, hipStream_t st) {
  if constexpr (KIND == kE4Final || KIND == kMxqFinal) {
    if (t.rows == 1) return launch_small_tile<KIND, SIZE, BF16_LAST, 1, 2, 16>(a, fl, t, count, st);
    if (t.rows == 16) return launch_small_tile<KIND, SIZE, BF16_LAST, 16, 1, 8>(a, fl, t, count, st);
    if (t.rows == 8 && t.waves == 16) return launch_small_tile<KIND, SIZE, BF16_LAST, 8, 1, 16>(a, fl, t, count, st);
  }
  if (t.rows == 4) launch_small_tile<KIND, SIZE, BF16_LAST, 4, 1, 16>(a, fl, t, count, st);
  else launch_small_tile<KIND, SIZE, BF16_LAST, 8, 1, 8>(a, fl, t, count, st);
}

template <int KIND, bool BF16_LAST>
void launch_small_size(const SysArgs& a, const FastLanes& fl, const SmallTile& t, int64_t count, hipStream_t st) {
  switch (a.size) {
    case 4: launch_small_ladder<KIND, 4, BF16_LAST>(a, fl, t, count, st); break;
    case 8: launch_small_ladder<KIND, 8, BF16_LAST>(a, fl, t, count, st); break;
    case 16: launch_small_ladder<KIND, 16, BF16_LAST>(a, fl, t, count, st); break;
    default: launch_small_ladder<KIND, 32, BF16_LAST>(a, fl, t, count, st); break;
  }
}

}  // namespace mxq_sys
