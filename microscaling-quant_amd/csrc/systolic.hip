// The systolic PE column on gfx950: Y = A^T B from MX codes and scales, every output element its own strictly
// sequential chain in the reference's order (mxq/matmul/_systolic.py:23-62):
//   for each block of K: scale map X_A[g] (x) X_B[g]
//     for each reduction of `size` k: S = 0; S = acc_add(S, product(a_k, b_k), lane k % size)
//       C = tile_add(C, S * scale)
// Parallelism is over M x N (and a batch of independent problems); nothing is split along K, so no summation
// order changes.  The work is VALU (integer and float32 bit manipulation), not MFMA: the matrix cores'
// accumulation would not round where the datapath does.
//
// Operands are strided and batched: element (r, c) of problem z of an operand sits at base + z*batch + r*ld + c.
//
// The fast datapaths (systolic_common.h: Datapath), for MXGEMMINI's e4 ladders (HW_FINAL's constants as literals), its
// ladders of wider lanes and MXQUANT's, are exact when the codes and scales they read are finite, max|a| < 2^100 and
// max|a| * max|b| is under the ladder's bound.  Their kernels:
//   k_systolic_tile   (systolic_tile_impl.h) tiles of 64 x 64 or 32 x 32 outputs.  While it computes, each workgroup
//                     keeps the largest |a|, |b| and scale it has read; if they allow it writes its tile and a 0 flag,
//                     otherwise only a 1 flag.
//   k_systolic_small  (systolic_small_impl.h) products of few outputs, whose waves share K; a workgroup whose operands
//                     are refused computes its outputs by the general rule itself.
//   k_systolic_fast   e4 ladders with blocks of other sizes than 32, in units of the lane's subnormal step:
//                     MXGEMMINI with size in {4, 8, 16, 32}, lanes (4, m <= 9) of non-decreasing m, optionally a
//                     last (8, 7) lane, prod_m <= every e4 lane's m (checked on the host).  A's rows are staged into
//                     LDS times 2^(6 + m) of their lane, so
//                        p = rint(trunc(a' * b))      float32 multiply, mask the dropped significand bits, round to
//                                                     an integer = lane(p) (the flush below 2^prod_floor is under
//                                                     half a step, so it is subsumed)
//                        S = rne_m(S + p)             the sum is an exact integer below 2^24; RNE at m fraction bits
//                     and the sum is rescaled by 2 when m steps up.  The bf16 lane and the tile add are one float32
//                     add of two values of at most 8 significant bits followed by RNE to bf16, which equals the
//                     reference's exact add with one rounding (double rounding through 24 bits is harmless for
//                     8-bit operands: 24 >= 2*8 + 1).  Its check and flags are k_systolic_tile's.
//   k_systolic_gen    the full per-step rule for any codes, any lanes (e <= 8), MXGEMMINI or MXQUANT, NaN, Inf,
//                     saturation and overflow included.  After a tile kernel its flagged form
//                     (k_systolic_gen_flagged) computes only the tiles whose flag is 1; alone (no fast datapath, or
//                     forced) it computes everything.
#include <algorithm>
#include <cmath>
#include <mutex>

#include "mxq_common.h"
#include "mxq_numerics.h"
#include "systolic_common.h"

namespace {

using namespace mxq_red;
using namespace mxq_sys;

constexpr int64_t kInnerLd = int64_t(1) << 26;     // row strides below this keep 32 * ld in a 32-bit offset

// Whether the rows of 32-row stage s may be left out of a reduction that ends before them, per 32-column
// group: of A only where every code is +-0 (0 * b = +-0 adds nothing), and only if every block scale holding
// those rows is finite; of B where codes and those scales are finite (0 * Inf would have made a NaN).  A byte
// per answer, 1 = may not.  A's groups are checked only at stages at or past their kstop (no tile reads the
// others).  One workgroup per stage and 256 columns (the first x blocks A's, the rest B's): a lane reads 4
// adjacent columns of 8 rows, so each row is read as one 1 KB piece.  With the caller's bytes for A
// (a.a_live), the launch has B's workgroups only.
constexpr int kSufCols = 256;
__global__ void __launch_bounds__(256) k_suffix_flags(const SysArgs a, int64_t ga, int64_t gb, uint8_t* fa,
                                                      uint8_t* fb) {
  __shared__ uint32_t bad_g[kSufCols / 32];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t s = blockIdx.y, z = blockIdx.z, xa = a.a_live ? 0 : (a.M + kSufCols - 1) / kSufCols;
  const bool is_a = (int64_t)blockIdx.x < xa;
  const int64_t c0 = (is_a ? (int64_t)blockIdx.x : (int64_t)blockIdx.x - xa) * kSufCols;
  if (threadIdx.x < kSufCols / 32) bad_g[threadIdx.x] = 0u;
  const Operand& op = is_a ? a.A : a.B;
  const Operand& xo = is_a ? a.XA : a.XB;
  const int64_t L = is_a ? a.M : a.N, K = a.K;
  const float* P = op.p + z * op.batch;
  const float* X = xo.p + z * xo.batch;
  const int64_t c = c0 + 4 * lane;                  // this lane's 4 columns, inside one 32-column group
  const bool needed = c < L && (!is_a || KT * s >= tile_kstop(a, z, c));
  bool bad = false;
  if (needed) {
    const bool vec = vec_ok(op, P) && c + 3 < L;
    float v[8][4];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int64_t r = KT * s + wave * 8 + i;
      const float* q = P + r * op.ld + c;
      if (r >= K) {
        v[i][0] = v[i][1] = v[i][2] = v[i][3] = 0.0f;
      } else if (vec) {
        const float4 t = *reinterpret_cast<const float4*>(q);
        v[i][0] = t.x; v[i][1] = t.y; v[i][2] = t.z; v[i][3] = t.w;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[i][e] = c + e < L ? q[e] : 0.0f;
      }
    }
    uint32_t mx = 0u, mxs = 0u;
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) mx = umax(mx, f2u(v[i][e]) & 0x7FFFFFFFu);
    if (wave == 0) {
      const int64_t r_end = (KT * s + KT < K ? KT * s + KT : K) - 1, bs = a.block_size;
      for (int64_t gg = KT * s / bs; gg <= r_end / bs; ++gg)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (c + e < L) mxs = umax(mxs, f2u(X[gg * xo.ld + c + e]) & 0x7FFFFFFFu);
    }
    bad = mxs >= 0x7F800000u || (is_a ? mx != 0u : mx >= 0x7F800000u);
  }
  const uint64_t m = __ballot(bad);
  __syncthreads();   // bad_g cleared
  if (lane < kSufCols / 32 && ((m >> (8 * lane)) & 0xFFu)) atomicOr(&bad_g[lane], 1u);
  __syncthreads();
  if (threadIdx.x < kSufCols / 32) {
    const int64_t g = c0 / 32 + threadIdx.x;
    if (g < (is_a ? ga : gb)) (is_a ? fa : fb)[(z * a.stages + s) * (is_a ? ga : gb) + g] = bad_g[threadIdx.x] ? 1u : 0u;
  }
}

// The fast kernel's dispatch order under the caller's hints: tiles by descending work (stages to reduce),
// skipped tiles (+0 writes) last.  Workgroups are handed to the XCDs and their shader engines in turn as their
// ids rise, and a later one waits for an earlier one's slot.  In the grid's own order a causal triangle gives
// the engines owning the low tile columns a whole row's work (skipping half the tiles then saves little), and
// k_end's row-dependent work lands unevenly on them too.  Sorted by work, each run of consecutive ids carries
// about equal work to every engine, heaviest first.  Two launches: k_tile_bucket gives every position its work
// bucket (one stage wide) over the whole grid, then k_tile_order, one workgroup, counting-sorts the positions.
constexpr int kOrderThreads = 1024, kOrderBuckets = 2048;

// Dispatch position p -> its tile in the grid's own order (rows last first); 32-bit: the host launches the
// order kernel only while every position fits.
__device__ __forceinline__ uint32_t grid_tile(const SysArgs& a, uint32_t p, uint32_t& z, uint32_t& ty,
                                              uint32_t& tx) {
  const uint32_t nx = (uint32_t)a.tiles_x, ny = (uint32_t)a.tiles_y;
  const uint32_t zy = p / nx;
  tx = p - zy * nx;
  z = zy / ny;
  ty = ny - 1u - (zy - z * ny);
  return (z * ny + ty) * nx + tx;
}


// Each dispatch position's work bucket (0: skipped; else 1 + stages to reduce, the last bucket holding
// everything longer) into `bucket`, one thread per position over the whole grid.
__global__ void __launch_bounds__(256) k_tile_bucket(const SysArgs a, uint32_t total, uint16_t* bucket) {
  const uint32_t p = blockIdx.x * 256u + threadIdx.x;
  if (p >= total) return;
  uint32_t z, ty, tx;
  grid_tile(a, p, z, ty, tx);
  const int64_t m0 = (int64_t)ty * a.fbm, n0 = (int64_t)tx * a.fbn;
  if (a.skip && tile_skipped(a, z, m0, n0, a.fbm, a.fbn)) {
    bucket[p] = 0;
    return;
  }
  const int64_t st = tile_kstop(a, z, m0) / KT;
  bucket[p] = (uint16_t)(1 + (st < kOrderBuckets - 2 ? st : kOrderBuckets - 2));
}

// The counting sort of the positions by bucket, heaviest first, in one workgroup: sixteen adjacent positions'
// buckets per thread per pass (two 16-byte loads).  Adjacent positions mostly share a bucket (a row of tiles has
// one, skipped tiles aside), so a thread takes its sixteen as runs of equal buckets and makes one LDS atomic
// per run, all issued before any result is used: the pass waits on one atomic's latency, where an atomic per
// position, each waiting on the one before, kept the single workgroup waiting for tens of microseconds.
constexpr int kOrderRun = 16;
constexpr uint32_t kNoBucket = 0xFFFFu;           // a position past the grid

// Each run of equal buckets among b (run starts at u when u == 0 or b[u] != b[u - 1]) adds its length to
// cur[bucket]; with `place`, pos[u] gets the position's place in its bucket (the run's base from the atomic,
// plus its index in the run).  Positions of bucket kNoBucket take no part.
template <bool PLACE>
__device__ __forceinline__ void count_runs(uint32_t* cur, const uint16_t (&b)[kOrderRun], uint32_t (&pos)[kOrderRun]) {
  uint32_t len[kOrderRun];
  len[kOrderRun - 1] = 1u;
#pragma unroll
  for (int u = kOrderRun - 2; u >= 0; --u) len[u] = b[u] == b[u + 1] ? len[u + 1] + 1u : 1u;
  uint32_t base[kOrderRun];
#pragma unroll
  for (int u = 0; u < kOrderRun; ++u) {
    const bool start = (u == 0 || b[u] != b[u - 1]) && b[u] != kNoBucket;
    base[u] = 0u;
    if (start) {
      if constexpr (PLACE) base[u] = atomicAdd(&cur[b[u]], len[u]);
      else atomicAdd(&cur[b[u]], len[u]);
    }
  }
  if constexpr (PLACE) {
#pragma unroll
    for (int u = 0; u < kOrderRun; ++u) pos[u] = (u == 0 || b[u] != b[u - 1]) ? base[u] : pos[u - 1] + 1u;
  }
}

// With STAGE (total <= kOrderStage), the positions' buckets stay in registers between the two passes (one read
// of them), and the order is placed in LDS and then written out in runs of consecutive positions (placed straight
// into global memory, one store instruction's lanes land 16 places apart).  Each thread's 16 adjacent positions
// step their tile coordinates along the row instead of dividing for each.
constexpr uint32_t kOrderStage = 36864;            // 144 KiB of LDS beside the 8 KiB of bucket counters

template <bool STAGE>
__global__ void __launch_bounds__(kOrderThreads) k_tile_order(const SysArgs a, uint32_t total,
                                                              const uint16_t* __restrict__ bucket, uint32_t* order) {
  constexpr int PB = kOrderBuckets / kOrderThreads;
  static_assert(PB * kOrderThreads == kOrderBuckets, "whole buckets per thread");
  constexpr uint32_t stride = (uint32_t)kOrderThreads * kOrderRun;
  constexpr int SI = STAGE ? (int)((kOrderStage + stride - 1) / stride) : 1;   // passes held in registers
  __shared__ uint32_t cur[kOrderBuckets];
  __shared__ uint32_t wsum[kOrderThreads / 64];
  __shared__ uint32_t stage[STAGE ? kOrderStage : 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int b = threadIdx.x; b < kOrderBuckets; b += kOrderThreads) cur[b] = 0u;
  auto load_run = [&](uint32_t p0, uint16_t (&b)[kOrderRun]) {
    if (p0 + kOrderRun <= total) {
      const uint4* q = reinterpret_cast<const uint4*>(bucket + p0);   // p0 is a multiple of 16: 32-byte aligned
      const uint4 lo = q[0], hi = q[1];
      const uint32_t w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        b[2 * u] = (uint16_t)(w[u] & 0xFFFFu);
        b[2 * u + 1] = (uint16_t)(w[u] >> 16);
      }
    } else {
#pragma unroll
      for (int u = 0; u < kOrderRun; ++u) b[u] = p0 + u < total ? bucket[p0 + u] : (uint16_t)kNoBucket;
    }
  };
  // pass 2's placement of positions p0 .. p0 + 15: tiles from one division, then stepped
  const uint32_t nx = (uint32_t)a.tiles_x, ny = (uint32_t)a.tiles_y;
  auto place = [&](uint32_t p0, const uint16_t (&b)[kOrderRun]) __attribute__((always_inline)) {
    uint32_t pos[kOrderRun];
    count_runs<true>(cur, b, pos);
    uint32_t z, ty, tx;
    uint32_t t = grid_tile(a, p0, z, ty, tx);
#pragma unroll
    for (int u = 0; u < kOrderRun; ++u) {
      if (p0 + u < total) {
        const uint32_t e = t | (a.order_skip && b[u] == 0 ? 0x80000000u : 0u);
        if constexpr (STAGE) stage[pos[u]] = e;
        else order[pos[u]] = e;
      }
      if (tx + 1u < nx) {                           // the next position: the next tile of the row, or of the
        ++tx;                                       // row above (rows run last first), or of the next problem
        ++t;
      } else {
        tx = 0u;
        if (ty > 0u) {
          --ty;
        } else {
          ++z;
          ty = ny - 1u;
        }
        t = (z * ny + ty) * nx;
      }
    }
  };
  uint16_t held[SI][kOrderRun];
  if constexpr (STAGE) {
#pragma unroll
    for (int i = 0; i < SI; ++i) load_run((uint32_t)i * stride + (uint32_t)threadIdx.x * kOrderRun, held[i]);
  }
  __syncthreads();
  // (a thread's runs past the grid take no part: skipped, not counted as empty)
  if constexpr (STAGE) {
#pragma unroll
    for (int i = 0; i < SI; ++i) {
      uint32_t pos[kOrderRun];
      if ((uint32_t)i * stride + (uint32_t)threadIdx.x * kOrderRun < total) count_runs<false>(cur, held[i], pos);
    }
  } else {
    for (uint32_t c0 = 0; c0 < total; c0 += stride) {
      uint16_t b[kOrderRun];
      uint32_t pos[kOrderRun];
      if (c0 + (uint32_t)threadIdx.x * kOrderRun >= total) break;
      load_run(c0 + (uint32_t)threadIdx.x * kOrderRun, b);
      count_runs<false>(cur, b, pos);
    }
  }
  __syncthreads();
  // cur[b] <- the first position of bucket b: the count of every bucket above it (heavier work first)
  uint32_t cnt[PB], sum = 0u;
#pragma unroll
  for (int u = 0; u < PB; ++u) {
    cnt[u] = cur[kOrderBuckets - 1 - (threadIdx.x * PB + u)];
    sum += cnt[u];
  }
  uint32_t incl = sum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t o = (uint32_t)__shfl_up((int)incl, off, 64);
    if (lane >= off) incl += o;
  }
  if (lane == 63) wsum[wave] = incl;
  __syncthreads();
  uint32_t at = incl - sum;
  for (int w = 0; w < wave; ++w) at += wsum[w];
#pragma unroll
  for (int u = 0; u < PB; ++u) {
    cur[kOrderBuckets - 1 - (threadIdx.x * PB + u)] = at;
    at += cnt[u];
  }
  __syncthreads();
  if constexpr (STAGE) {
#pragma unroll
    for (int i = 0; i < SI; ++i) {
      const uint32_t p0 = (uint32_t)i * stride + (uint32_t)threadIdx.x * kOrderRun;
      if (p0 < total) place(p0, held[i]);
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < total; i += kOrderThreads) order[i] = stage[i];
  } else {
    for (uint32_t c0 = 0; c0 < total; c0 += stride) {
      uint16_t b[kOrderRun];
      if (c0 + (uint32_t)threadIdx.x * kOrderRun >= total) break;
      load_run(c0 + (uint32_t)threadIdx.x * kOrderRun, b);
      place(c0 + (uint32_t)threadIdx.x * kOrderRun, b);
    }
  }
}

// BM x BN outputs per workgroup, (BM / 16) x (BN / 16) per thread.  Held to four waves a SIMD (128 VGPRs): left
// alone the 64 x 64 instances take 129 to 137.
// HWF: the lanes are HW_FINAL's (SIZE 16, bf16 last), whose constants are then immediates.
template <int SIZE, bool BF16_LAST, int BM, int BN, bool HWF>
__global__ void __launch_bounds__(256, 4) k_systolic_fast(const SysArgs args, const FastLanes fl) {
  constexpr int TM = BM / 16, TN = BN / 16, NT = 256;
  static_assert(!HWF || (SIZE == 16 && BF16_LAST), "HW_FINAL has 16 lanes, the last bf16");
  const LaneConsts<HWF> lc{fl};
  static_assert((BM / TM) * (BN / TN) == NT, "256 threads");
  __shared__ __align__(16) Smem<BM, BN> sm;
  __shared__ uint32_t red[4][4];
  __shared__ uint32_t live[2][4];   // per staged buffer and wave: bit 0, A has a nonzero code; bit 1, B has;
                                    // bits 2-3, a staged block scale denies the short tile add (scale_denies)
  __shared__ float xs_a[2][BM], xs_b[2][BN];   // the stage's block scales (block size 32)
  const int tn = threadIdx.x % (BN / TN), tm = threadIdx.x / (BN / TN);
  // A stage whose A tile or B tile is all +-0 makes every product +-0, so every sum +-0 and every tile add
  // C + (+-0) * (finite scale) = C: the workgroup skips its lanes (its scales are still read and checked).
  auto note_live = [&](int to, uint32_t ma, uint32_t mb, uint32_t denies) {
    const uint32_t v = (__any(ma != 0u) ? 1u : 0u) | (__any(mb != 0u) ? 2u : 0u) |
                       (__any((denies & 1u) != 0u) ? 4u : 0u) | (__any((denies & 2u) != 0u) ? 8u : 0u);
    if ((threadIdx.x & 63) == 0) live[to][threadIdx.x >> 6] = v;
  };
  // Row tiles are dispatched last row first.  Where A is zero above a diagonal (attention's P^T under a causal
  // mask) the late rows carry the most nonzero stages: starting them first keeps them out of the tail.
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
    ty = args.tiles_y - 1 - blockIdx.y;
    tx = blockIdx.x;
  }
  const int64_t m0 = ty * BM, n0 = tx * BN;
  const float* A = args.A.p + z * args.A.batch;
  const float* B = args.B.p + z * args.B.batch;
  const float* XA = args.XA.p + z * args.XA.batch;
  const float* XB = args.XB.p + z * args.XB.batch;
  const bool va = vec_ok(args.A, A), vb = vec_ok(args.B, B);
  const int bs = args.block_size;
  const int64_t K = args.K, M = args.M, N = args.N;

  float C[TM][TN];
#pragma unroll
  for (int x = 0; x < TM; ++x)
#pragma unroll
    for (int y = 0; y < TN; ++y) C[x][y] = 0.0f;

  // a tile made only of groups the caller does not need is written as +0, uncomputed (the same decision in
  // every thread)
  if (args.skip) {
    if (args.order_skip ? marked : tile_skipped(args, z, m0, n0, BM, BN)) {
      if (threadIdx.x == 0) args.flags[(z * args.tiles_y + ty) * args.tiles_x + tx] = 0u;
      if (!args.c_end || n0 < args.c_end[z * args.kend_groups + m0 / 64])
        write_tile<TM, TN>(args, z, m0 + tm * TM, n0 + tn * TN, C);
      return;
    }
  }
  // the reduction runs to kstop: past the caller's k_end for these columns of A (a multiple of the stage height;
  // the rows skipped are checked below)
  const int64_t kstop = tile_kstop(args, z, m0);

  uint32_t max_a = 0u, max_b = 0u, max_x = 0u;   // largest |a|, |b| and scale this thread has read
  TileLoader<BM, NT> la;
  TileLoader<BN, NT> lb;
  ScaledRows<BM, NT, SIZE> rows;
  rows.init(fl, va);
  // STAGED (32-row tiles; the 64 x 64 instance would lose a wave per SIMD to the registers these take): an
  // interior tile loads whole stages without bounds checks (TileLoader::load_inner), and with block size 32,
  // where a stage is one block, the block scales are staged with it: thread t < BM reads XA's for the tile's
  // column t, BM <= t < BM + BN XB's for column t - BM, each checked once (its magnitude into max_x, whether it
  // allows the short tile add into the stage's live bits).  Otherwise each thread reads the scales of its
  // rows and columns as the reductions reach a new block.
  constexpr bool STAGED = BM == 32;
  const bool inner = STAGED && va && vb && m0 + BM <= M && n0 + BN <= N && args.A.ld < kInnerLd &&
                     args.B.ld < kInnerLd;
  const bool xs_staged = STAGED && bs == KT;
  float xv = 0.0f;
  auto load_stage = [&](int64_t k) {
    if (inner && k + KT <= K) {
      la.load_inner(A + k * args.A.ld + m0, (uint32_t)args.A.ld);
      lb.load_inner(B + k * args.B.ld + n0, (uint32_t)args.B.ld);
    } else {
      la.load(A, args.A.ld, K, M, k, m0, va);
      lb.load(B, args.B.ld, K, N, k, n0, vb);
    }
    if (xs_staged) {
      const int t = threadIdx.x;
      const int64_t g = k / KT;
      xv = 0.0f;
      if (t < BM) {
        if (m0 + t < M) xv = XA[g * args.XA.ld + m0 + t];
      } else if (t < BM + BN) {
        if (n0 + t - BM < N) xv = XB[g * args.XB.ld + n0 + t - BM];
      }
    }
  };
  auto store_stage = [&](int to) {
    const uint32_t ma = la.max_bits(), mb = lb.max_bits();
    max_a = umax(max_a, ma);
    max_b = umax(max_b, mb);
    uint32_t denies = 0u;
    if (xs_staged) {
      const int t = threadIdx.x;
      max_x = umax(max_x, f2u(xv) & 0x7FFFFFFFu);
      denies = scale_denies(xv, fl.xs_lo, fl.xs_hi);
      if (t < BM) xs_a[to][t] = xv;
      else if (t < BM + BN) xs_b[to][t - BM] = xv;
    }
    note_live(to, ma, mb, denies);
    rows.apply(la.v);
    la.store(sm.a[to], va);
    lb.store(sm.b[to], vb);
  };
  int buf = 0;
  if (kstop > 0) {                                // rows at and past kstop are never read
    load_stage(0);
    store_stage(0);
  }
  __syncthreads();

  float scale[TM][TN];
  bool short_add = false;  // this block's scales make bf16(S * scale) exact
  bool large = false;      // some scale so far was above xs_hi
  int in_block = 0;      // k of the current reduction within its block
  int64_t g = 0;         // its block
  for (int64_t k0 = 0; k0 < kstop; k0 += KT) {
    const bool more = k0 + KT < kstop;
    if (more) load_stage(k0 + KT);
    const int kend = (int)((K - k0 < KT) ? (K - k0) : KT);
    const uint32_t lv = live[buf][0] | live[buf][1] | live[buf][2] | live[buf][3];
    const bool zero_stage = (lv & 3u) != 3u;
    // rows past K are zero in LDS: their products are +0 and leave every lane's sum unchanged, so a short
    // last reduction runs as a whole one
    for (int r0 = 0; r0 < kend; r0 += SIZE) {
      if (in_block == 0 && xs_staged) {
        float xa[TM], xb[TN];
#pragma unroll
        for (int x = 0; x < TM; ++x) xa[x] = xs_a[buf][tm * TM + x];
#pragma unroll
        for (int y = 0; y < TN; ++y) xb[y] = xs_b[buf][tn * TN + y];
#pragma unroll
        for (int x = 0; x < TM; ++x)
#pragma unroll
          for (int y = 0; y < TN; ++y) scale[x][y] = xa[x] * xb[y];
        large = large || (lv & 8u) != 0u;                        // one decision per workgroup and block
        short_add = (lv & 4u) == 0u && !large;
      } else if (in_block == 0) {
        float xa[TM], xb[TN];
#pragma unroll
        for (int x = 0; x < TM; ++x) {
          const int64_t mm = m0 + tm * TM + x;
          xa[x] = mm < M ? XA[g * args.XA.ld + mm] : 0.0f;
          max_x = umax(max_x, f2u(xa[x]) & 0x7FFFFFFFu);
        }
#pragma unroll
        for (int y = 0; y < TN; ++y) {
          const int64_t nn = n0 + tn * TN + y;
          xb[y] = nn < N ? XB[g * args.XB.ld + nn] : 0.0f;
          max_x = umax(max_x, f2u(xb[y]) & 0x7FFFFFFFu);
        }
#pragma unroll
        for (int x = 0; x < TM; ++x)
#pragma unroll
          for (int y = 0; y < TN; ++y) scale[x][y] = xa[x] * xb[y];
        uint32_t denies = 0u;
#pragma unroll
        for (int x = 0; x < TM; ++x) denies |= scale_denies(xa[x], fl.xs_lo, fl.xs_hi);
#pragma unroll
        for (int y = 0; y < TN; ++y) denies |= scale_denies(xb[y], fl.xs_lo, fl.xs_hi);
        large = large || __any((denies & 2u) != 0u) != 0;        // one decision per wave and block
        short_add = __all(denies == 0u) != 0 && !large;
      }
      if (zero_stage) {
        in_block += SIZE;
        if (in_block == bs) {
          in_block = 0;
          ++g;
        }
        continue;
      }
      float S[TM][TN];
#pragma unroll
      for (int i = 0; i < SIZE; ++i) {
        float a[TM];
        if constexpr (TM == 4) {
          const float4 a4 = *reinterpret_cast<const float4*>(&sm.a[buf][r0 + i][tm * TM]);
          a[0] = a4.x; a[1] = a4.y; a[2] = a4.z; a[3] = a4.w;
        } else {
          const float2 a2 = *reinterpret_cast<const float2*>(&sm.a[buf][r0 + i][tm * TM]);
          a[0] = a2.x; a[1] = a2.y;
        }
        float b[TN];
        if constexpr (TN == 4) {
          const float4 b4 = *reinterpret_cast<const float4*>(&sm.b[buf][r0 + i][tn * TN]);
          b[0] = b4.x; b[1] = b4.y; b[2] = b4.z; b[3] = b4.w;
        } else {
          const float2 b2 = *reinterpret_cast<const float2*>(&sm.b[buf][r0 + i][tn * TN]);
          b[0] = b2.x; b[1] = b2.y;
        }
        if (BF16_LAST && i == SIZE - 1) {
          // bf16 lane: S (an e4 value, at most 8 significant bits) plus the truncated, flushed product
          // (prod_m + 1 <= 8 bits), one float32 add and bit RNE to bf16
#pragma unroll
          for (int x = 0; x < TM; ++x)
#pragma unroll
            for (int y = 0; y < TN; ++y) {
              float t = u2f(f2u(a[x] * b[y]) & fl.pmask);
              t = fabsf(t) < fl.flush_thr ? 0.0f : t;
              S[x][y] = fma_rne(S[x][y] * lc.out_scale() + t, 65536.0f);
            }
        } else if (i == 0) {
          // the first lane: S = lane(p).  p has at most prod_m + 1 <= m + 1 significant bits (an integer at or
          // above 2^prod_m steps; rounded to one below), so the lane's RNE at m fraction bits keeps it as is.
#pragma unroll
          for (int x = 0; x < TM; ++x)
#pragma unroll
            for (int y = 0; y < TN; ++y) S[x][y] = __builtin_rintf(u2f(f2u(a[x] * b[y]) & fl.pmask));
        } else {
          if (lc.steps_up(i)) {
#pragma unroll
            for (int x = 0; x < TM; ++x)
#pragma unroll
              for (int y = 0; y < TN; ++y) S[x][y] *= lc.rescale(i);
          }
          // e4 lane in units of the lane's subnormal step 2^-(6+m)
#pragma unroll
          for (int x = 0; x < TM; ++x)
#pragma unroll
            for (int y = 0; y < TN; ++y) {
              const float p = __builtin_rintf(u2f(f2u(a[x] * b[y]) & fl.pmask));
              S[x][y] = lc.rne(S[x][y] + p, i);
            }
        }
      }
      if (!BF16_LAST) {
#pragma unroll
        for (int x = 0; x < TM; ++x)
#pragma unroll
          for (int y = 0; y < TN; ++y) S[x][y] *= lc.out_scale();
      }
      // tile_add: C (a bf16 value, never -0) plus bf16(S * scale), one rounding to bf16.  The short form's branch is
      // taken only by the ladders that end in a bf16 lane (512 x 2048 outputs, K = 2048, blocks of 64: HW_FINAL 333 ->
      // 301 us; e4m4 lanes 407 with it, 387 without)
      if (BF16_LAST && short_add) {
#pragma unroll
        for (int x = 0; x < TM; ++x)
#pragma unroll
          for (int y = 0; y < TN; ++y) C[x][y] = fma_rne(__builtin_fmaf(S[x][y], scale[x][y], C[x][y]), 65536.0f);
      } else {
#pragma unroll
        for (int x = 0; x < TM; ++x)
#pragma unroll
          for (int y = 0; y < TN; ++y) C[x][y] = bf16_bits(C[x][y] + bf16_bits(S[x][y] * scale[x][y]));
      }
      in_block += SIZE;
      if (in_block == bs) {
        in_block = 0;
        ++g;
      }
    }
    if (more) store_stage(buf ^ 1);
    __syncthreads();
    buf ^= 1;
  }

  // rows past kstop: the results are exact only if A holds +-0 there, B and every remaining block scale are
  // finite (k_suffix_flags' bytes for this tile's groups and the stages it left out); bit j of `bad` for the
  // tile's 32-column group j of A (j < BM / 32), then of B
  constexpr int GT = BM / 32 + BN / 32;
  uint32_t bad = 0u;
  if (kstop < K) {
    const int64_t s0 = kstop / KT, ga = (M + 31) / 32, gb = (N + 31) / 32;
    for (int64_t i = threadIdx.x; i < (args.stages - s0) * GT; i += 256) {
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

  // the workgroup's verdict: its maxima over everything it read
  for (int off = 32; off > 0; off >>= 1) {
    max_a = umax(max_a, (uint32_t)__shfl_xor((int)max_a, off, 64));
    max_b = umax(max_b, (uint32_t)__shfl_xor((int)max_b, off, 64));
    max_x = umax(max_x, (uint32_t)__shfl_xor((int)max_x, off, 64));
    bad |= (uint32_t)__shfl_xor((int)bad, off, 64);
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    red[0][wave] = max_a;
    red[1][wave] = max_b;
    red[2][wave] = max_x;
    red[3][wave] = bad;
  }
  __syncthreads();
  const uint32_t wa = umax(umax(red[0][0], red[0][1]), umax(red[0][2], red[0][3]));
  const uint32_t wb = umax(umax(red[1][0], red[1][1]), umax(red[1][2], red[1][3]));
  const uint32_t wx = umax(umax(red[2][0], red[2][1]), umax(red[2][2], red[2][3]));
  const uint32_t wbad = red[3][0] | red[3][1] | red[3][2] | red[3][3];
  const bool ok = wbad == 0u && wa < kFastAMaxBits && wb < 0x7F800000u && wx < 0x7F800000u &&
                  u2f(wa) * u2f(wb) <= args.fast_prod_max;
  // the flag: bit 0, the general kernel computes the tile; bits 1..GT, which groups' left-out rows failed
  // their check (a piece of the tile reduces over all of K when its group of A or of B did, else to kstop)
  if (threadIdx.x == 0)
    args.flags[(z * args.tiles_y + ty) * args.tiles_x + tx] = ok ? 0u : 1u | (wbad << 1);
  if (!ok) return;
  write_tile<TM, TN>(args, z, m0 + tm * TM, n0 + tn * TN, C);
}

// ------------------------------------------------------------------------------- general datapath
// The BM x BN outputs at (m0, n0) of problem z.
// The reduction runs over rows [0, kstop) of A and B (kstop = K, or a multiple of 32 the fast kernel's check
// allows to stop at).
template <int BM, int BN, int TM, int TN>
__device__ __forceinline__ void gen_tile_at(const SysArgs& args, int64_t z, int64_t m0, int64_t n0, int64_t kstop,
                                            Smem<BM, BN>& sm) {
  constexpr int NT = (BM / TM) * (BN / TN);
  const int tn = threadIdx.x % (BN / TN), tm = threadIdx.x / (BN / TN);
  const float* A = args.A.p + z * args.A.batch;
  const float* B = args.B.p + z * args.B.batch;
  const float* XA = args.XA.p + z * args.XA.batch;
  const float* XB = args.XB.p + z * args.XB.batch;
  const bool va = vec_ok(args.A, A), vb = vec_ok(args.B, B);
  const int size = args.size, bs = args.block_size;
  const int64_t K = args.K, M = args.M, N = args.N;
  float C[TM][TN];
#pragma unroll
  for (int x = 0; x < TM; ++x)
#pragma unroll
    for (int y = 0; y < TN; ++y) C[x][y] = 0.0f;
  TileLoader<BM, NT> la;
  TileLoader<BN, NT> lb;
  int buf = 0;
  const int64_t kl = kstop < K ? kstop : K;       // rows at and past kstop are never read (they load as zeros)
  la.load(A, args.A.ld, kl, M, 0, m0, va);
  lb.load(B, args.B.ld, kl, N, 0, n0, vb);
  la.store(sm.a[0], va);
  lb.store(sm.b[0], vb);
  __syncthreads();
  float scale[TM][TN];
  int in_block = 0;
  int64_t g = 0;
  for (int64_t k0 = 0; k0 < kstop; k0 += KT) {
    const bool more = k0 + KT < kstop;
    if (more) {
      la.load(A, args.A.ld, K, M, k0 + KT, m0, va);
      lb.load(B, args.B.ld, K, N, k0 + KT, n0, vb);
    }
    const int kend = (int)((K - k0 < KT) ? (K - k0) : KT);
    for (int r0 = 0; r0 < kend; r0 += size) {
      if (in_block == 0) {
#pragma unroll
        for (int x = 0; x < TM; ++x) {
          const int64_t mm = m0 + tm * TM + x;
          const float xa = mm < M ? XA[g * args.XA.ld + mm] : 0.0f;
#pragma unroll
          for (int y = 0; y < TN; ++y) {
            const int64_t nn = n0 + tn * TN + y;
            const float xb = nn < N ? XB[g * args.XB.ld + nn] : 0.0f;
            scale[x][y] = xa * xb;
          }
        }
      }
      // the reduction ends at its size, the block's end or K's end, whichever is first
      int cnt = size;
      if (in_block + cnt > bs) cnt = bs - in_block;
      if (k0 + r0 + cnt > K) cnt = (int)(K - k0 - r0);
      float S[TM][TN];
#pragma unroll
      for (int x = 0; x < TM; ++x)
#pragma unroll
        for (int y = 0; y < TN; ++y) S[x][y] = 0.0f;
      for (int i = 0; i < cnt; ++i) {
        const int kk = r0 + i;
        const int e = args.lane_e[i], m = args.lane_m[i];
#pragma unroll
        for (int x = 0; x < TM; ++x) {
          const float a = sm.a[buf][kk][tm * TM + x];
#pragma unroll
          for (int y = 0; y < TN; ++y) {
            const float b = sm.b[buf][kk][tn * TN + y];
            S[x][y] = gen_acc(S[x][y], gen_product(a, b, args.ar), e, m, args.ar);
          }
        }
      }
#pragma unroll
      for (int x = 0; x < TM; ++x)
#pragma unroll
        for (int y = 0; y < TN; ++y) C[x][y] = gen_tile(C[x][y], S[x][y] * scale[x][y], args.ar);
      in_block += size;
      if (in_block >= bs) {
        in_block = 0;
        ++g;
      }
    }
    if (more) {
      la.store(sm.a[buf ^ 1], va);
      lb.store(sm.b[buf ^ 1], vb);
    }
    __syncthreads();
    buf ^= 1;
  }
  float* Cz = args.C + z * args.batch_c;
#pragma unroll
  for (int x = 0; x < TM; ++x) {
    const int64_t mm = m0 + tm * TM + x;
    if (mm >= M) continue;
    const float* row = args.epi_on ? epi_row(args, z, mm) : nullptr;
#pragma unroll
    for (int y = 0; y < TN; ++y) {
      const int64_t nn = n0 + tn * TN + y;
      if (nn < N) Cz[mm * args.ldc + nn] = args.epi_on ? epi_apply(args, row, nn, C[x][y]) : C[x][y];
    }
  }
}

// Where a general piece of a tile the fast kernel flagged (flag bits as it writes them) stops: at the fast
// kernel's stop under k_end when the rows left out passed the check for this piece's own columns of A and B
// (A +-0 there, B and the scales finite), else at K.  The fast lanes' arithmetic adds nothing for a +-0 code of
// A (its product flushes to +0, the lanes keep the sum, the tile add keeps C), the premise of the fast kernel's
// own stop; so the piece's bits are the same either way, and rows past k_end that passed are never read.
__device__ __forceinline__ int64_t piece_kstop(const SysArgs& a, uint32_t flag, int64_t z, int64_t m0, int64_t n0,
                                               int64_t tm0, int64_t tn0) {
  if (!a.k_end) return a.K;
  const int64_t ks = tile_kstop(a, z, tm0);
  if (ks >= a.K) return a.K;
  const uint32_t bad = flag >> 1;                 // bit j: group j of A (j < fbm / 32), then of B
  const int ja = (int)((m0 - tm0) / 32), jb = a.fbm / 32 + (int)((n0 - tn0) / 32);
  return ((bad >> ja) & 1u) || ((bad >> jb) & 1u) ? a.K : ks;
}

// only_flagged: the grid is the fast kernel's tiles (it ran first); a workgroup whose tile has its flag set
// computes that tile's BM x BN pieces in turn, the others return at once.  Otherwise one piece per workgroup.
template <int BM, int BN, int TM, int TN>
__global__ void __launch_bounds__((BM / TM) * (BN / TN), 4) k_systolic_gen(const SysArgs args) {
  __shared__ Smem<BM, BN> sm;
  gen_tile_at<BM, BN, TM, TN>(args, blockIdx.z, (int64_t)blockIdx.y * BM, (int64_t)blockIdx.x * BN, args.K, sm);
}

// After a fast kernel, the tiles it flagged, recomputed in BM x BN pieces, `pieces` a tile: workgroup g takes piece
// g % pieces of the set tiles among [g / pieces * per, ...) of the `total` (in the flags' order), 256 flags read at a
// time and the set ones listed in LDS.  At most 1024 workgroups, so a launch whose tiles are all exact (the usual case)
// costs the loads of the flags, not a workgroup per tile that exits at once (9 us for the 32768 tiles of one attention
// product).  A workgroup a piece and not a tile: with 64 x 64 tiles all refused, 512 x 2048 outputs of e4m4 lanes, K =
// 2048, took 20.6 ms on 256 workgroups (7.5 on 1024), 512 x 4096 of HW_FINAL, K =
// 4096, 43 (29).
template <int BM, int BN, int TM, int TN>
__global__ void __launch_bounds__((BM / TM) * (BN / TN), 4) k_systolic_gen_flagged(const SysArgs args, int64_t total,
                                                                                  int64_t per, uint32_t pieces) {
  static_assert(32 % BM == 0 && 32 % BN == 0, "a general tile lies inside one fast tile");
  static_assert((BM / TM) * (BN / TN) == 256, "a flag per thread");
  __shared__ Smem<BM, BN> sm;
  __shared__ uint32_t list[256];
  __shared__ uint32_t nl;
  const uint32_t share = blockIdx.x / pieces, piece = blockIdx.x - share * pieces;
  const uint32_t across = (uint32_t)args.fbn / BN, pm = piece / across * BM, pn = piece % across * BN;
  const int64_t t0 = (int64_t)share * per, t1 = t0 + per < total ? t0 + per : total;
  for (int64_t c0 = t0; c0 < t1; c0 += 256) {
    if (threadIdx.x == 0) nl = 0u;
    __syncthreads();
    const int64_t t = c0 + threadIdx.x;
    if (t < t1 && args.flags[t] != 0u) list[atomicAdd(&nl, 1u)] = threadIdx.x;
    __syncthreads();
    const uint32_t n = nl;
    for (uint32_t j = 0; j < n; ++j) {
      const int64_t tt = c0 + list[j];
      const uint32_t flag = args.flags[tt];
      const int64_t zy = tt / args.tiles_x, tx = tt - zy * args.tiles_x;
      const int64_t z = zy / args.tiles_y, ty = zy - z * args.tiles_y;
      const int64_t tm0 = ty * args.fbm, tn0 = tx * args.fbn;
      const int64_t m0 = tm0 + pm, n0 = tn0 + pn;
      if (m0 < args.M && n0 < args.N) {
        gen_tile_at<BM, BN, TM, TN>(args, z, m0, n0, piece_kstop(args, flag, z, m0, n0, tm0, tn0), sm);
        __syncthreads();   // the next piece restages sm
      }
    }
    __syncthreads();         // list and nl are rewritten for the next 256 flags
  }
}

// ------------------------------------------------------------------------------------------- host side
// A bound on |product| under which no e4 lane can overflow: with n e4 lanes of at least m_min fraction bits,
// a rounding in the normal range grows a value by a factor of at most 1 + u, u = 2^-(m_min+1), and one in the
// lane's subnormal range by at most 2^-7 absolute, so |S_k| <= P n (1 + u)^(n+1) + n 2^-7; the lanes stay
// finite while that is below 2^8 - 2^(6 - m_min) (the midpoint to 2^8 at m_min bits).
float fast_prod_bound(const int32_t* e, const int32_t* m, int size) {
  int n = 0, mmin = 99;
  for (int i = 0; i < size; ++i) {
    if (e[i] != 4) continue;
    ++n;
    mmin = m[i] < mmin ? m[i] : mmin;
  }
  if (n == 0) return 0.0f;
  const double u = std::ldexp(1.0, -(mmin + 1));
  const double bound = (256.0 - std::ldexp(1.0, 6 - mmin) - n / 128.0) / (n * std::pow(1.0 + u, n + 1));
  return (float)std::floor(bound);   // an integer, safely below the real bound
}

bool lanes_fast(const int32_t* e, const int32_t* m, int size, const mxq_arith_spec& ar) {
  if (ar.kind != MXQ_ARITH_MXGEMMINI || ar.prod_m > 7 || ar.prod_m < 0) return false;
  if (size != 4 && size != 8 && size != 16 && size != 32) return false;
  int prev = -1, mmax = 0, mmin = 99;
  for (int i = 0; i < size; ++i) {
    if (e[i] == 8 && m[i] == 7 && i == size - 1) continue;
    if (e[i] != 4 || m[i] < 1 || m[i] > 9 || m[i] < prev) return false;
    prev = m[i];
    mmax = m[i] > mmax ? m[i] : mmax;
    mmin = m[i] < mmin ? m[i] : mmin;
  }
  if (mmin == 99) return false;                                   // no e4 lane at all
  if (ar.prod_m > mmin) return false;                             // products must sit on every e4 grid
  if (ar.has_floor && !(ar.flush_thr <= pow2f(-7 - mmax))) return false;   // flush under half a step
  if (!(ar.sat_limit >= fast_prod_bound(e, m, size))) return false;   // saturation never reached
  if (e[size - 1] == 8) {
    if (prev > 7) return false;                                   // the bf16 lane holds the e4 sum exactly
    if (!ar.has_floor || !(ar.flush_thr >= pow2f(-126))) return false;   // products under 2^-126 are flushed
  }
  return true;
}

FastLanes make_fast_lanes(const int32_t* e, const int32_t* m, int size, const mxq_arith_spec& ar) {
  FastLanes fl{};
  int prev = -1;
  for (int i = 0; i < size; ++i) {
    fl.rescale[i] = 1.0f;
    if (e[i] == 8) continue;                                      // the bf16 lane: A staged unscaled
    const int mi = m[i];
    fl.a_exp[i] = 6 + mi;
    if (prev >= 0) fl.rescale[i] = pow2f(mi - prev);
    fl.split[i] = (float)((1u << (23 - mi)) + 1u);
    fl.magic[i] = 1.5f * pow2f(17 - mi);
    prev = mi;
  }
  fl.out_scale = pow2f(-(6 + prev));
  fl.pmask = ~((1u << (23 - ar.prod_m)) - 1u);
  fl.flush_thr = ar.has_floor ? ar.flush_thr : 0.0f;
  // The short tile add needs S * scale exact in bf16 and normal.  S has at most 8 significant bits with a bf16 last
  // lane, or when the last e4 lane's m is at most 7.  A nonzero S is at least s_min: an e4 sum is a multiple of its
  // last lane's step; after a bf16 lane, min(2^-(6 + m_last), flush_thr * 2^-prod_m) (a kept product has prod_m + 1
  // significant bits at or above the flush threshold, so any nonzero sum of the two is at least the smaller of
  // their steps).  |S| < 2^9.  With scales of magnitude 2^-L .. 2^H, S * xa * xb is normal when
  // 2L <= 126 + log2(s_min).  C stays below 2^112, as its rounding needs, with H = 45: each block adds less than
  // 2^99, and a sum of bf16 values stops growing once its half step exceeds what is added, below 2^109.
  fl.xs_lo = 1u;                                                 // empty range: always the rounded tile add
  fl.xs_hi = 0u;
  const bool bf16_last = e[size - 1] == 8;
  if (bf16_last ? ar.has_floor != 0 : prev <= 7) {
    int log_min = -(6 + prev);
    if (bf16_last) log_min = std::min(log_min, (int)std::floor(std::log2((double)ar.flush_thr)) - ar.prod_m);
    const int L = std::min(59, (126 + log_min) / 2);
    if (L >= 0 && 126 + log_min >= 0) {
      fl.xs_lo = (uint32_t)(127 - L) << 23;
      fl.xs_hi = (uint32_t)(127 + std::min(L, 45)) << 23;
    }
  }
  return fl;
}

// Whether MXGEMMINI's wide datapath (kWide) takes these lanes, its constants and its bound on max|a| * max|b|: lanes
// of e >= 5 and m <= 10, neither ever falling (so a lane holds the sum of the one before it, and a reduction cut
// short by K's end ends as it stands), every kept product on the lanes' grids; no product saturates, no sum overflows.
bool lanes_wide(const int32_t* e, const int32_t* m, int size, const mxq_arith_spec& ar, FastLanes* fl, float* prod_max) {
  if (ar.kind != MXQ_ARITH_MXGEMMINI || ar.prod_m < 0 || ar.prod_m > 7 || !ar.has_floor) return false;
  if (size != 4 && size != 8 && size != 16 && size != 32) return false;
  if (!(ar.flush_thr >= pow2f(-60)) || !(ar.flush_thr <= 1.0f)) return false;
  const int last_bit = (int)std::floor(std::log2((double)ar.flush_thr)) - ar.prod_m;   // of a kept product
  for (int i = 0; i < size; ++i) {
    if (e[i] < 5 || e[i] > 8 || m[i] < ar.prod_m || m[i] > 10) return false;
    if (i > 0 && (e[i] < e[i - 1] || m[i] < m[i - 1])) return false;
    if (2 - (1 << (e[i] - 1)) - m[i] > last_bit) return false;
  }
  // |sum| <= size * P * (1 + 2^-(m+1))^size < 2^(emax of the first lane)
  const double top = std::ldexp(1.0, std::min((1 << (e[0] - 1)) - 1, 40));
  const double sums = size * std::pow(1.0 + std::ldexp(1.0, -(m[0] + 1)), size);
  *prod_max = (float)std::min((double)ar.sat_limit, std::floor(top / sums));
  if (!(*prod_max >= 1.0f)) return false;
  *fl = FastLanes{};
  for (int i = 0; i < size; ++i) {
    fl->pw[i] = (float)(1u << (23 - m[i]));
    fl->low[i] = 1.0f - fl->pw[i];
  }
  fl->pmask = ~((1u << (23 - ar.prod_m)) - 1u);
  fl->flush_thr = ar.flush_thr;
  // a tile is rounded to bf16 as a normal number when its scales are 2^-L .. 2^H; C stays below 2^112 as in
  // make_fast_lanes
  const int L = std::min(59, (126 + last_bit) / 2);
  const int H = std::min(45, (98 - (int)std::ceil(std::log2(sums * *prod_max))) / 2);
  fl->xs_lo = (uint32_t)(127 - L) << 23;
  fl->xs_hi = (uint32_t)(127 + std::max(H, 0)) << 23;
  return true;
}

// Whether the fast MXQUANT datapath takes these lanes (kMxq, or kMxqHigh when no nonzero sum falls below a lane's
// least value), its constants and its bound on max|a| * max|b|: no product and no sum saturates.  A reduction cut
// short by K's end ends as it stands where later lanes hold the sum (e and m never falling).
bool lanes_mxquant(const int32_t* e, const int32_t* m, int size, const mxq_arith_spec& ar, int64_t K, FastLanes* fl,
                   float* prod_max, bool* high) {
  if (ar.kind != MXQ_ARITH_MXQUANT || (size != 4 && size != 8 && size != 16 && size != 32)) return false;
  if (ar.prod_e < 2 || ar.prod_e > 8 || ar.prod_m < 1 || ar.prod_m > 22) return false;
  int emin = 8, mmin = 22;
  bool rising = true;
  *high = true;
  const int Lp = (1 << (ar.prod_e - 1)) - 1;
  for (int i = 0; i < size; ++i) {
    if (e[i] < 2 || e[i] > 8 || m[i] < 1 || m[i] > 22) return false;
    emin = std::min(emin, (int)e[i]);
    mmin = std::min(mmin, (int)m[i]);
    if (i > 0 && (e[i] < e[i - 1] || m[i] < m[i - 1])) rising = false;
    if (e[i] != 8 && (1 << (e[i] - 1)) - 1 < Lp + ar.prod_m) *high = false;
  }
  if (!rising && K % size != 0) return false;
  // |p| <= P (1 + 2^-(prod_m+1)) or 2^-Lp; each sum grows by a lane's rounding, or to its least value
  const int Lmin = (1 << (emin - 1)) - 1;
  const double up = 1.0 + std::ldexp(1.0, -(ar.prod_m + 1)), us = std::pow(1.0 + std::ldexp(1.0, -(mmin + 1)), size);
  const double least = std::ldexp(1.0, -Lp) + std::ldexp(1.0, -Lmin);
  const double bound = std::min(std::ldexp(1.0, std::min(Lp, 60)) / up,
                                (std::ldexp(1.0, std::min(Lmin, 60)) / (size * us) - least) / up);
  if (!(bound > 0.0)) return false;
  *prod_max = (float)(bound * (1.0 - 1e-6));
  *fl = FastLanes{};
  fl->prod = qtorch_of(ar.prod_e, ar.prod_m);
  for (int i = 0; i < size; ++i) fl->lane[i] = qtorch_of(e[i], m[i]);
  return true;
}

template <int SIZE, bool BF16_LAST, bool HWF>
void launch_fast_tile(dim3 grid, hipStream_t st, const SysArgs& a, const FastLanes& fl) {
  if (a.fbm == 64) k_systolic_fast<SIZE, BF16_LAST, 64, 64, HWF><<<grid, 256, 0, st>>>(a, fl);
  else if (a.fbn == 64) k_systolic_fast<SIZE, BF16_LAST, 32, 64, HWF><<<grid, 256, 0, st>>>(a, fl);
  else k_systolic_fast<SIZE, BF16_LAST, 32, 32, HWF><<<grid, 256, 0, st>>>(a, fl);
}

template <int SIZE>
void launch_fast_size(bool bf16_last, dim3 grid, hipStream_t st, const SysArgs& a, const FastLanes& fl) {
  if (bf16_last) launch_fast_tile<SIZE, true, false>(grid, st, a, fl);
  else launch_fast_tile<SIZE, false, false>(grid, st, a, fl);
}

bool is_hw_final(const int32_t* e, const int32_t* m, int size) {
  if (size != 16 || e[15] != 8 || m[15] != 7) return false;
  for (int i = 0; i < 15; ++i)
    if (e[i] != 4 || m[i] != hw_final_m(i)) return false;
  return true;
}

void launch_fast(int size, bool bf16_last, bool hwf, dim3 grid, hipStream_t st, const SysArgs& a,
                 const FastLanes& fl) {
  if (hwf) {
    launch_fast_tile<16, true, true>(grid, st, a, fl);
    return;
  }
  switch (size) {
    case 4: launch_fast_size<4>(bf16_last, grid, st, a, fl); break;
    case 8: launch_fast_size<8>(bf16_last, grid, st, a, fl); break;
    case 16: launch_fast_size<16>(bf16_last, grid, st, a, fl); break;
    default: launch_fast_size<32>(bf16_last, grid, st, a, fl); break;
  }
}

// Which kernel computes a call, and its tile.
struct Plan {
  enum Kernel { kGeneral = MXQ_SYS_GENERAL, kSmall = MXQ_SYS_SMALL, kTile = MXQ_SYS_TILE, kFast = MXQ_SYS_FAST } kernel;
  SmallTile small;
  int bm, bn;              // the tile kernels' tile
};

// What a launch takes, in microseconds: `start`, `each` for every 256 workgroups (one a CU) begun, and for every 2048
// rows of K `fill` and a `round` for every 256 workgroups, at least `alone`, which that many of one wave a SIMD take; the
// last three times `cost`, a datapath's (by LaneKind; 0: no such instance).  K counts rounded up to what a workgroup
// takes at once: a block of a tile kernel, or a small kernel's round of one reduction for every wave and group of columns
// (up to 1024 rows: 128 x 2048 outputs of K = 64 take 4-row tiles of 16 columns 117 us, tiles of 32 x 32 12).
// Fitted to every kernel's time on 39 shapes of 1 x 1000 to 2048 x 4096 outputs at K = 32 to 2048, under HW_FINAL
// (within 3 to 8 % each), `cost` under the other datapaths.  On average the shape chosen takes 0.5 % longer than the
// fastest, 18 % at the worst of 950.
struct Shape {
  Plan::Kernel kernel;
  int rows, log_cols, waves;
  double start, each, fill, round, alone;
  double cost[6];
};
constexpr Shape kShapes[] = {
    // (HW_FINAL: 512 x 2048 outputs at K = 32 and 2048, then 200 x 2048)
    {Plan::kTile, 64, 6, 8, 5.1, 2.2, 61, 215, 278, {1, 1.35, 1.40, 2.39, 2.10, 2.10}},    // 13, 282; 12, 293
    {Plan::kTile, 32, 5, 4, 5.9, 0.6, 60, 55, 164, {1, 1.32, 1.36, 2.24, 1.96, 1.96}},     // 14, 286; 10, 181
    {Plan::kSmall, 16, 6, 8, 2.4, 1.1, 22, 74, 105, {1, 0, 0, 2.06, 0, 0}},                // 28, 322; 15, 160
    {Plan::kSmall, 8, 6, 8, 2.5, 1.1, 14, 43, 64, {1, 1.28, 1.28, 1.83, 1.70, 1.70}},      // 34, 369; 19, 183
    {Plan::kSmall, 8, 6, 16, 1.9, 2.5, 0, 51, 0, {1, 0, 0, 1.86, 0, 0}},                   // 74, 422; 38, 205
    {Plan::kSmall, 8, 5, 16, 2.1, 1.5, 0, 31, 0, {1, 0, 0, 1.70, 0, 0}},                   // 147, 514; 66, 214
    {Plan::kSmall, 8, 5, 8, 2.5, 0.7, 5, 25, 37, {1, 1.30, 1.29, 1.73, 1.69, 1.69}},       // 64, 419; 30, 176
    {Plan::kSmall, 4, 6, 16, 1.9, 2.6, 0, 33, 33, {1, 1.18, 1.22, 1.63, 1.58, 1.58}},      // 114, 561; 50, 241
    {Plan::kSmall, 4, 5, 16, 1.9, 2.1, 0, 19, 0, {1, 1.16, 1.21, 1.53, 1.51, 1.51}},       // 225, 651; 92, 266
    {Plan::kSmall, 4, 4, 16, 1.8, 0.0, 0, 15, 0, {1, 1.08, 1.13, 1.33, 1.30, 1.30}},       // 465, 987; 183, 384
    {Plan::kFast, 64, 6, 4, 5.1, 1.9, 174, 203, 533, {1, 1.23, 0, 0, 0, 0}},               // 16, 567; 16, 548
    {Plan::kFast, 32, 6, 4, 5.7, 1.1, 110, 106, 305, {1, 1.26, 0, 0, 0, 0}},               // 13, 326; 12, 320
    {Plan::kFast, 32, 5, 4, 5.9, 0.8, 99, 52, 190, {1, 1.34, 0, 0, 0, 0}},                 // 14, 299; 11, 200
};

Plan plan_launch(const SysArgs& a, int64_t count, int kind) {
  // hints that leave rows of A unread (a_live) or outputs unstored (c_end) need a tile kernel, whose own limits are
  // blocks of 32 and a lane's offset in 32 bits; k_systolic_small's are its 32-bit rows and lane offsets: of B, and of
  // the 64 * waves / rows rows of A its threads reach from one address (small_fits)
  const bool small_ok = !a.c_end && !a.a_live && a.K < (int64_t(1) << 30) && a.B.ld < (int64_t(1) << 18);
  const bool tile_ok = a.block_size == KT && a.A.ld < (int64_t(1) << 28) && a.B.ld < (int64_t(1) << 28);
  const bool every_small = kind == kE4Final || kind == kMxqFinal;
  auto small_fits = [&](int rows, int waves) {
    return small_ok && a.A.ld < (int64_t(1) << 32) / (64 * waves / rows) && mxq::ceil_div(a.M, rows) <= 65535;
  };
  Plan p{};
  if (a.M == 1 && every_small && small_fits(1, 16)) {
    // one row: 32 columns a workgroup while that leaves half the CUs one (K = 2048, 5632 columns: 23 us, 35 with 16,
    // 25 with 64), 64 when that makes one for every CU (32000 columns: 65, 85 with 32)
    auto wgs = [&](int log_cw) { return mxq::ceil_div(a.N, int64_t(1) << log_cw) * count; };
    p.kernel = Plan::kSmall;
    p.small = {1, wgs(6) >= 256 ? 6 : wgs(5) >= 128 ? 5 : 4, 16};
    return p;
  }
  double best = 0.0;
  for (const Shape& sh : kShapes) {
    const bool small = sh.kernel == Plan::kSmall;
    if (sh.cost[kind] == 0.0 || (small && !small_fits(sh.rows, sh.waves))) continue;
    if (sh.kernel == Plan::kTile && !tile_ok) continue;
    // k_systolic_fast takes what k_systolic_tile does not, and the ladders whose constants are no literals, some of
    // which it runs faster (e4m4 lanes, 2048 x 4096 outputs of K = 200: 245 us on 64 x 64 tiles, 282)
    if (sh.kernel == Plan::kFast && tile_ok && kind != kE4) continue;
    // A small kernel's last columns, where they are not a whole group, go by checked loads, and its workgroups there end
    // last.  Per ladder: shorter reductions pay its LDS round trip and tile add more often, 32 lanes' constants spill; and
    // k_systolic_fast's ragged rows go a float at a time.
    double cost = sh.cost[kind];
    if (small) {
      cost *= a.size == 4 ? (sh.rows == 4 ? 1.7 : 1.25) : a.size == 8 ? (sh.rows == 4 ? 1.2 : 1.05) : a.size == 32 ? 1.08 : 1.0;
      const bool whole = a.N % (int64_t(1) << sh.log_cols) == 0;
      cost *= whole ? 0.97 : sh.log_cols == 6 ? 1.10 : sh.log_cols == 5 ? 1.05 : 1.02;
      if (!whole && a.size == 32) cost *= 1.12;
    } else if (a.size == 32) {
      cost *= sh.kernel == Plan::kTile && sh.rows == 32 ? 1.13 : 1.07;
    } else {
      cost *= sh.kernel == Plan::kTile ? (a.size < 16 ? 0.97 : 1.0) : a.size == 4 ? 1.1 : a.size == 8 ? 0.93 : 1.0;
    }
    if (sh.kernel == Plan::kFast && (a.M % 4 != 0 || a.N % 4 != 0)) cost *= 1.1;
    // (one wave a SIMD waits as long as it issues: a datapath's longer code costs it less)
    const double alone = sh.alone * (small ? cost : 1.0 + 0.45 * (cost - 1.0));
    const int64_t wgs = mxq::ceil_div(a.M, sh.rows) * mxq::ceil_div(a.N, int64_t(1) << sh.log_cols) * count;
    const double n = (double)mxq::ceil_div(wgs, 256);
    const int64_t at_once = small ? (int64_t)sh.waves * (64 >> sh.log_cols) * a.size : KT;
    double t = std::max(alone, cost * (sh.fill + sh.round * n)) * (double)(mxq::ceil_div(a.K, at_once) * at_once) / 2048.0;
    if (!small && a.k_end) t *= 0.6;                  // a causal mask's half, and the uneven rest of it
    t += sh.start + sh.each * n;
    if (!small && (a.skip || a.k_end)) t += 20.0;     // the dispatch order's and the suffix check's launches
    if (p.kernel == Plan::kGeneral || t < best) {
      best = t;
      p.kernel = sh.kernel;
      p.small = {sh.rows, sh.log_cols, sh.waves};
      p.bm = sh.rows;
      p.bn = 1 << sh.log_cols;
    }
  }
  return p;
}

// The fast datapath of these lanes (-1: none), its constants and its bound on max|a| * max|b|.
int datapath_of(const int32_t* e, const int32_t* m, int size, const mxq_arith_spec& ar, int64_t K, FastLanes* fl,
                float* prod_max) {
  const bool hwf = is_hw_final(e, m, size);
  bool high = false;
  if (K <= 0) return -1;
  if (lanes_fast(e, m, size, ar)) {
    *fl = make_fast_lanes(e, m, size, ar);
    *prod_max = fast_prod_bound(e, m, size);
    return hwf ? kE4Final : kE4;
  }
  if (lanes_wide(e, m, size, ar, fl, prod_max)) return kWide;
  if (lanes_mxquant(e, m, size, ar, K, fl, prod_max, &high)) return high ? kMxqHigh : hwf ? kMxqFinal : kMxq;
  return -1;
}

bool lanes_valid(const int32_t* e, const int32_t* m, int size) {
  for (int i = 0; i < size; ++i) {
    const bool ok = (e[i] == 8 && m[i] == 23) || (e[i] >= 1 && e[i] <= 8 && m[i] >= 1 && m[i] <= 22);
    if (!ok) return false;
  }
  return true;
}

int run_systolic(const SysArgs& base, const int32_t* lane_e, const int32_t* lane_m, int64_t count,
                 int32_t force_general, hipStream_t st) {
  const mxq_arith_spec& ar = base.ar;
  SysArgs a = base;
  for (int i = 0; i < a.size; ++i) { a.lane_e[i] = (int8_t)lane_e[i]; a.lane_m[i] = (int8_t)lane_m[i]; }
  FastLanes fl;
  const int kind = force_general ? -1 : datapath_of(lane_e, lane_m, a.size, ar, a.K, &fl, &a.fast_prod_max);
  const bool bf16_last = lane_e[a.size - 1] == 8, hwf = is_hw_final(lane_e, lane_m, a.size);
  const Plan plan = kind < 0 ? Plan{} : plan_launch(a, count, kind);
  if (plan.kernel == Plan::kSmall) {
    mxq::KernelTimer timer("systolic_small", st);
    if (kind <= kE4) launch_small_e4(kind, bf16_last, a, fl, plan.small, count, st);
    else if (kind == kWide) launch_small_wide(a, fl, plan.small, count, st);
    else launch_small_mxquant(kind, a, fl, plan.small, count, st);
    return mxq::check_launch("mxq_systolic small");
  }
  const dim3 grid_g((unsigned)mxq::ceil_div(a.N, 32), (unsigned)mxq::ceil_div(a.M, 32), (unsigned)count);
  if (plan.kernel != Plan::kGeneral) {
    a.fbm = plan.bm;
    a.fbn = plan.bn;
    a.tiles_x = mxq::ceil_div(a.N, a.fbn);
    a.tiles_y = mxq::ceil_div(a.M, a.fbm);
    const dim3 grid_f((unsigned)a.tiles_x, (unsigned)a.tiles_y, (unsigned)count);
    // workspace: a flag per 32 x 32 tile (W), the dispatch order (W), the suffix bytes of A's and B's groups
    const int64_t W = mxq::ceil_div(a.M, 32) * mxq::ceil_div(a.N, 32) * count;
    const int64_t total = a.tiles_x * a.tiles_y * count;
    if (a.k_end) {
      const int64_t stages = mxq::ceil_div(a.K, KT), ga = mxq::ceil_div(a.M, 32), gb = mxq::ceil_div(a.N, 32);
      if (stages <= 65535) {
        uint8_t* fa = reinterpret_cast<uint8_t*>(a.flags + 2 * W);
        uint8_t* fb = fa + count * stages * ga;
        a.stages = stages;
        const int64_t blocks = (a.a_live ? 0 : mxq::ceil_div(a.M, kSufCols)) + mxq::ceil_div(a.N, kSufCols);
        k_suffix_flags<<<dim3((unsigned)blocks, (unsigned)stages, (unsigned)count), 256, 0, st>>>(a, ga, gb, fa, fb);
        a.suf_a = a.a_live ? a.a_live : fa;
        a.suf_b = fb;
      } else {
        a.k_end = nullptr;   // the hint is dropped: every reduction runs to K
      }
    }
    if ((a.skip || a.k_end) && total <= (int64_t)0xFFFFFFFFu) {
      // the buckets live in the flag area until the fast kernel rewrites it
      uint32_t* order = a.flags + W;
      uint16_t* bucket = reinterpret_cast<uint16_t*>(a.flags);
      a.order_skip = a.skip && total <= (int64_t)0x80000000u ? 1 : 0;
      k_tile_bucket<<<(unsigned)mxq::ceil_div(total, 256), 256, 0, st>>>(a, (uint32_t)total, bucket);
      if (total <= kOrderStage) k_tile_order<true><<<1, kOrderThreads, 0, st>>>(a, (uint32_t)total, bucket, order);
      else k_tile_order<false><<<1, kOrderThreads, 0, st>>>(a, (uint32_t)total, bucket, order);
      a.order = order;
    }
    {
      mxq::KernelTimer timer("systolic_fast", st);
      if (plan.kernel == Plan::kFast) launch_fast(a.size, bf16_last, hwf, grid_f, st, a, fl);
      else if (kind <= kE4) launch_tile_e4(kind, bf16_last, grid_f, a, fl, st);
      else if (kind == kWide) launch_tile_wide(grid_f, a, fl, st);
      else launch_tile_mxquant(kind, grid_f, a, fl, st);
    }
    if (int rc = mxq::check_launch("mxq_systolic fast")) return rc;
    mxq::KernelTimer timer("systolic_general", st);
    const int64_t tiles = a.tiles_x * a.tiles_y * count;
    const uint32_t pieces = (uint32_t)(a.fbm / 32 * (a.fbn / 32));
    const int64_t shares = std::min(tiles, (int64_t)(1024 / pieces));
    if (shares > 0)
      k_systolic_gen_flagged<32, 32, 2, 2><<<(unsigned)(shares * pieces), 256, 0, st>>>(a, tiles, mxq::ceil_div(tiles, shares),
                                                                                       pieces);
  } else {
    mxq::KernelTimer timer("systolic_general", st);
    k_systolic_gen<32, 32, 2, 2><<<grid_g, 256, 0, st>>>(a);
  }
  return mxq::check_launch("mxq_systolic");
}

void take_hints(SysArgs& a, const mxq_systolic_hints* hints) {
  if (!hints) return;
  a.skip = hints->skip;
  a.skip_rows = mxq::ceil_div(a.M, 32);
  a.skip_cols = mxq::ceil_div(a.N, 32);
  a.k_end = hints->k_end;
  a.kend_groups = mxq::ceil_div(a.M, 64);
  a.a_live = hints->k_end ? hints->a_live : nullptr;
  a.c_end = hints->skip ? hints->c_end : nullptr;
}

int check_common(int64_t K, int64_t M, int64_t N, int64_t count, const int32_t* lane_e, const int32_t* lane_m,
                 int32_t size, int32_t block_size, const mxq_arith_spec* arith) {
  if (!arith || !lane_e || !lane_m) return mxq::invalid("mxq_systolic: NULL spec or lanes");
  if (K < 0 || M < 0 || N < 0 || count < 0) return mxq::invalid("mxq_systolic: negative shape");
  if (mxq::ceil_div(M, 32) > 65535 || count > 65535) return mxq::invalid("mxq_systolic: M or batch too large");
  if (size < 1 || size > kMaxLanes) return mxq::invalid("mxq_systolic: size must be in [1, 64]");
  if (block_size < 1 || block_size % size) return mxq::invalid("mxq_systolic: size must divide block_size");
  if (KT % size) return mxq::invalid("mxq_systolic: size must divide 32");
  if (arith->kind != MXQ_ARITH_MXGEMMINI && arith->kind != MXQ_ARITH_MXQUANT)
    return mxq::invalid("mxq_systolic: bad arithmetic");
  if (!lanes_valid(lane_e, lane_m, size)) return mxq::invalid("mxq_systolic: unsupported lane widths");
  return MXQ_OK;
}

}  // namespace

extern "C" int mxq_systolic_fast_lanes(const int32_t* lane_e, const int32_t* lane_m, int32_t size,
                                       const mxq_arith_spec* arith) {
  if (!arith || !lane_e || !lane_m || size < 1 || size > kMaxLanes || !lanes_valid(lane_e, lane_m, size)) return 0;
  return lanes_fast(lane_e, lane_m, size, *arith) ? 1 : 0;
}

extern "C" int mxq_systolic_plan_of(const mxq_systolic_layout* layout, int64_t count, int64_t K, int64_t M, int64_t N,
                                    const int32_t* lane_e, const int32_t* lane_m, int32_t size, int32_t block_size,
                                    const mxq_arith_spec* arith, const mxq_systolic_hints* hints,
                                    mxq_systolic_plan* plan) {
  if (int rc = check_common(K, M, N, count, lane_e, lane_m, size, block_size, arith)) return rc;
  if (!plan) return mxq::invalid("mxq_systolic_plan_of: NULL plan");
  SysArgs a{};
  a.A.ld = layout ? layout->ld_a : M;
  a.B.ld = layout ? layout->ld_b : N;
  a.K = K; a.M = M; a.N = N; a.size = size; a.block_size = block_size;
  take_hints(a, hints);
  FastLanes fl;
  const int kind = datapath_of(lane_e, lane_m, size, *arith, K, &fl, &a.fast_prod_max);
  const Plan p = kind < 0 ? Plan{} : plan_launch(a, count, kind);
  *plan = mxq_systolic_plan{p.kernel, 32, 32, 4};                 // k_systolic_gen's tile
  if (p.kernel == Plan::kSmall) *plan = {p.kernel, p.small.rows, 1 << p.small.log_cw, p.small.waves};
  if (p.kernel == Plan::kTile) *plan = {p.kernel, p.bm, p.bn, p.bm / 8};
  if (p.kernel == Plan::kFast) *plan = {p.kernel, p.bm, p.bn, 4};
  return MXQ_OK;
}

extern "C" int mxq_systolic(const float* P_A, const float* X_A, const float* P_B, const float* X_B, float* C,
                            int64_t K, int64_t M, int64_t N, const int32_t* lane_e, const int32_t* lane_m,
                            int32_t size, int32_t block_size, const mxq_arith_spec* arith, uint32_t* workspace,
                            int32_t force_general, mxq_stream_t stream) {
  if (int rc = check_common(K, M, N, 1, lane_e, lane_m, size, block_size, arith)) return rc;
  if (M == 0 || N == 0) return MXQ_OK;
  if (!P_A || !X_A || !P_B || !X_B || !C || !workspace) return mxq::invalid("mxq_systolic: NULL pointer");
  SysArgs a{};
  a.A = {P_A, M, 0}; a.XA = {X_A, M, 0}; a.B = {P_B, N, 0}; a.XB = {X_B, N, 0};
  a.C = C; a.ldc = N; a.batch_c = 0; a.flags = workspace;
  a.K = K; a.M = M; a.N = N; a.size = size; a.block_size = block_size; a.ar = *arith;
  return run_systolic(a, lane_e, lane_m, 1, force_general, mxq::as_stream(stream));
}

extern "C" int mxq_systolic_batched(const float* P_A, const float* X_A, const float* P_B, const float* X_B,
                                    float* C, const mxq_systolic_layout* layout, int64_t count, int64_t K,
                                    int64_t M, int64_t N, const int32_t* lane_e, const int32_t* lane_m, int32_t size,
                                    int32_t block_size, const mxq_arith_spec* arith,
                                    const mxq_systolic_hints* hints, const mxq_systolic_epilogue* epilogue,
                                    uint32_t* workspace, int32_t force_general, mxq_stream_t stream) {
  if (int rc = check_common(K, M, N, count, lane_e, lane_m, size, block_size, arith)) return rc;
  if (!layout) return mxq::invalid("mxq_systolic_batched: NULL layout");
  const mxq_systolic_layout& L = *layout;
  if (L.ld_a < M || L.ld_b < N || L.ld_xa < M || L.ld_xb < N || L.ld_c < N)
    return mxq::invalid("mxq_systolic_batched: a row stride is shorter than its row");
  if (L.batch_a < 0 || L.batch_b < 0 || L.batch_xa < 0 || L.batch_xb < 0 || L.batch_c < 0)
    return mxq::invalid("mxq_systolic_batched: negative batch stride");
  // the problems' outputs one after another, or side by side within each row (problem z's row r at
  // z * batch_c + r * ld_c, the rows of all problems together no longer than ld_c); any other layout is refused
  if (count > 1 && M > 0 && N > 0 && L.batch_c < (M - 1) * L.ld_c + N &&
      !(L.batch_c >= N && (count - 1) * L.batch_c + N <= L.ld_c))
    return mxq::invalid("mxq_systolic_batched: outputs of two problems overlap");
  if (epilogue && (epilogue->m < 1 || epilogue->m > 0x7FFFFFFF || epilogue->z_per_b < 1 ||
                   epilogue->z_per_b > 0x7FFFFFFF || epilogue->z0 < 0 || epilogue->z0 + count > 0x7FFFFFFF))
    return mxq::invalid("mxq_systolic_batched: epilogue needs m >= 1 and z_per_b >= 1 (below 2^31), z0 >= 0 and "
                        "z0 + count below 2^31");
  if (M == 0 || N == 0 || count == 0) return MXQ_OK;
  if (!P_A || !X_A || !P_B || !X_B || !C || !workspace) return mxq::invalid("mxq_systolic_batched: NULL pointer");
  SysArgs a{};
  a.A = {P_A, L.ld_a, L.batch_a}; a.XA = {X_A, L.ld_xa, L.batch_xa};
  a.B = {P_B, L.ld_b, L.batch_b}; a.XB = {X_B, L.ld_xb, L.batch_xb};
  a.C = C; a.ldc = L.ld_c; a.batch_c = L.batch_c; a.flags = workspace;
  a.K = K; a.M = M; a.N = N; a.size = size; a.block_size = block_size; a.ar = *arith;
  take_hints(a, hints);
  if (epilogue) {
    a.epi_on = 1;
    a.epi = *epilogue;
  }
  return run_systolic(a, lane_e, lane_m, count, force_general, mxq::as_stream(stream));
}

// ------------------------------------------------------------------------ the allocation-free entry point
// mxq_systolic_noalloc keeps the fast kernel's per-tile flags (its only scratch when no hints are given) in this
// array instead of a caller's workspace.  Each GPU holds its own copy for the life of the process.  In host code
// the name `scratch` is a stand-in, not a device address: the kernels get the address hipGetSymbolAddress gives
// on each device, looked up once per device on that device's first call and kept in g_scratch.
constexpr int64_t kScratchWords = int64_t(1) << 18;                 // 1 MiB: ceil(M/32) * ceil(N/32) flags
static __device__ __align__(256) uint32_t scratch[kScratchWords];

namespace {

constexpr int kMaxDevices = 64;

// Per device: the scratch array's address, and the guard against calls that overlap on the GPU: an event
// recorded behind each call's kernels on its stream.  A call on another stream while that event is pending
// would share the array with a running call, so it is refused (MXQ_EBUSY); calls on one stream are ordered by
// the stream and need no test.  Calls made while their stream is being captured into a graph neither test nor
// record (the graph's replays are the caller's to order).
struct ScratchSlot {
  uint32_t* p = nullptr;
  hipEvent_t done = nullptr;
  hipStream_t last = nullptr;
  bool pending = false;        // `done` was recorded by a call outside capture
};
std::mutex g_scratch_mu;       // held from the guard's test through the launch and the record
ScratchSlot g_scratch[kMaxDevices];

int hip_fail(const char* what, hipError_t err) {
  mxq::set_error(std::string("mxq_systolic_noalloc: ") + what + ": " + hipGetErrorString(err));
  return MXQ_EHIP;
}

// The current device (which must be the stream's) and its slot, set up on the device's first call.
int slot_on_device(hipStream_t st, ScratchSlot** out) {
  int dev = -1;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) return hip_fail("hipGetDevice", err);
  if (dev < 0 || dev >= kMaxDevices) return mxq::invalid("mxq_systolic_noalloc: device index out of range");
  if (st) {
    int sdev = -1;
    err = hipStreamGetDevice(st, &sdev);
    if (err != hipSuccess) return hip_fail("hipStreamGetDevice", err);
    if (sdev != dev) return mxq::invalid("mxq_systolic_noalloc: the stream belongs to another device than the current one");
  }
  ScratchSlot& sl = g_scratch[dev];
  if (!sl.p) {
    void* p = nullptr;
    err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (err != hipSuccess || !p) return hip_fail("hipGetSymbolAddress", err);
    err = hipEventCreateWithFlags(&sl.done, hipEventDisableTiming);
    if (err != hipSuccess) return hip_fail("hipEventCreateWithFlags", err);
    sl.p = static_cast<uint32_t*>(p);
  }
  *out = &sl;
  return MXQ_OK;
}

}  // namespace

extern "C" int mxq_systolic_noalloc(const float* P_A, const float* X_A, const float* P_B, const float* X_B,
                                    float* C, int64_t K, int64_t M, int64_t N, const int32_t* lane_e,
                                    const int32_t* lane_m, int32_t size, int32_t block_size,
                                    const mxq_arith_spec* arith, int32_t force_general, mxq_stream_t stream) {
  if (int rc = check_common(K, M, N, 1, lane_e, lane_m, size, block_size, arith)) return rc;
  if (M == 0 || N == 0) return MXQ_OK;
  if (!P_A || !X_A || !P_B || !X_B || !C) return mxq::invalid("mxq_systolic_noalloc: NULL pointer");
  if (mxq::ceil_div(M, 32) * mxq::ceil_div(N, 32) > kScratchWords)
    return mxq::invalid("mxq_systolic_noalloc: ceil(M/32) * ceil(N/32) exceeds its 262144 tile flags "
                        "(use mxq_systolic with a workspace)");
  hipStream_t st = mxq::as_stream(stream);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  ScratchSlot* sl = nullptr;
  if (int rc = slot_on_device(st, &sl)) return rc;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  hipError_t err = hipStreamIsCapturing(st, &cap);
  if (err != hipSuccess) return hip_fail("hipStreamIsCapturing", err);
  const bool captured = cap != hipStreamCaptureStatusNone;
  if (!captured && sl->pending && sl->last != st) {
    err = hipEventQuery(sl->done);
    if (err == hipErrorNotReady) {
      mxq::set_error("mxq_systolic_noalloc: a call on another stream is still running on this GPU and holds its "
                     "scratch array; order the calls (one stream, or an event between them)");
      return MXQ_EBUSY;
    }
    if (err != hipSuccess) return hip_fail("hipEventQuery", err);
  }
  // every flag the general kernel reads is written by the fast kernel of the same call first: nothing in the
  // array has to start at zero
  SysArgs a{};
  a.A = {P_A, M, 0}; a.XA = {X_A, M, 0}; a.B = {P_B, N, 0}; a.XB = {X_B, N, 0};
  a.C = C; a.ldc = N; a.batch_c = 0; a.flags = sl->p;
  a.K = K; a.M = M; a.N = N; a.size = size; a.block_size = block_size; a.ar = *arith;
  if (int rc = run_systolic(a, lane_e, lane_m, 1, force_general, st)) return rc;
  if (!captured) {
    err = hipEventRecord(sl->done, st);
    if (err != hipSuccess) return hip_fail("hipEventRecord", err);
    sl->last = st;
    sl->pending = true;
  }
  return MXQ_OK;
}

extern "C" int64_t mxq_systolic_workspace(int64_t K, int64_t M, int64_t N, int64_t count) {
  if (K < 0 || M <= 0 || N <= 0 || count <= 0) return 1;
  // a flag per smallest fast tile, room for the dispatch order of the largest number of fast tiles, and a byte
  // per problem, 32-row stage and 32-column group of A and of B (the rows k_end leaves out)
  const int64_t suffix = count * mxq::ceil_div(K, KT) * (mxq::ceil_div(M, 32) + mxq::ceil_div(N, 32));
  return 2 * mxq::ceil_div(M, 32) * mxq::ceil_div(N, 32) * count + mxq::ceil_div(suffix, 4);
}
