// Fused MX block quantization for gfx950.
//
// A tensor is viewed as (outer, n, inner) with the block axis n in the middle.  Three layouts:
//   split    (block 32): eight lanes of a wavefront (or 32) share one block column of VEC adjacent columns, four rows
//            each (or one); their maxima meet through cross-lane exchanges; the block stays in registers.
//   row      (inner == 1, block 32): eight lanes own one contiguous block, four elements each.
//   strided  (any other block size): one thread per block column, the block read twice.
// Kernels are specialised on the element rule and, for the OCP grid and the microxcaling step, on the
// rounding mode.
// Step 1 (the scale) runs once per block and column; step 2 (the element grid) once per element.  The
// division by the scale is a multiply by its reciprocal when the scale is a normal power of two (then both
// are the same correctly rounded value) and an IEEE division otherwise (the 1e-38 floor is not a power of two).
#pragma once
#include "mxq_common.h"
#include "mxq_numerics.h"
#include "ocp_hw.h"

#include <stdlib.h>
#include <type_traits>

namespace mxq_quant {


struct bf16_t { uint16_t v; };
struct f16_t { uint16_t v; };

__device__ __forceinline__ float to_f32(float x) { return x; }
__device__ __forceinline__ float to_f32(bf16_t x) { return u2f((uint32_t)x.v << 16); }
__device__ __forceinline__ float to_f32(f16_t x) { return (float)__builtin_bit_cast(_Float16, x.v); }

// VEC adjacent elements at any element's address: gfx950's vector memory takes them there as one access.
template <typename T, int VEC>
struct __attribute__((packed, aligned(sizeof(T)))) VecT { T v[VEC]; };

template <typename T, int VEC>
__device__ __forceinline__ void load_vec(const T* p, float (&out)[VEC]) {
  const VecT<T, VEC> r = *reinterpret_cast<const VecT<T, VEC>*>(p);
#pragma unroll
  for (int j = 0; j < VEC; ++j) out[j] = to_f32(r.v[j]);
}

template <int VEC>
__device__ __forceinline__ void store_vec(float* p, const float (&in)[VEC]) {
  VecT<float, VEC> r;
#pragma unroll
  for (int j = 0; j < VEC; ++j) r.v[j] = in[j];
  *reinterpret_cast<VecT<float, VEC>*>(p) = r;
}

// Codes are written once and not read back by this kernel: streaming (non-temporal) stores.
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));   // at any element's address
template <int VEC>
__device__ __forceinline__ void store_vec_nt(float* p, const float (&in)[VEC]) {
  if constexpr (VEC == 4) {
    f32x4 r = {in[0], in[1], in[2], in[3]};
    __builtin_nontemporal_store(r, reinterpret_cast<f32x4_any*>(p));
  } else {
#pragma unroll
    for (int j = 0; j < VEC; ++j) __builtin_nontemporal_store(in[j], p + j);
  }
}

// Where a kernel's codes and scales go; the sink also runs step 2 (the element rule) on the scaled values z.
//   FloatSink  float32 P and X, the reference's outputs (codes written with streaming stores).
//   ByteSink   one element-code byte per element and one E8M0 byte per scale (mx_encode, e8m0_encode); a value
//              neither format holds sets *err (a zero block's scale is free, its value being 0 under any).
// `at` is an element index of P (or X); VEC consecutive elements, at any of them.
struct FloatSink {
  float* P;
  float* X;
  static constexpr int kBytes = 4;
  template <int ELEM, int MODE, int VEC>
  __device__ __forceinline__ void elems(int64_t at, const float (&z)[VEC], const mxq_block_spec& s) const {
    float q[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) q[j] = elem_qm<ELEM, MODE>(z[j], s);
    store_vec_nt<VEC>(P + at, q);
  }
  template <int VEC>
  __device__ __forceinline__ void scales(int64_t at, const float (&xs)[VEC], const bool (&)[VEC]) const {
    store_vec<VEC>(X + at, xs);
  }
  // The OCP grid rounded to nearest even by the hardware conversions (ocp_hw.h; the caller has checked the
  // range): the rows of a lane's strip of VEC (4 or 8) columns, rows [0, live) stored.
  template <int ROWS, int VEC>
  __device__ __forceinline__ void hw_rows(int64_t at, int64_t stride, const float (&v)[ROWS][VEC], int live,
                                          const mxq_block_spec& s) const {
    float z[ROWS * VEC];
#pragma unroll
    for (int i = 0; i < ROWS; ++i)
#pragma unroll
      for (int j = 0; j < VEC; ++j) z[VEC * i + j] = v[i][j];
    mxq_ocp_hw::values<ROWS * VEC>(z, s.e, s.m);
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      if (i >= live) break;
#pragma unroll
      for (int q = 0; q < VEC / 4; ++q) {
        const float o[4] = {z[VEC * i + 4 * q], z[VEC * i + 4 * q + 1], z[VEC * i + 4 * q + 2], z[VEC * i + 4 * q + 3]};
        store_vec_nt<4>(P + at + (int64_t)i * stride + 4 * q, o);
      }
    }
  }
  // The first `live` of four scaled values, converted as hw_rows does.
  __device__ __forceinline__ void hw_four(int64_t at, const float (&v)[4], int live, const mxq_block_spec& s) const {
    float z[4] = {v[0], v[1], v[2], v[3]};
    mxq_ocp_hw::four_values(z, s.e, s.m);
    if (live == 4) {
      store_vec_nt<4>(P + at, z);
    } else {
#pragma unroll
      for (int j = 0; j < 3; ++j)
        if (j < live) P[at + j] = z[j];
    }
  }
  __device__ __forceinline__ bool hw_format(const mxq_block_spec&) const { return true; }
};

template <int VEC>
__device__ __forceinline__ void store_bytes(uint8_t* p, uint32_t w) {
  __builtin_memcpy(p, &w, VEC);
}

// W words of code bytes (1, 2 or 4: 4, 8 or 16 bytes, at any address), one store.
// The byte sink's stores: plain, not streaming.  A wave writes 64 bytes of a code row and the next wave the rest of
// its 128-byte line; streaming stores of those halves wrote 1.28x the code and scale bytes (bf16 8192 x 8192: 88.4 MB for 69.2),
// plain ones exactly them, in the same time.  (The float sink's rows are whole lines; its streaming stores keep
// 268 MB of codes out of L2 and run faster than plain ones.)
template <int W>
__device__ __forceinline__ void store_words(uint8_t* p, const uint32_t (&w)[W]) {
  __builtin_memcpy(p, w, 4 * W);
}

// The element format's constants for the byte sink's short encoder.
struct CodeConsts {
  uint32_t nmin;      // bit pattern of 2^emin, the smallest normal
  uint32_t nshift;    // 23 - m
  uint32_t nsub;      // (127 - bias) << m: float32 exponent bias to the format's, in code position
  uint32_t lowmask;   // the float32 fraction bits below the format's m
  uint32_t maxbits;   // bit pattern of the largest finite value
  float sub_mul;      // 2^(m - emin): a subnormal value in units of the format's subnormal step
  int sign_at;        // e + m
};

__host__ __device__ inline CodeConsts code_consts(int e, int m) {
  CodeConsts k{};
  const int bias = (1 << (e - 1)) - 1, emin = 1 - bias;
  k.nmin = (uint32_t)(emin + 127) << 23;
  k.nshift = (uint32_t)(23 - m);
  k.nsub = (uint32_t)(127 - bias) << m;
  k.lowmask = (1u << (23 - m)) - 1u;
  int emax = (1 << e) - 1 - bias;                  // largest exponent field's exponent
  uint32_t mmax = (1u << m) - 1u;                   // largest mantissa there
  if (e == 5 && m == 2) emax -= 1;                  // E5M2: the top exponent field is Inf / NaN
  if (e == 4 && m == 3) mmax -= 1;                  // E4M3: S.1111.111 is NaN
  k.maxbits = ((uint32_t)(emax + 127) << 23) | (mmax << (23 - m));
  k.sub_mul = __builtin_bit_cast(float, (uint32_t)(m - emin + 127) << 23);
  k.sign_at = e + m;
  return k;
}

// The code of a value the element rule put on the format's grid: normal, (bits >> (23 - m)) less the exponent
// bias difference; subnormal (or zero), its multiple of the subnormal step.  `good` is false for anything
// else (beyond the largest finite value, a special, or off the grid: the qtorch grid's smallest values), which
// then takes mx_encode.
__device__ __forceinline__ uint32_t short_encode(float q, const CodeConsts& k, bool& good) {
  const uint32_t u = f2u(q), a = u & 0x7FFFFFFFu;
  const bool nrm = a >= k.nmin;
  const float t = u2f(a) * k.sub_mul;
  const uint32_t cs = __float2uint_rz(t);            // saturating convert: any t is defined
  const uint32_t mag = nrm ? (a >> k.nshift) - k.nsub : cs;
  good = a <= k.maxbits && (nrm ? (a & k.lowmask) == 0u : (float)cs == t);
  return mag | ((u >> 31) << k.sign_at);
}

struct ByteSink {
  uint8_t* P;
  uint8_t* X;
  int32_t* err;
  int e, m;
  CodeConsts k;
  uint32_t maxcode;    // the code of the largest finite value
  static constexpr int kBytes = 1;
  // mxgemmini's ocp grid without `via` yields the code from its own roundings (ocp_code_t); every other rule
  // rounds to float32 and the code is read off the value (short_encode).  Specials, and values the grid made
  // that the format lacks, take mx_encode.
  template <int ELEM, int MODE, int VEC>
  __device__ __forceinline__ void elems(int64_t at, const float (&z)[VEC], const mxq_block_spec& s) const {
    if constexpr (VEC == 8 || VEC == 16) {
      uint32_t w[VEC / 4];
#pragma unroll
      for (int q = 0; q < VEC / 4; ++q) {
        const float z4[4] = {z[4 * q], z[4 * q + 1], z[4 * q + 2], z[4 * q + 3]};
        w[q] = word<ELEM, MODE, 4>(z4, s);
      }
      store_words<VEC / 4>(P + at, w);
    } else {
      store_bytes<VEC>(P + at, word<ELEM, MODE, VEC>(z, s));
    }
  }
  // The codes of VEC (at most 4) scaled values, code j in byte j.
  template <int ELEM, int MODE, int VEC>
  __device__ __forceinline__ uint32_t word(const float (&z)[VEC], const mxq_block_spec& s) const {
    uint32_t w = 0u;
    bool all_good = true;
    if constexpr (ELEM == MXQ_ELEM_OCP && MODE >= 0) {
      if (s.via_e == 0) {
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
          bool good;
          w |= ocp_code_t<MODE>(z[j], e, m, maxcode, &good) << (8 * j);
          all_good = all_good && good;
        }
        return all_good ? w : general_codes<ELEM, MODE, VEC>(z, s);
      }
    }
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      bool good;
      w |= short_encode(elem_qm<ELEM, MODE>(z[j], s), k, good) << (8 * j);
      all_good = all_good && good;
    }
    return all_good ? w : general_codes<ELEM, MODE, VEC>(z, s);
  }
  template <int ELEM, int MODE, int VEC>
  __device__ __forceinline__ uint32_t general_codes(const float (&z)[VEC], const mxq_block_spec& s) const {
    bool ok = true;
    uint32_t w = 0u;
#pragma unroll
    for (int j = 0; j < VEC; ++j) w |= mx_encode(elem_qm<ELEM, MODE>(z[j], s), e, m, &ok) << (8 * j);
    if (!ok) atomicOr(err, 1);
    return w;
  }
  // hw_rows of FloatSink with the codes themselves (the byte format is the element format: e, m == s.e, s.m).
  template <int ROWS, int VEC>
  __device__ __forceinline__ void hw_rows(int64_t at, int64_t stride, const float (&v)[ROWS][VEC], int live,
                                          const mxq_block_spec& s) const {
    float z[ROWS * VEC];
#pragma unroll
    for (int i = 0; i < ROWS; ++i)
#pragma unroll
      for (int j = 0; j < VEC; ++j) z[VEC * i + j] = v[i][j];
    // the conversions take at most 32 values: in chunks of rows
    constexpr int CH = ROWS * VEC <= 32 ? ROWS * VEC : 32;
    uint32_t w[ROWS * VEC / 4];
#pragma unroll
    for (int c0 = 0; c0 < ROWS * VEC; c0 += CH) {
      float zc[CH];
      uint32_t wc[CH / 4];
#pragma unroll
      for (int k = 0; k < CH; ++k) zc[k] = z[c0 + k];
      mxq_ocp_hw::codes<CH>(zc, s.e, s.m, wc);
#pragma unroll
      for (int k = 0; k < CH / 4; ++k) w[c0 / 4 + k] = wc[k];
    }
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      if (i >= live) break;
      uint32_t row[VEC / 4];
#pragma unroll
      for (int q = 0; q < VEC / 4; ++q) row[q] = w[i * (VEC / 4) + q];
      store_words<VEC / 4>(P + at + (int64_t)i * stride, row);
    }
  }
  __device__ __forceinline__ void hw_four(int64_t at, const float (&v)[4], int live, const mxq_block_spec& s) const {
    uint32_t w[1];
    mxq_ocp_hw::four_codes(v, s.e, s.m, w);
    if (live == 4) {
      store_words<1>(P + at, w);
    } else {
#pragma unroll
      for (int j = 0; j < 3; ++j)
        if (j < live) P[at + j] = (uint8_t)(w[0] >> (8 * j));
    }
  }
  // the codes the conversions give are the byte format's when it is the grid's
  __device__ __forceinline__ bool hw_format(const mxq_block_spec& s) const { return e == s.e && m == s.m; }
  template <int VEC>
  __device__ __forceinline__ void scales(int64_t at, const float (&xs)[VEC], const bool (&zero)[VEC]) const {
    bool ok = true;
    uint32_t w[(VEC + 3) / 4] = {};
#pragma unroll
    for (int j = 0; j < VEC; ++j) w[j / 4] |= e8m0_encode(xs[j], zero[j], &ok) << (8 * (j % 4));
    if constexpr (VEC >= 8) store_words<VEC / 4>(X + at, w);
    else store_bytes<VEC>(X + at, w[0]);
    if (!ok) atomicOr(err, 2);
  }
};

// (o, b, column group) of a flat thread index over outer * nb * groups.
__device__ __forceinline__ void split_index(int64_t t, int64_t groups, int64_t nb, int64_t& o, int64_t& b,
                                            int64_t& g) {
  if (t < 0x7FFFFFFF && groups < 0x7FFFFFFF && nb < 0x7FFFFFFF) {
    const uint32_t tt = (uint32_t)t, gg = (uint32_t)groups, nn = (uint32_t)nb;
    const uint32_t ob = tt / gg;
    g = tt - ob * gg;
    o = ob / nn;
    b = ob - (uint32_t)o * nn;
  } else {
    const int64_t ob = t / groups;
    g = t - ob * groups;
    o = ob / nb;
    b = ob - o * nb;
  }
}

// z = v / X for the VEC block columns of a lane: a multiply by the exact reciprocal when every scale of the
// wave is a normal power of two (the same correctly rounded value), the IEEE division otherwise.
template <int VEC>
__device__ __forceinline__ bool wave_needs_div(const Div (&d)[VEC]) {
  bool need = false;
#pragma unroll
  for (int j = 0; j < VEC; ++j) need |= (d[j].inv == 0.0f);
  return __any(need);
}

// Whether a wave's scaled values may take the hardware conversions (ocp_hw.h), and `hs`, the spec that names them
// their element format.  Every scaled value has to be finite and within their range (a column's largest |z| is its
// maximum scaled, the division being monotone) and the grid has to saturate where they do (max_norm the format's
// own).  microxcaling's "even" (mxq/microxcaling/elemwise.py:29-60) is the OCP grid at nearest even, saturating at
// max_norm, with one exception: the float32 just below half the smallest subnormal step, which its float32
// floor(|A| + 0.5) rounds up to that step.  So with every value and scaled value finite and none of that magnitude,
// the values, clamped here to +-max_norm, go to the conversions.
// N: the values a lane converts at once.  am, d: the block columns' maxima (as bit patterns) and divisors; v: the lane's scaled values.
template <int ELEM, int N, typename SINK, int COLS, int ROWS, int VEC>
__device__ __forceinline__ bool hw_gate(const SINK& out, const mxq_block_spec& s, mxq_block_spec& hs,
                                        const uint32_t (&am)[COLS], const Div (&d)[COLS], bool div,
                                        float (&v)[ROWS][VEC]) {
  constexpr bool MS = ELEM == MXQ_ELEM_MICROSOFT;
  if constexpr (MS) hs.m = s.m - 2;                  // microxcaling's mbits count the sign and hidden bits
  if (!(s.via_e == 0 && mxq_ocp_hw::has_hw_n<N>(hs.e, hs.m) && out.hw_format(hs) &&
        s.max_norm == mxq_ocp_hw::fmt_max(hs.e, hs.m)))
    return false;
  const float lim = MS ? INFINITY : mxq_ocp_hw::hw_limit(hs.e, hs.m);
  bool ok = true;
#pragma unroll
  for (int j = 0; j < COLS; ++j) {                   // finite inputs and scaled values (a NaN scale fails)
    const float a = u2f(am[j]);
    const float zm = !s.scale_rule ? a : (div ? apply_div(a, d[j]) : a * d[j].inv);
    ok = ok && am[j] < 0x7F800000u && zm < lim;
  }
  if constexpr (MS) {
    const int emin = 2 - (1 << (hs.e - 1));
    const uint32_t odd = (uint32_t)(127 + emin - hs.m - 1) << 23;  // 2^(emin - m - 1), then one float below
#pragma unroll
    for (int i = 0; i < ROWS; ++i)
#pragma unroll
      for (int j = 0; j < VEC; ++j) ok = ok && (f2u(v[i][j]) & 0x7FFFFFFFu) != odd - 1u;
  }
  const bool hw = __all(ok);
  if constexpr (MS) {
    if (hw) {
#pragma unroll
      for (int i = 0; i < ROWS; ++i)
#pragma unroll
        for (int j = 0; j < VEC; ++j) v[i][j] = fminf(fmaxf(v[i][j], -s.max_norm), s.max_norm);
    }
  }
  return hw;
}

// Any block size (read twice: once for the amax, once for the elements), one thread per block column of
// VEC adjacent columns, inner % VEC == 0.  A thread walks its block alone, so rows that are not whole fours take a column
// or two a thread rather than four with the last group moved back: 4096 x 513 float32 in blocks of 64 33 us (47 with
// four), 4096 x 4097 56 (72).
template <typename T, int ELEM, int MODE, int VEC, typename SINK>
__global__ void __launch_bounds__(256) k_quant_strided(const T* __restrict__ V, const SINK out, int64_t outer,
                                                       int64_t n, int64_t inner, int64_t bs, int64_t nb,
                                                       mxq_block_spec s) {
  const int64_t groups = inner / VEC;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= outer * nb * groups) return;
  int64_t o, b, g;
  split_index(t, groups, nb, o, b, g);
  const int64_t k0 = b * bs;
  const int64_t rows = (n - k0 < bs) ? n - k0 : bs;
  const int64_t off = (o * n + k0) * inner + g * VEC;
  float amax[VEC];
#pragma unroll
  for (int j = 0; j < VEC; ++j) amax[j] = 0.0f;
  for (int64_t r = 0; r < rows; ++r) {
    float v[VEC];
    load_vec<T, VEC>(V + off + r * inner, v);
#pragma unroll
    for (int j = 0; j < VEC; ++j) amax[j] = amax_combine(amax[j], fabsf(v[j]));
  }
  Div d[VEC];
  float xs[VEC];
#pragma unroll
  for (int j = 0; j < VEC; ++j) {
    xs[j] = block_scale(amax[j], s);
    d[j] = make_div(xs[j]);
  }
  for (int64_t r = 0; r < rows; ++r) {
    float v[VEC], z[VEC];
    load_vec<T, VEC>(V + off + r * inner, v);
#pragma unroll
    for (int j = 0; j < VEC; ++j) z[j] = s.scale_rule ? apply_div(v[j], d[j]) : v[j];
    out.template elems<ELEM, MODE, VEC>(off + r * inner, z, s);
  }
  bool zero[VEC];
#pragma unroll
  for (int j = 0; j < VEC; ++j) zero[j] = amax[j] == 0.0f;
  out.template scales<VEC>((o * nb + b) * inner + g * VEC, xs, zero);
}

// Block size 32 with R lanes of one wavefront sharing a block column: lane l of a wave takes row part
// r = l / (64 / R) (rows [r * 32/R, (r+1) * 32/R) of the block) and column group cg_base + l % (64 / R); the R
// partial maxima meet through cross-lane exchanges.  Few values per lane keep many waves resident, which is
// what hides the HBM latency here (measured on MI355X: R = 8, VEC = 4 is the fastest layout on 8192 x 8192
// bf16 and on 4096 x 512 float32).
//   * The wave's index is uniform, so the (outer, block, column-group) split of it runs in scalar registers.
//   * A whole block (all but a tail) loads without per-row conditions; lanes past the last column group read
//     the last one's columns and store nothing.
//   * Rows of any length and address: a group of VEC columns is one access wherever it begins (rows that
//     were not whole fours had a column a lane: a call on 5632 x 333 float32 20.9 -> 10.7 us, 4096 x 2049 27.9 -> 19.9).
//   * The block maximum is the largest |v| bit pattern (non-negative floats order like their patterns, and
//     every NaN pattern lies above +Inf, so a NaN wins as torch.amax's does).
//   * The R lanes of a column group hold the same maxima after the exchanges; lane r computes the scales of
//     columns r, r + R, ... alone and the others read them (ceil(VEC / R) scale rule evaluations per lane
//     instead of VEC).
// WHOLE: inner % VEC == 0 (the column's clamp, 64-bit work in every lane, costs 8192 x 8192 bfloat16 64 -> 67 us).
template <typename T, int ELEM, int MODE, int VEC, int R, bool WHOLE, typename SINK>
__global__ void __launch_bounds__(256) k_quant_split(const T* __restrict__ V, const SINK out, int64_t outer,
                                                     int64_t n, int64_t inner, mxq::DivU31 nb_div,
                                                     mxq::DivU31 wpr_div, mxq_block_spec s) {
  constexpr int CPW = 64 / R;          // column groups per wave
  constexpr int ROWS = 32 / R;         // rows per lane
  constexpr int PER = (VEC + R - 1) / R;  // scales each lane evaluates
  const int64_t groups = WHOLE ? inner / VEC : (inner + VEC - 1) / VEC;
  const int lane = threadIdx.x & 63;
  const int64_t nb = nb_div.d, waves_per_row = wpr_div.d;
  // the launch keeps the wave count below 2^31
  const uint32_t wave = blockIdx.x * (256 / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if ((int64_t)wave >= outer * nb * waves_per_row) return;   // whole waves only: the exchanges below see every lane
  const uint32_t wr = mxq::divu31(wave, wpr_div);      // (o, b) flattened
  const uint32_t o32 = mxq::divu31(wr, nb_div);
  const int64_t o = o32, b = wr - o32 * nb_div.d;
  const int64_t k0 = b * 32;
  const int rows = (int)((n - k0 < 32) ? n - k0 : 32);
  const int c = lane % CPW, r = lane / CPW;
  const int64_t cg = (int64_t)(wave - wr * wpr_div.d) * CPW + c;
  const bool live = cg < groups;
  // the last group ends on the last column, sharing some with the group before it (the same values stored twice)
  const int64_t col = WHOLE ? (live ? cg : 0) * VEC : (cg * VEC < inner - VEC ? cg * VEC : inner - VEC);
  const T* src = V + (o * n + k0 + r * ROWS) * inner + col;

  float v[ROWS][VEC];
  uint32_t am[VEC];
#pragma unroll
  for (int j = 0; j < VEC; ++j) am[j] = 0u;
  if (rows == 32) {
#pragma unroll
    for (int i = 0; i < ROWS; ++i) load_vec<T, VEC>(src + (int64_t)i * inner, v[i]);
  } else {
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      if (r * ROWS + i < rows) {
        load_vec<T, VEC>(src + (int64_t)i * inner, v[i]);
      } else {
#pragma unroll
        for (int j = 0; j < VEC; ++j) v[i][j] = 0.0f;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < ROWS; ++i)
#pragma unroll
    for (int j = 0; j < VEC; ++j) am[j] = max(am[j], f2u(v[i][j]) & 0x7FFFFFFFu);
#pragma unroll
  for (int step = CPW; step < 64; step <<= 1)
#pragma unroll
    for (int j = 0; j < VEC; ++j) am[j] = max(am[j], (uint32_t)__shfl_xor((int)am[j], step, 64));
  // lane r evaluates the scales of columns r, r + R, ... of its group (those below VEC); every lane then reads
  // column j's from lane c + (j % R) * CPW
  float own[PER];
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    uint32_t mine = am[q * R];
#pragma unroll
    for (int jj = 1; jj < R; ++jj)
      if (q * R + jj < VEC) mine = (r == jj) ? am[q * R + jj] : mine;
    own[q] = block_scale(u2f(mine), s);
  }
  float xs[VEC];
  Div d[VEC];
#pragma unroll
  for (int j = 0; j < VEC; ++j) {
    xs[j] = __shfl(own[j / R], c + (j % R) * CPW, 64);
    d[j] = make_div(xs[j]);
  }
  const bool div = s.scale_rule && wave_needs_div<VEC>(d);
  if (div) {
#pragma unroll
    for (int i = 0; i < ROWS; ++i)
#pragma unroll
      for (int j = 0; j < VEC; ++j) v[i][j] = apply_div(v[i][j], d[j]);
  } else if (s.scale_rule) {
#pragma unroll
    for (int i = 0; i < ROWS; ++i)
#pragma unroll
      for (int j = 0; j < VEC; ++j) v[i][j] = v[i][j] * d[j].inv;
  }
  constexpr bool HW = VEC >= 4 && MODE == MXQ_RNE && (ELEM == MXQ_ELEM_OCP || ELEM == MXQ_ELEM_MICROSOFT);
  mxq_block_spec hs = s;
  bool hw = false;
  if constexpr (HW) hw = hw_gate<ELEM, ROWS * VEC>(out, s, hs, am, d, div, v);
  if (!live) return;
  const int64_t dst = (o * n + k0 + r * ROWS) * inner + col;
  if constexpr (HW) {
    if (hw) out.template hw_rows<ROWS, VEC>(dst, inner, v, rows == 32 ? ROWS : rows - r * ROWS, hs);
  }
  if (!hw) {
    // the element grid in software, one row at a time from a second read of the row (the same loads and the
    // same scaling give the same values): the registers of this rare path are one row's, so the kernel's
    // count is the conversions' path's and more waves fit on a SIMD
#pragma unroll 1
    for (int i = 0; i < ROWS; ++i) {
      if (rows == 32 || r * ROWS + i < rows) {
        float z[VEC];
        load_vec<T, VEC>(src + (int64_t)i * inner, z);
        if (div) {
#pragma unroll
          for (int j = 0; j < VEC; ++j) z[j] = apply_div(z[j], d[j]);
        } else if (s.scale_rule) {
#pragma unroll
          for (int j = 0; j < VEC; ++j) z[j] = z[j] * d[j].inv;
        }
        out.template elems<ELEM, MODE, VEC>(dst + (int64_t)i * inner, z, s);
      }
    }
  }
  if (r == 0) {
    bool zero[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) zero[j] = am[j] == 0u;
    out.template scales<VEC>((o * nb + b) * inner + col, xs, zero);
  }
}

// inner == 1, blocks of 32 contiguous elements of rows of any length n: eight lanes per block, four elements a
// lane (those past the row's end are 0 and are not stored), one access wherever they begin.  A wave takes Q runs
// of eight blocks, and lane l of a block's eight evaluates the scale of its l % Q-th run for the others: the scale
// rule, some hundred instructions, is what Q = 1 spends most of its time on.
// Half-precision rows of 2001 values to E2M3, 2331 of them: 71 -> 12.6 us, 16,384: 451 -> 35 us (their blocks went
// one a wave through k_quant_split, an element a lane); of 2048, 16,384: 44 -> 33 us, through microxcaling's grid
// 72 -> 33 us (no conversions were used for contiguous blocks).  What is left is memory: 33 us is 6.1 TB/s.
template <typename T, int ELEM, int MODE, int Q, bool WHOLE, typename SINK>
__global__ void __launch_bounds__(256) k_quant_row(const T* __restrict__ V, const SINK out, int64_t nblocks,
                                                   int64_t outer, int64_t n, mxq::DivU31 nb_div, mxq_block_spec s) {
  static_assert(Q >= 1 && Q <= 8, "a lane evaluates one scale");
  const int lane = threadIdx.x & 63, l8 = lane & 7;
  const int64_t total = outer * n;
  const int64_t first = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * (8 * Q) + (lane >> 3);
  // this lane's four elements of run q: their place, and how many of them there are
  auto place = [&](int q, int64_t& blk, int64_t& off) {
    blk = first + 8 * q;
    if constexpr (WHOLE) {                              // rows are whole blocks: no row to find, no part of one
      off = blk * 32 + l8 * 4;
      return blk < nblocks ? 4 : 0;
    }
    const int64_t o = mxq::divu31((uint32_t)blk, nb_div);
    const int64_t k = (blk - o * nb_div.d) * 32 + l8 * 4;
    off = o * n + k;
    return blk < nblocks ? (int)(n - k < 4 ? n - k : 4) : 0;
  };
  // every run's load is issued before any is waited for: four elements from each lane's place whatever the row
  // holds there, moved back where that would leave the tensor (of at least four elements)
  VecT<T, 4> w[Q];
  int64_t blk[Q], off[Q];
  int left[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    left[q] = place(q, blk[q], off[q]);
    w[q] = *reinterpret_cast<const VecT<T, 4>*>(V + (off[q] < total - 4 ? off[q] : total - 4));
  }
  float v[Q][4];
  uint32_t am[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    if (!WHOLE && off[q] > total - 4) {              // the tensor's last elements
      const int64_t back = off[q] - (total - 4);
#pragma unroll
      for (int j = 0; j < 3; ++j) w[q].v[j] = back == 1 ? w[q].v[j + 1] : back == 2 ? w[q].v[j < 2 ? j + 2 : 3] : w[q].v[3];
    }
    am[q] = 0u;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[q][j] = WHOLE || j < left[q] ? to_f32(w[q].v[j]) : 0.0f;
      am[q] = max(am[q], f2u(v[q][j]) & 0x7FFFFFFFu);
    }
  }
  // all 64 lanes take part in the exchanges; lanes past the end belong to no live block
#pragma unroll
  for (int step = 1; step < 8; step <<= 1)
#pragma unroll
    for (int q = 0; q < Q; ++q) am[q] = max(am[q], (uint32_t)__shfl_xor((int)am[q], step, 8));
  uint32_t mine = am[0];
#pragma unroll
  for (int q = 1; q < Q; ++q) mine = l8 % Q == q ? am[q] : mine;
  const float own = block_scale(u2f(mine), s);
  Div d[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) d[q] = make_div(Q == 1 ? own : __shfl(own, q, 8));
  constexpr bool HW = MODE == MXQ_RNE && (ELEM == MXQ_ELEM_OCP || ELEM == MXQ_ELEM_MICROSOFT);
  if constexpr (WHOLE && !HW) {
    // whole rows through a software grid: straight through, without the code for parts of a lane's four (to bytes, ties
    // away, 8192 x 8192 half-precision values 84 us, 97 by the general code below)
    static_assert(Q == 1, "a software grid takes one run a wave");
    if (left[0] == 0) return;
    float z[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) z[j] = s.scale_rule ? apply_div(v[0][j], d[0]) : v[0][j];
    out.template elems<ELEM, MODE, 4>(off[0], z, s);
    if (l8 == 0) {
      const float x1[1] = {own};
      const bool z1[1] = {am[0] == 0u};
      out.template scales<1>(blk[0], x1, z1);
    }
    return;
  }
  const bool div = s.scale_rule && wave_needs_div<Q>(d);
  mxq_block_spec hs = s;
  bool hw = false;
  if constexpr (HW) {
    if (div) {
#pragma unroll
      for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int j = 0; j < 4; ++j) v[q][j] = apply_div(v[q][j], d[q]);
    } else if (s.scale_rule) {
#pragma unroll
      for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int j = 0; j < 4; ++j) v[q][j] = v[q][j] * d[q].inv;
    }
    hw = hw_gate<ELEM, 32>(out, s, hs, am, d, div, v);   // four_values takes every format
    if (hw) {
#pragma unroll
      for (int q = 0; q < Q; ++q)
        if (left[q] > 0) out.hw_four(off[q], v[q], left[q], hs);
    }
  }
  if constexpr (!HW) {                                 // software grids: from the registers
#pragma unroll
    for (int q = 0; q < Q; ++q) {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[q][j] = !s.scale_rule ? v[q][j] : (div ? apply_div(v[q][j], d[q]) : v[q][j] * d[q].inv);
      if (left[q] == 4) {
        out.template elems<ELEM, MODE, 4>(off[q], v[q], s);
      } else {
#pragma unroll 1
        for (int j = 0; j < left[q]; ++j) {
          const float z[1] = {j == 0 ? v[q][0] : j == 1 ? v[q][1] : v[q][2]};
          out.template elems<ELEM, MODE, 1>(off[q] + j, z, s);
        }
      }
    }
  } else if (!hw) {
    // the element grid in software, a run at a time from a second read of its elements, so that its registers are
    // one run's
#pragma unroll 1
    for (int q = 0; q < Q; ++q) {
      int64_t b, at;
      const int count = place(q, b, at);
      const Div dq = make_div(__shfl(own, q, 8));
      auto scaled = [&](float x) { return !s.scale_rule ? x : (div ? apply_div(x, dq) : x * dq.inv); };
      if (count == 4) {
        float z[4];
        load_vec<T, 4>(V + at, z);
#pragma unroll
        for (int j = 0; j < 4; ++j) z[j] = scaled(z[j]);
        out.template elems<ELEM, MODE, 4>(at, z, s);
      } else {
#pragma unroll 1
        for (int j = 0; j < count; ++j) {
          const float z[1] = {scaled(to_f32(V[at + j]))};
          out.template elems<ELEM, MODE, 1>(at + j, z, s);
        }
      }
    }
  }
#pragma unroll
  for (int q = 0; q < Q; ++q)
    if (l8 == q && blk[q] < nblocks) {
      const float x1[1] = {own};
      const bool z1[1] = {mine == 0u};
      out.template scales<1>(blk[q], x1, z1);
    }
}

// ------------------------------------------------------ code bytes of the OCP grid at nearest even, one pass
// k_pack_rne: the byte sink for the OCP element grid rounded to nearest even and saturating at the format's own
// largest value (block.mxgemmini's rounding_mode="rne" without `via`), blocks of 32 along the axis, eight
// adjacent columns a lane, R lanes of a wave per block column (32 / R rows each), as k_quant_split lays them out.
// Written for the instruction count of the common wave, whose inputs and scaled values are finite and whose
// block scales are normal powers of two:
//   * 16-bit inputs stay packed two to a register; the column maxima are packed 16-bit maxima (|x| patterns
//     order as the values do, a NaN above Inf, as in float32).
//   * one lane of each column's R evaluates the scale rule and hands the others its E8M0 byte, which is all
//     they need: the reciprocal of a normal power of two 2^k is 2^-k, read off the byte.
//   * z = fma(v, 1/X, +0): v / X correctly rounded, -0 made +0 (the grid's sign for an exact zero);
//     clamped to +-max (the grid saturates: rounding a clamped value gives the saturated one), then converted
//     by gfx950's scaled conversions at scale 1, which round to nearest even with true subnormals.
//   * FP6 through the FP8 conversions: E2M3 is E4M3's grid on z * 2^-6 and E3M2 is E5M2's on z * 2^-12 (the
//     same mantissa widths; the exponent offsets map one format's subnormal step and binades onto the other's),
//     whose code bytes, with the top exponent bits zero, move the sign from bit 7 to bit 5.  FP4 converts two
//     values into a byte, spread to one a byte.
// A wave with any other block (a non-finite value, a scale that is not a normal power of two) takes
// k_quant_split's software element path for all of its blocks.
namespace pkr {

template <typename T>
struct In;                                            // a lane's row of eight values: loads and maxima
template <>
struct In<float> {
  static constexpr int NW = 8, NA = 8;                // words per row, words of column maxima
  static constexpr uint32_t kFin = 0x7F800000u;       // |x| patterns below this are finite
  __device__ static void load(const float* p, uint32_t (&w)[NW]) {
    __builtin_memcpy(w, p, 16);
    __builtin_memcpy(w + 4, p + 4, 16);
  }
  __device__ static void amax(uint32_t (&am)[NA], const uint32_t (&w)[NW]) {
#pragma unroll
    for (int j = 0; j < NW; ++j) am[j] = max(am[j], w[j] & 0x7FFFFFFFu);
  }
  __device__ static uint32_t column(const uint32_t (&am)[NA], int j) { return am[j]; }
  __device__ static float f32(uint32_t a) { return u2f(a); }
  __device__ static float value(const uint32_t (&w)[NW], int j) { return u2f(w[j]); }
};
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t max_u16x2(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a),
                                                               __builtin_bit_cast(u16x2, b)));
}
struct In16 {
  static constexpr int NW = 4, NA = 4;
  template <typename T>
  __device__ static void load(const T* p, uint32_t (&w)[NW]) {
    __builtin_memcpy(w, p, 16);
  }
  __device__ static void amax(uint32_t (&am)[NA], const uint32_t (&w)[NW]) {
#pragma unroll
    for (int j = 0; j < NW; ++j) am[j] = max_u16x2(am[j], w[j] & 0x7FFF7FFFu);
  }
  __device__ static uint32_t column(const uint32_t (&am)[NA], int j) { return (am[j >> 1] >> (16 * (j & 1))) & 0xFFFFu; }
};
template <>
struct In<bf16_t> : In16 {
  static constexpr uint32_t kFin = 0x7F80u;
  __device__ static float f32(uint32_t a) { return u2f(a << 16); }
  __device__ static float value(const uint32_t (&w)[NW], int j) {
    return (j & 1) ? u2f(w[j >> 1] & 0xFFFF0000u) : u2f(w[j >> 1] << 16);
  }
};
template <>
struct In<f16_t> : In16 {
  static constexpr uint32_t kFin = 0x7C00u;
  __device__ static float f32(uint32_t a) { return (float)__builtin_bit_cast(_Float16, (uint16_t)a); }
  __device__ static float value(const uint32_t (&w)[NW], int j) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)(w[j >> 1] >> (16 * (j & 1))));
  }
};

// Per element format (e, m): the pre-scale exponent of the conversion used, the clamp, the four codes.
template <int E, int M>
struct Code {
  static_assert((E == 4 && M == 3) || (E == 5 && M == 2) || (E == 2 && M == 3) || (E == 3 && M == 2) ||
                (E == 2 && M == 1), "an OCP MX element format");
  static constexpr int SH = (E == 2 && M == 3) ? 6 : ((E == 3 && M == 2) ? 12 : 0);   // z * 2^-SH converted
  static constexpr float MAXV = (E == 4) ? 448.0f : (E == 5) ? 57344.0f : (M == 3) ? 7.5f : (E == 3) ? 28.0f : 6.0f;
  static constexpr float CLAMP = MAXV / (float)(1u << SH);
  __device__ static uint32_t four(float z0, float z1, float z2, float z3) {
    if constexpr (E == 2 && M == 1) {
      uint32_t r = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(0u, z0, z1, 1.0f, 0);     // byte 0: z1 z0 nibbles
      r = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(r, z2, z3, 1.0f, 2);              // byte 2: z3 z2
      return (r & 0x000F000Fu) | ((r & 0x00F000F0u) << 4);
    } else {
      mxq_ocp_hw::s2v r = {0, 0};
      if constexpr (M == 3) {                                                         // E4M3, E2M3
        r = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(r, z0, z1, 1.0f, false);
        r = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(r, z2, z3, 1.0f, true);
      } else {                                                                        // E5M2, E3M2
        r = __builtin_amdgcn_cvt_scalef32_pk_bf8_f32(r, z0, z1, 1.0f, false);
        r = __builtin_amdgcn_cvt_scalef32_pk_bf8_f32(r, z2, z3, 1.0f, true);
      }
      const uint32_t w = __builtin_bit_cast(uint32_t, r);
      if constexpr (SH != 0) return (w & 0x1F1F1F1Fu) | ((w >> 2) & 0x20202020u);   // sign: bit 7 -> bit 5
      else return w;
    }
  }
};

}  // namespace pkr

template <typename T, int E, int M, int R>
__global__ void __launch_bounds__(256) k_pack_rne(const T* __restrict__ V, const ByteSink out, int64_t outer, int64_t n,
                                                  int64_t inner, mxq::DivU31 nb_div, mxq::DivU31 wpr_div,
                                                  mxq_block_spec s) {
  using In = pkr::In<T>;
  using Cd = pkr::Code<E, M>;
  constexpr int VEC = 8, CPW = 64 / R, ROWS = 32 / R, PER = VEC / R;
  static_assert(R == 4 || R == 8, "4 or 8 lanes per block column");
  const int64_t groups = (inner + VEC - 1) / VEC;
  const int lane = threadIdx.x & 63;
  const int64_t nb = nb_div.d;
  const uint32_t wave = blockIdx.x * (256 / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if ((int64_t)wave >= outer * nb * wpr_div.d) return;   // whole waves only: the exchanges below see every lane
  const uint32_t wr = mxq::divu31(wave, wpr_div);
  const uint32_t o32 = mxq::divu31(wr, nb_div);
  const int64_t o = o32, b = wr - o32 * nb_div.d;
  const int64_t k0 = b * 32;
  const int rows = (int)((n - k0 < 32) ? n - k0 : 32);
  const int c = lane % CPW, r = lane / CPW;
  const int64_t cg = (int64_t)(wave - wr * wpr_div.d) * CPW + c;
  const bool live = cg < groups;
  // the last group ends on the last column, sharing some with the group before it (the same values stored twice)
  const int64_t col = cg * VEC < inner - VEC ? cg * VEC : inner - VEC;
  const T* src = V + (o * n + k0 + r * ROWS) * inner + col;

  uint32_t w[ROWS][In::NW];
  uint32_t am[In::NA];
#pragma unroll
  for (int j = 0; j < In::NA; ++j) am[j] = 0u;
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    if (rows == 32 || r * ROWS + i < rows) {
      In::load(src + (int64_t)i * inner, w[i]);
    } else {
#pragma unroll
      for (int j = 0; j < In::NW; ++j) w[i][j] = 0u;
    }
    In::amax(am, w[i]);
  }
#pragma unroll
  for (int step = CPW; step < 64; step <<= 1)
#pragma unroll
    for (int j = 0; j < In::NA; ++j) {
      const uint32_t other = (uint32_t)__shfl_xor((int)am[j], step, 64);
      if constexpr (In::NA == 8) am[j] = max(am[j], other);
      else am[j] = pkr::max_u16x2(am[j], other);
    }
  // lane r evaluates the scales of columns r, r + R, ...; a column's E8M0 byte when its maximum is finite and
  // its scale a normal power of two, else 0
  float own_x[PER];
  uint32_t own_b[PER];
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    uint32_t mine = In::column(am, q * R);
#pragma unroll
    for (int jj = 1; jj < R; ++jj) mine = (r == jj) ? In::column(am, q * R + jj) : mine;
    own_x[q] = block_scale(In::f32(mine), s);
    const uint32_t u = f2u(own_x[q]), be = u >> 23;
    own_b[q] = (mine < In::kFin && (u & 0x807FFFFFu) == 0u && be >= 1u && be <= 254u) ? be : 0u;
  }
  uint32_t eb[VEC];
  bool fast = true;
#pragma unroll
  for (int j = 0; j < VEC; ++j) {
    eb[j] = (uint32_t)__shfl((int)own_b[j / R], c + (j % R) * CPW, 64);
    fast = fast && eb[j] != 0u;
  }
  const int64_t dst = (o * n + k0 + r * ROWS) * inner + col;
  const int64_t xat = (o * nb + b) * inner + col;
  if (__all(fast)) {
    if (!live) return;
    float inv[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      const int ex = 254 - (int)eb[j] - Cd::SH;                     // 2^-(k + SH), normal or subnormal
      inv[j] = u2f(ex >= 1 ? (uint32_t)ex << 23 : 1u << (22 + ex));
    }
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      float z[VEC];
#pragma unroll
      for (int j = 0; j < VEC; ++j)
        z[j] = __builtin_amdgcn_fmed3f(__builtin_fmaf(In::value(w[i], j), inv[j], 0.0f), -Cd::CLAMP, Cd::CLAMP);
      const uint32_t w0 = Cd::four(z[0], z[1], z[2], z[3]), w1 = Cd::four(z[4], z[5], z[6], z[7]);
      if (rows == 32 || r * ROWS + i < rows) store_words<2>(out.P + dst + (int64_t)i * inner, {w0, w1});
    }
    if (r == 0)
      store_words<2>(out.X + xat, {eb[0] | eb[1] << 8 | eb[2] << 16 | eb[3] << 24,
                                   eb[4] | eb[5] << 8 | eb[6] << 16 | eb[7] << 24});
    return;
  }
  // the software element path for the whole wave (k_quant_split's, on the same scales and divisions)
  float xs[VEC];
  Div d[VEC];
#pragma unroll
  for (int j = 0; j < VEC; ++j) {
    xs[j] = __shfl(own_x[j / R], c + (j % R) * CPW, 64);
    d[j] = make_div(xs[j]);
  }
  if (!live) return;
  // rows read again from memory (the same values), so that this rare path holds one row's registers
#pragma unroll 1
  for (int i = 0; i < ROWS; ++i) {
    if (rows == 32 || r * ROWS + i < rows) {
      uint32_t wi[In::NW];
      In::load(src + (int64_t)i * inner, wi);
#pragma unroll 1
      for (int h = 0; h < VEC; h += 4) {                 // four codes at a time: fewer registers again
        float z[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float v = In::value(wi, h + j);
          z[j] = s.scale_rule ? apply_div(v, d[h + j]) : v;
        }
        out.template elems<MXQ_ELEM_OCP, MXQ_RNE, 4>(dst + (int64_t)i * inner + h, z, s);
      }
    }
  }
  if (r == 0) {
    bool zero[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) zero[j] = In::column(am, j) == 0u;
    out.template scales<VEC>(xat, xs, zero);
  }
}

// V = M^T with M (inner x n) row-major in memory, blocks of 32 along n: every block is 32 contiguous elements
// of a row of M.  A workgroup quantizes a tile of 64 rows of M x 64 of n (two blocks per row): loads along M's
// rows (coalesced), eight lanes of four elements per block whose maxima meet through exchanges, and the codes
// pass through LDS to leave along P's rows (P is V-shaped: n x inner).  The same scale and element rules as
// the other layouts, per block; no copy of the transposed input is made.
constexpr int kTT = 64;

template <typename T, int ELEM, int MODE>
__global__ void __launch_bounds__(256) k_quant_t(const T* __restrict__ M, float* __restrict__ P,
                                                 float* __restrict__ X, int64_t n, int64_t inner, int64_t tiles_k,
                                                 int vec_in, int vec_out, mxq_block_spec s) {
  __shared__ float tile[kTT][kTT + 1];               // [position along n][row of M]
  const int64_t tc = blockIdx.x / tiles_k, tk = blockIdx.x - tc * tiles_k;
  const int64_t c0 = tc * kTT, k0 = tk * kTT;
  const bool full = c0 + kTT <= inner && k0 + kTT <= n;
  const int tid = threadIdx.x;
#pragma unroll
  for (int it = 0; it < 4; ++it) {
    const int id = it * 256 + tid;
    const int row = id >> 4, quad = id & 15;          // 8 consecutive lanes: one row, one block of 32
    const int64_t c = c0 + row, k = k0 + quad * 4;
    float v[4];
    if (full && vec_in) {
      load_vec<T, 4>(M + c * n + k, v);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (c < inner && k + e < n) ? to_f32(M[c * n + k + e]) : 0.0f;
    }
    uint32_t am = 0u;
#pragma unroll
    for (int e = 0; e < 4; ++e) am = max(am, f2u(v[e]) & 0x7FFFFFFFu);
    am = max(am, (uint32_t)__shfl_xor((int)am, 1, 8));
    am = max(am, (uint32_t)__shfl_xor((int)am, 2, 8));
    am = max(am, (uint32_t)__shfl_xor((int)am, 4, 8));
    const float xs = block_scale(u2f(am), s);
    const Div d = make_div(xs);
#pragma unroll
    for (int e = 0; e < 4; ++e) tile[quad * 4 + e][row] = elem_qm<ELEM, MODE>(s.scale_rule ? apply_div(v[e], d) : v[e], s);
    if ((quad & 7) == 0 && c < inner && k < n) X[(k >> 5) * inner + c] = xs;
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < 4; ++it) {
    const int id = it * 256 + tid;
    const int key = id >> 4, cq = (id & 15) * 4;
    const int64_t k = k0 + key, c = c0 + cq;
    float q[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) q[e] = tile[key][cq + e];
    if (full && vec_out) {
      store_vec_nt<4>(P + k * inner + c, q);
    } else if (k < n) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c + e < inner) P[k * inner + c + e] = q[e];
    }
  }
}

template <typename T, int ELEM, int MODE>
int launch_quant_t(const T* M, float* P, float* X, int64_t n, int64_t inner, const mxq_block_spec& q,
                   hipStream_t st) {
  mxq::KernelTimer timer("block_quantize", st);
  const int64_t tiles_k = mxq::ceil_div(n, kTT), tiles = mxq::ceil_div(inner, kTT) * tiles_k;
  if (tiles > INT32_MAX) return mxq::invalid("mxq_block_quantize_t: tensor too large");
  const int vec_in = n % 4 == 0 && reinterpret_cast<uintptr_t>(M) % (4 * sizeof(T)) == 0;
  const int vec_out = inner % 4 == 0 && reinterpret_cast<uintptr_t>(P) % 16 == 0;
  k_quant_t<T, ELEM, MODE><<<dim3((unsigned)tiles), 256, 0, st>>>(M, P, X, n, inner, tiles_k, vec_in, vec_out, q);
  return mxq::check_launch("mxq_block_quantize_t");
}

// ------------------------------------------------------------------------------------------ host side
inline int validate(const mxq_block_spec& s) {
  using mxq::invalid;
  if (s.scale_rule < MXQ_SCALE_NONE || s.scale_rule > MXQ_SCALE_OCP_NO_CLIP) return invalid("bad scale_rule");
  if (s.elem < MXQ_ELEM_NONE || s.elem > MXQ_ELEM_MICROSOFT) return invalid("bad elem rule");
  if (s.rounding < 0 || s.rounding > 2) return invalid("bad rounding code");
  if ((s.scale_rule == MXQ_SCALE_OCP || s.scale_rule == MXQ_SCALE_OCP_NO_CLIP) && (s.scale_bits < 1 || s.scale_bits > 30))
    return invalid("bad scale_bits");
  if (s.scale_rule == MXQ_SCALE_OCP_NO_CLIP && s.elem != MXQ_ELEM_MICROSOFT)
    return invalid("ocp_no_clip needs the microsoft element rule's format");
  if (s.elem == MXQ_ELEM_QTORCH || s.elem == MXQ_ELEM_IEEE) {
    if (!((s.e == 8 && s.m == 23) || (s.e >= 1 && s.e <= 8 && s.m >= 1 && s.m <= 22)))
      return invalid("unsupported widths e=" + std::to_string(s.e) + ", m=" + std::to_string(s.m));
  }
  if (s.elem == MXQ_ELEM_OCP) {
    if (!(s.e >= 2 && s.e <= 5 && s.m >= 1 && s.m <= 3)) return invalid("ocp grid needs an OCP element format");
    if (s.via_e && !((s.via_e == 8 && s.via_m == 23) || (s.via_e >= 1 && s.via_e <= 8 && s.via_m >= 1 && s.via_m <= 22)))
      return invalid("unsupported via widths");
  }
  if (s.elem == MXQ_ELEM_MICROSOFT && !(s.e >= 2 && s.e <= 8 && s.m >= 2 && s.m <= 24))
    return invalid("bad microxcaling format parameters");
  return MXQ_OK;
}

// k_pack_rne for blocks of 32 along the axis, inner >= 8: four lanes per block column (eight rows each) while that gives the chip at least 2048 waves,
// else eight (four rows each).
template <typename T>
int launch_pack_rne(const T* V, const ByteSink& out, int64_t outer, int64_t n, int64_t inner, int64_t nb,
                    const mxq_block_spec& q, hipStream_t st) {
  const int64_t groups = mxq::ceil_div(inner, 8);
  if (outer * nb * mxq::ceil_div(groups, 8) >= (int64_t(1) << 31))
    return mxq::invalid("block quantize: tensor too large (2^31 waves of 2048 elements)");
  auto go = [&](auto r_const) {
    constexpr int R = decltype(r_const)::value;
    const int64_t wpr = mxq::ceil_div(groups, 64 / R);
    const dim3 grid = mxq::grid_for(outer * nb * wpr * 64, 256);
    const mxq::DivU31 dnb = mxq::make_divu31((uint32_t)nb), dwpr = mxq::make_divu31((uint32_t)wpr);
    auto run = [&](auto kern) { kern<<<grid, 256, 0, st>>>(V, out, outer, n, inner, dnb, dwpr, q); };
    if (q.e == 4) run(k_pack_rne<T, 4, 3, R>);
    else if (q.e == 5) run(k_pack_rne<T, 5, 2, R>);
    else if (q.e == 3) run(k_pack_rne<T, 3, 2, R>);
    else if (q.m == 3) run(k_pack_rne<T, 2, 3, R>);
    else run(k_pack_rne<T, 2, 1, R>);
  };
  if (outer * nb * mxq::ceil_div(groups, 16) >= 2048) go(std::integral_constant<int, 4>{});
  else go(std::integral_constant<int, 8>{});
  return mxq::check_launch("mxq_block_quantize_packed");
}

// bs < 0: the transposed layout (outer 1, block 32, V read as M^T), k_quant_t (float32 outputs only).
template <typename T, int ELEM, int MODE, typename SINK>
int launch_quant(const T* V, const SINK& out, int64_t outer, int64_t n, int64_t inner, int64_t bs,
                 const mxq_block_spec& q, hipStream_t st) {
  if constexpr (SINK::kBytes == 4) {
    if (bs < 0) return launch_quant_t<T, ELEM, MODE>(V, out.P, out.X, n, inner, q, st);
  } else if (bs < 0) {
    return mxq::invalid("mxq_block_quantize_packed: no transposed layout");
  }
  mxq::KernelTimer timer("block_quantize", st);
  const int64_t nb = mxq::ceil_div(n, bs);
  // Codes that replace their inputs (P is V): no lane may read another's elements, so rows that a lane's columns do not
  // divide take fewer columns a lane instead of a last group moved back over its neighbour's.
  bool in_place = false;
  if constexpr (SINK::kBytes == 4) in_place = static_cast<const void*>(V) == static_cast<const void*>(out.P);
  // contiguous blocks: rows of whole blocks in any number (no row to find); others count their blocks in 31 bits
  if (inner == 1 && bs == 32 && outer * n >= 4 &&
      (n % 32 == 0 || (!in_place && outer * nb < (int64_t(1) << 31) && n < (int64_t(1) << 31)))) {
    const int64_t nblocks = outer * nb;
    auto go = [&](auto q_const) {
      constexpr int Q = decltype(q_const)::value;
      const dim3 grid = mxq::grid_for(mxq::ceil_div(nblocks, Q) * 8, 256);
      if (n % 32 == 0) k_quant_row<T, ELEM, MODE, Q, true><<<grid, 256, 0, st>>>(V, out, nblocks, outer, n, {}, q);
      else k_quant_row<T, ELEM, MODE, Q, false><<<grid, 256, 0, st>>>(V, out, nblocks, outer, n,
                                                                       mxq::make_divu31((uint32_t)nb), q);
    };
    // Q = 4 for the grids the conversions take, while it leaves the chip two waves a SIMD (16,384 rows of 2001
    // half-precision values: 35 us); a software grid is VALU work enough to hide the rest (16,384 x 2048
    // float32 through mxquant's: 53 us at Q = 4, 48 at Q = 1)
    if constexpr (MODE == MXQ_RNE && (ELEM == MXQ_ELEM_OCP || ELEM == MXQ_ELEM_MICROSOFT)) {
      if (nblocks >= 2048 * 8 * 4) {
        go(std::integral_constant<int, 4>{});
        return mxq::check_launch("mxq_block_quantize");
      }
    }
    go(std::integral_constant<int, 1>{});
    return mxq::check_launch("mxq_block_quantize");
  }
  if constexpr (SINK::kBytes == 1 && ELEM == MXQ_ELEM_OCP && MODE == MXQ_RNE) {
    // narrow rows that are no whole eights leave k_pack_rne's eight columns a lane partly empty and its last group to
    // overlapping accesses: 512 x 37 6.1 us, by k_quant_split 5.1; 131,072 x 12 10.6 and 9.9
    if (bs == 32 && q.via_e == 0 && out.e == q.e && out.m == q.m && mxq_ocp_hw::has_hw(q.e, q.m) &&
        q.max_norm == mxq_ocp_hw::fmt_max(q.e, q.m) && (inner % 8 == 0 || inner >= 64))
      return launch_pack_rne(V, out, outer, n, inner, nb, q, st);
  }
  if (bs == 32) {
    // Columns a lane (VEC) and lanes a block column (R, 32 / R rows each), by the full waves that four columns at R = 8
    // make.  Measured on inputs and outputs that leave the caches, float32 codes from float32 (bytes from bfloat16), us:
    //                           VEC 4, R 8    4, 32    2, 32    1, 32
    //   nearest even, by the conversions (the OCP grid; microxcaling's is alike)
    //     4096 x 512                  6.3      7.7     11.5     24.9      (bytes 7.9, 10.5, 15.9, 21.9)
    //     5632 x 333                  7.8     11.4     13.6     21.8      (8.6, 11.3, 14.8, 18.5)
    //     4096 x 100, 400 waves       4.8      5.1      5.1      6.6      (6.7, 6.5, 7.0, 7.0)
    //     512 x 37                    3.8      3.9      3.6      3.8      (5.8, 5.3, 5.2, 4.5)
    //   software grids (mxquant; bytes: the OCP grid, ties away), whose four rows a lane take longer
    //     4096 x 1536                13.2     21.3     32.3     74.8      (14.2, 24.0, 33.5, 52.5)
    //     4096 x 512                  7.9      7.8     11.5     25.0      (8.9, 11.3, 14.4, 20.0)
    //     1000 x 333                  6.7      4.9      4.9      6.0      (8.2, 6.3, 6.1, 6.5)
    //     512 x 37                    5.5      3.8      3.5      3.8      (6.9, 5.2, 4.7, 4.2)
    //   rows of eight columns and fewer, whose waves R = 8 leaves three quarters empty
    //     262,144 x 7                 8.6      6.9      8.6     12.3      (14.4, 10.2, 12.1, 13.9)
    // So R = 8 from 400 full waves with the conversions, from 2048 (bytes 1024) without, R = 32 for narrow rows, and
    // single columns or pairs where four make few.  mxquant's bytes, all encoding, keep R = 32 (131,072 x 12: 66 us, 84 at
    // R = 8).  Code bytes take eight columns (8-byte stores: a wave's eight lanes write 64 contiguous bytes of a row) once
    // that fills the chip: 8192 x 8192 to bytes, ties away, 66 us, 75 with four.
    constexpr bool BYTES = SINK::kBytes == 1;
    constexpr bool HW = MODE == MXQ_RNE && (ELEM == MXQ_ELEM_OCP || ELEM == MXQ_ELEM_MICROSOFT);
    auto go = [&](auto vec_const, auto r_const, auto whole_const) {
      constexpr int VEC = decltype(vec_const)::value, R = decltype(r_const)::value;
      const int64_t wpr = mxq::ceil_div(mxq::ceil_div(inner, VEC), 64 / R);
      k_quant_split<T, ELEM, MODE, VEC, R, decltype(whole_const)::value, SINK>
          <<<mxq::grid_for(outer * nb * wpr * 64, 256), 256, 0, st>>>(V, out, outer, n, inner, mxq::make_divu31((uint32_t)nb),
                                                                      mxq::make_divu31((uint32_t)wpr), q);
    };
    using One = std::integral_constant<int, 1>;
    using Two = std::integral_constant<int, 2>;
    using Four = std::integral_constant<int, 4>;
    using Eight = std::integral_constant<int, 8>;
    using Half = std::integral_constant<int, 32>;          // (half a wave to a block column)
    // the kernel indexes waves in 32 bits
    const bool narrow = inner < 4 || (in_place && inner % 4 != 0);
    const int64_t widest = !narrow ? (BYTES && inner >= 8 ? 8 : 4) : (inner % 2 == 0 ? 2 : 1);
    if (outer * nb * mxq::ceil_div(mxq::ceil_div(inner, widest), 2) >= (int64_t(1) << 31))
      return mxq::invalid("block quantize: tensor too large (2^31 waves of 2048 elements)");
    const int64_t full = outer * nb * mxq::ceil_div(inner, 4) / 8;
    constexpr bool ENCODE = BYTES && ELEM == MXQ_ELEM_QTORCH;
    if (narrow) {
      const bool many = outer * nb * mxq::ceil_div(inner, 4) >= 8 * 1024;
      if (inner % 2 == 0) many ? go(Two{}, Eight{}, std::true_type{}) : go(Two{}, Half{}, std::true_type{});
      else many ? go(One{}, Eight{}, std::true_type{}) : go(One{}, Half{}, std::true_type{});
    } else if (full < (ENCODE ? 64 : inner <= 8 ? 128 : HW && BYTES ? 400 : 200)) {
      if constexpr (BYTES || ELEM == MXQ_ELEM_MICROSOFT) go(One{}, Half{}, std::true_type{});
      else go(Two{}, Half{}, std::false_type{});
    } else if (ENCODE || inner <= 8 || full < (HW ? 400 : BYTES ? 1024 : 2048)) {
      go(Four{}, Half{}, std::false_type{});
    } else if constexpr (!ENCODE) {
      if (BYTES && inner >= 64 && outer * nb * mxq::ceil_div(inner, 8) / 8 >= 8 * 1024) {
        if constexpr (BYTES) inner % 8 == 0 ? go(Eight{}, Eight{}, std::true_type{}) : go(Eight{}, Eight{}, std::false_type{});
      } else if (inner % 4 == 0) go(Four{}, Eight{}, std::true_type{});
      else go(Four{}, Eight{}, std::false_type{});
    }
    return mxq::check_launch("mxq_block_quantize");
  }
  const int svec = inner % 4 == 0 ? 4 : (inner % 2 == 0 ? 2 : 1);
  const dim3 grid = mxq::grid_for(outer * nb * (inner / svec), 256);
  if (svec == 4) k_quant_strided<T, ELEM, MODE, 4, SINK><<<grid, 256, 0, st>>>(V, out, outer, n, inner, bs, nb, q);
  else if (svec == 2) k_quant_strided<T, ELEM, MODE, 2, SINK><<<grid, 256, 0, st>>>(V, out, outer, n, inner, bs, nb, q);
  else k_quant_strided<T, ELEM, MODE, 1, SINK><<<grid, 256, 0, st>>>(V, out, outer, n, inner, bs, nb, q);
  return mxq::check_launch("mxq_block_quantize");
}

template <typename T, int ELEM, typename SINK>
int launch_mode(const T* V, const SINK& out, int64_t outer, int64_t n, int64_t inner, int64_t bs,
                const mxq_block_spec& q, hipStream_t st) {
  switch (q.rounding) {
    case MXQ_RNE: return launch_quant<T, ELEM, MXQ_RNE>(V, out, outer, n, inner, bs, q, st);
    case MXQ_TIES_AWAY: return launch_quant<T, ELEM, MXQ_TIES_AWAY>(V, out, outer, n, inner, bs, q, st);
    default: return launch_quant<T, ELEM, MXQ_TRUNC>(V, out, outer, n, inner, bs, q, st);
  }
}

// Float32 outputs: every element rule.  Bytes: the rules whose grids are the OCP element formats' (mxgemmini's
// ocp grid, block.ocp's microxcaling step) and mxquant's qtorch grid (whose smallest values some formats lack:
// those set the error word).
template <typename T, typename SINK>
int dispatch_elem(const T* V, const SINK& out, int64_t outer, int64_t n, int64_t inner, int64_t bs,
                  const mxq_block_spec& q, hipStream_t st) {
  switch (q.elem) {
    case MXQ_ELEM_QTORCH: return launch_quant<T, MXQ_ELEM_QTORCH, -1>(V, out, outer, n, inner, bs, q, st);
    case MXQ_ELEM_OCP: return launch_mode<T, MXQ_ELEM_OCP>(V, out, outer, n, inner, bs, q, st);
    case MXQ_ELEM_MICROSOFT: return launch_mode<T, MXQ_ELEM_MICROSOFT>(V, out, outer, n, inner, bs, q, st);
    default: break;
  }
  if constexpr (SINK::kBytes == 4) {
    if (q.elem == MXQ_ELEM_IEEE) return launch_quant<T, MXQ_ELEM_IEEE, -1>(V, out, outer, n, inner, bs, q, st);
    return launch_quant<T, MXQ_ELEM_NONE, -1>(V, out, outer, n, inner, bs, q, st);
  } else {
    return mxq::invalid("mxq_block_quantize_packed: the element rule has no byte format");
  }
}

}  // namespace mxq_quant
