// out = P * expand(X) over the (outer, n, inner) view with blocks of bs along n, from float32 codes and scales
// (FloatSource) or from their bytes (ByteSource).
//
//   k_dequant_cols   inner >= 4: a thread takes four adjacent columns (the last group ends on the last column) of
//                    ROWS rows of one block, all of them under one load of four scales
//   k_dequant_row    inner == 1: a thread takes four adjacent elements of a row, which lie in two blocks at most
//   k_dequant_few    rows of 2 and 3 columns, rows or blocks under 4 elements: an access or two columns a thread
//   k_dequant_any    sizes whose indexes pass 31 bits
//
// Memory bounds them.  Four elements are one access wherever they begin: gfx950 takes 4 to 16 bytes at any
// element's address, so rows of any length run as whole fours do.
// Measured: 8192 x 5632 bytes of E3M2 54 -> 36 us (232 MB, 6.4 TB/s; a thread walked a block column a byte at a
// time); float32 codes, rows of 2001, 2331 of them 14.6 -> 9.5 us, calls on 4096 x 2049 17.8 -> 12.0 us; 8192 x 8192
// 87 us before and now (6.2 TB/s).
#pragma once
#include "quantize_impl.h"

namespace mxq_quant {

struct FloatSource {
  static constexpr int kRows = 1;
  const float* P;
  const float* X;
  template <int VEC>
  __device__ __forceinline__ void codes(int64_t at, float (&v)[VEC]) const { load_vec<float, VEC>(P + at, v); }
  template <int VEC>
  __device__ __forceinline__ void scales(int64_t at, float (&x)[VEC]) const { load_vec<float, VEC>(X + at, x); }
};

// Code bytes of the element format (E, M) and E8M0 bytes.  Codes decode through gfx950's conversions, exactly, but
// for Inf and NaN codes, which mx_decode gives their patterns; FP6 as the FP8 of the same mantissa width (the sign
// moved to bit 7), scaled by the difference of the exponent offsets.
template <int E, int M>
struct ByteSource {
  static constexpr int kRows = 4;
  const uint8_t* P;
  const uint8_t* X;
  __device__ static uint32_t special(uint32_t w) {            // nonzero: a byte of w is an Inf or NaN code
    if constexpr (E == 4) return ((w & 0x7F7F7F7Fu) + 0x01010101u) & 0x80808080u;
    else if constexpr (E == 5) return ((w & 0x7F7F7F7Fu) + 0x04040404u) & 0x80808080u;
    else return 0u;
  }
  template <int VEC>
  __device__ __forceinline__ void codes(int64_t at, float (&v)[VEC]) const {
    uint32_t w = 0u;
    __builtin_memcpy(&w, P + at, VEC);
    if (VEC < 4 || special(w)) {
#pragma unroll
      for (int j = 0; j < VEC; ++j) v[j] = mx_decode((w >> (8 * j)) & 0xFFu, E, M);
    } else if constexpr (VEC == 4) {
      mxq_ocp_hw::f2v a, b;
      if constexpr (E == 2 && M == 1) {
        w &= 0x0F0F0F0Fu;
        w |= w >> 4;                                          // bytes 0 and 2: two codes each
        a = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 0);
        b = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 2);
      } else {
        constexpr bool FP6 = E + M == 5;
        if constexpr (FP6) w = (w & 0x1F1F1F1Fu) | ((w & 0x20202020u) << 2);
        if constexpr (M == 3) {
          a = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(w, 1.0f, false);
          b = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(w, 1.0f, true);
        } else {
          a = __builtin_amdgcn_cvt_scalef32_pk_f32_bf8(w, 1.0f, false);
          b = __builtin_amdgcn_cvt_scalef32_pk_f32_bf8(w, 1.0f, true);
        }
        if constexpr (FP6) {
          const float up = M == 3 ? 64.0f : 4096.0f;
          a.x *= up; a.y *= up; b.x *= up; b.y *= up;
        }
      }
      v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y;
    }
  }
  template <int VEC>
  __device__ __forceinline__ void scales(int64_t at, float (&x)[VEC]) const {
    uint32_t w = 0u;
    __builtin_memcpy(&w, X + at, VEC);
#pragma unroll
    for (int j = 0; j < VEC; ++j) x[j] = e8m0_decode((w >> (8 * j)) & 0xFFu);
  }
};

// `chunks`: ROWS-row pieces of n; bs is a multiple of ROWS, so that a piece lies in one block.
template <int ROWS, typename SRC>
__global__ void __launch_bounds__(256) k_dequant_cols(const SRC src, float* __restrict__ out, uint32_t count,
                                                      int64_t n, int64_t inner, int64_t nb, mxq::DivU31 groups,
                                                      mxq::DivU31 chunks, mxq::DivU31 bs) {
  const uint32_t t = blockIdx.x * 256u + threadIdx.x;
  if (t >= count) return;
  const uint32_t rc = mxq::divu31(t, groups), g = t - rc * groups.d;
  const uint32_t o = mxq::divu31(rc, chunks), k0 = (rc - o * chunks.d) * ROWS;
  const int64_t col = 4 * (int64_t)g < inner - 4 ? 4 * (int64_t)g : inner - 4;
  const int64_t at = (o * n + k0) * inner + col;
  float x[4];
  src.template scales<4>((o * nb + mxq::divu31(k0, bs)) * inner + col, x);
  auto scaled = [&](int64_t where, float (&v)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = v[j] * x[j];
    store_vec_nt<4>(out + where, v);
  };
  if constexpr (ROWS == 1) {
    float v[4];
    src.template codes<4>(at, v);
    scaled(at, v);
  } else if (n - k0 >= ROWS) {
    float v[ROWS][4];
#pragma unroll
    for (int i = 0; i < ROWS; ++i) src.template codes<4>(at + i * inner, v[i]);
#pragma unroll
    for (int i = 0; i < ROWS; ++i) scaled(at + i * inner, v[i]);
  } else {
    for (int64_t row = at; row < ((int64_t)o + 1) * n * inner; row += inner) {
      float v[4];
      src.template codes<4>(row, v);
      scaled(row, v);
    }
  }
}

// Rows of n elements, blocks of bs >= 4.
template <typename SRC>
__global__ void __launch_bounds__(256) k_dequant_row(const SRC src, float* __restrict__ out, uint32_t count, int64_t n,
                                                     int64_t nb, mxq::DivU31 groups, mxq::DivU31 bs) {
  const uint32_t t = blockIdx.x * 256u + threadIdx.x;
  if (t >= count) return;
  const uint32_t r = mxq::divu31(t, groups), g = t - r * groups.d;
  const uint32_t k = 4 * g < (uint32_t)n - 4u ? 4 * g : (uint32_t)n - 4u;
  const uint32_t b = mxq::divu31(k, bs), next = (b + 1) * bs.d;
  float x0[1], x1[1], v[4];
  src.template codes<4>(r * n + k, v);
  src.template scales<1>(r * nb + b, x0);
  x1[0] = x0[0];
  if (k + 3 >= next) src.template scales<1>(r * nb + b + 1, x1);
#pragma unroll
  for (uint32_t j = 0; j < 4; ++j) v[j] = v[j] * (k + j >= next ? x1[0] : x0[0]);
  store_vec_nt<4>(out + r * n + k, v);
}

// VEC adjacent columns a thread, any shape whose element count fits 31 bits (262,144 x 2 float32 in blocks of 32: 2.9 us,
// 3.7 with k_dequant_any's 64-bit divisions; 4096 x 512 along its rows in blocks of 3: 5.8 and 7.1).
template <int VEC, typename SRC>
__global__ void __launch_bounds__(256) k_dequant_few(const SRC src, float* __restrict__ out, uint32_t count,
                                                     mxq::DivU31 groups, mxq::DivU31 n, mxq::DivU31 bs, uint32_t nb) {
  const uint32_t t = blockIdx.x * 256u + threadIdx.x;
  if (t >= count) return;
  const uint32_t row = mxq::divu31(t, groups), g = t - row * groups.d;
  const uint32_t o = mxq::divu31(row, n), k = row - o * n.d;
  float v[VEC], x[VEC];
  src.template codes<VEC>((int64_t)t * VEC, v);
  src.template scales<VEC>(((int64_t)(o * nb + mxq::divu31(k, bs)) * groups.d + g) * VEC, x);
#pragma unroll
  for (int j = 0; j < VEC; ++j) v[j] = v[j] * x[j];
  store_vec_nt<VEC>(out + (int64_t)t * VEC, v);
}

template <int VEC, typename SRC>
__global__ void __launch_bounds__(256) k_dequant_any(const SRC src, float* __restrict__ out, int64_t count, int64_t n,
                                                     int64_t inner, int64_t bs, int64_t nb) {
  for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < count; t += (int64_t)gridDim.x * 256) {
    const int64_t at = t * VEC, row = at / inner, o = row / n, k = row - o * n;
    float v[VEC], x[VEC];
    src.template codes<VEC>(at, v);
    src.template scales<VEC>((o * nb + k / bs) * inner + (at - row * inner), x);
#pragma unroll
    for (int j = 0; j < VEC; ++j) v[j] = v[j] * x[j];
    store_vec_nt<VEC>(out + at, v);
  }
}

// ROWS > 1 (the source's kRows) once its threads are at least kDequantFill, 8 waves a SIMD.
constexpr int64_t kDequantFill = 8 * 1024 * 64;

// `in_place`: out is where the float32 codes lie, so no thread may read another's (a last group moved back over its
// neighbour's columns does): rows that are no whole fours go to the kernels whose groups divide them.
template <typename SRC>
void launch_dequant(const SRC& src, float* out, int64_t outer, int64_t n, int64_t inner, int64_t bs, hipStream_t st,
                    bool in_place = false) {
  const int64_t nb = mxq::ceil_div(n, bs), lim = (int64_t)1 << 31, all = outer * n * inner;
  if (inner >= 4 && (!in_place || inner % 4 == 0) && outer * n * mxq::ceil_div(inner, 4) < lim && bs < lim) {
    const int64_t groups = mxq::ceil_div(inner, 4);
    auto go = [&](auto rows_const) {
      constexpr int ROWS = decltype(rows_const)::value;
      const int64_t chunks = mxq::ceil_div(n, ROWS), count = outer * chunks * groups;
      k_dequant_cols<ROWS><<<mxq::grid_for(count, 256), 256, 0, st>>>(
          src, out, (uint32_t)count, n, inner, nb, mxq::make_divu31((uint32_t)groups),
          mxq::make_divu31((uint32_t)chunks), mxq::make_divu31((uint32_t)bs));
    };
    if (bs % SRC::kRows == 0 && outer * mxq::ceil_div(n, SRC::kRows) * groups >= kDequantFill)
      go(std::integral_constant<int, SRC::kRows>{});
    else
      go(std::integral_constant<int, 1>{});
  } else if (inner == 1 && n >= 4 && (!in_place || n % 4 == 0) && n < lim && bs >= 4 && bs < lim && outer * mxq::ceil_div(n, 4) < lim) {
    const int64_t groups = mxq::ceil_div(n, 4), count = outer * groups;
    k_dequant_row<<<mxq::grid_for(count, 256), 256, 0, st>>>(src, out, (uint32_t)count, n, nb,
                                                            mxq::make_divu31((uint32_t)groups),
                                                            mxq::make_divu31((uint32_t)bs));
  } else if (all < lim && bs < lim) {
    auto go = [&](auto vec_const) {
      constexpr int VEC = decltype(vec_const)::value;
      k_dequant_few<VEC><<<mxq::grid_for(all / VEC, 256), 256, 0, st>>>(
          src, out, (uint32_t)(all / VEC), mxq::make_divu31((uint32_t)(inner / VEC)), mxq::make_divu31((uint32_t)n),
          mxq::make_divu31((uint32_t)bs), (uint32_t)nb);
    };
    if (inner % 2 == 0) go(std::integral_constant<int, 2>{});
    else go(std::integral_constant<int, 1>{});
  } else {
    auto go = [&](auto vec_const) {
      constexpr int VEC = decltype(vec_const)::value;
      const int64_t blocks = mxq::ceil_div(all / VEC, 256);
      k_dequant_any<VEC><<<dim3((unsigned)(blocks < (1 << 22) ? blocks : (1 << 22))), 256, 0, st>>>(
          src, out, all / VEC, n, inner, bs, nb);
    };
    if (inner % 4 == 0) go(std::integral_constant<int, 4>{});
    else go(std::integral_constant<int, 1>{});
  }
}

}  // namespace mxq_quant
