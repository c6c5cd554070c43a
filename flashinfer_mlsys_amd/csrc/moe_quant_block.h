// The arithmetic of one 1 x 128 activation block's FP8 quantisation (reference
// solution/triton/dsl-temp1.py:479-484), shared by the quantiser kernel and the
// router GEMM's fused path so that both write the same bytes:
//   scale = max(amax, 1e-12) / 448
//   code  = e4m3(clamp(x / scale, -448, 448)), correctly rounded fp32 quotient, round
//           to nearest even (v_cvt_pk_fp8_f32).
#pragma once

#include <type_traits>

#include "moe_common.h"

namespace moe {

__device__ __forceinline__ float qblock_scale(float amax) { return fmaxf(amax, 1e-12f) / 448.0f; }

// x / s, correctly rounded, for a bf16 value x and its block's scale s: q = x y with y
// within 3 ulps of 1 / s, then one residual step, q + y (x - s q) in fused operations (the
// correction step of Markstein's division for machines with a fused multiply-add, 1990).
// That is the correctly rounded quotient for every pair of a bf16 maximum and a bf16
// value (their 128 x 128 significands, checked one by one: the steps scale exactly with
// the exponents, and a quotient that does not round to the code 0 has |q| >= 2^-10 and
// s >= 2e-15, far above the smallest normal number): 3 instructions a value against the
// dozen of a division. An infinite scale (s and y set to 0) gives 0 for finite values and
// NaN for infinite ones, as the division; the quotient's sign is the value's, also where
// it is zero.
struct QDiv {
  float s, y;
};
__device__ __forceinline__ QDiv qblock_div(float scale) {
  const bool fin = scale < __builtin_inff();
  return QDiv{fin ? scale : 0.f, fin ? __builtin_amdgcn_rcpf(scale) : 0.f};
}
__device__ __forceinline__ float qblock_quot(float x, const QDiv& d) {
  const float q = x * d.y;
  return copysignf(fmaf(fmaf(-d.s, q, x), d.y, q), x);
}

// Four values -> four e4m3 codes, first value in the low byte.
__device__ __forceinline__ uint32_t qblock_pack4(float a, float b, float c, float d, const QDiv& s) {
  const float qa = fminf(fmaxf(qblock_quot(a, s), -448.f), 448.f), qb = fminf(fmaxf(qblock_quot(b, s), -448.f), 448.f);
  const float qc = fminf(fmaxf(qblock_quot(c, s), -448.f), 448.f), qd = fminf(fmaxf(qblock_quot(d, s), -448.f), 448.f);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(qa, qb, 0, false) & 0xffffu;
  const uint32_t hi = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(qc, qd, 0, false) & 0xffffu;
  return lo | (hi << 16);
}

// The scale of a block with a finite maximum, bit for bit amax / 448 (the same residual step).
__device__ __forceinline__ float qblock_scale_finite(float amax) {
  const float m = fmaxf(amax, 1e-12f), q = m * (1.0f / 448.0f);
  return fmaf(fmaf(-448.0f, q, m), 1.0f / 448.0f, q);
}

// The codes of eight finite values (bf16 pairs w, as floats v): no clamp (the largest
// quotient is 448 (1 + 2^-23), which rounds to 448), the signs of zeros from the values.
__device__ __forceinline__ void qblock_pack8_finite(const uint32_t (&w)[4], const float (&v)[8], const QDiv& d,
                                                    uint32_t (&o)[2]) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    float q[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float x = v[4 * h + i], q0 = x * d.y;
      q[i] = fmaf(fmaf(-d.s, q0, x), d.y, q0);
    }
    int c = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], 0, false);
    c = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], c, true);
    // the four values' high bytes: bytes 1 and 3 of either word
    o[h] = (uint32_t)c | (__builtin_amdgcn_perm(w[2 * h + 1], w[2 * h], 0x07050301u) & 0x80808080u);
  }
}

// Maximum of a 16-lane row's magnitudes as bf16 bits (8 values a lane, two per word), in
// every lane: above 0x7f80 if any is NaN. (lane ^ 1, lane ^ 2, half row and row mirrored.)
__device__ __forceinline__ uint32_t row16_max_bf16(const uint32_t (&w)[4]) {
  typedef unsigned short v2us __attribute__((ext_vector_type(2)));
  v2us m = __builtin_bit_cast(v2us, w[0] & 0x7fff7fffu);
#pragma unroll
  for (int i = 1; i < 4; ++i) {
    const uint32_t u = w[i] & 0x7fff7fffu;
    m = __builtin_elementwise_max(m, __builtin_bit_cast(v2us, u));
  }
  const uint32_t b = __builtin_bit_cast(uint32_t, m);
  uint32_t r = max(b & 0xffffu, b >> 16);
  auto step = [&](auto ctrl) {
    r = max(r, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)r, decltype(ctrl)::value, 0xf, 0xf, true));
  };
  step(std::integral_constant<int, 0xB1>{});
  step(std::integral_constant<int, 0x4E>{});
  step(std::integral_constant<int, 0x141>{});
  step(std::integral_constant<int, 0x140>{});
  return r;
}

// Eight bf16 (two per 32-bit word, first in the low half) -> fp32.
__device__ __forceinline__ void bf16x8_to_f32(const uint32_t (&w)[4], float (&v)[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = __uint_as_float(w[i] << 16);
    v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
  }
}

}  // namespace moe
