// Frequency encoding and BF16 conversion shared by the MLP kernels.
#pragma once

#include "mlp_kernels.h"

namespace pt {
namespace mlp {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

// float -> bf16 bits, round to nearest even (v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint16_t f2bf(float x) {
  return __builtin_bit_cast(uint16_t, __bf16(x));
}
__device__ __forceinline__ uint32_t f2bf2(float lo, float hi) {
  const bf16x2_t v = {__bf16(lo), __bf16(hi)};
  return __builtin_bit_cast(uint32_t, v);
}

// Column order of the encoded input inside the kernels: the 24 sines and
// cosines of feature d at 24 d (three aligned 16-byte stores instead of 24
// two-byte ones), the raw features at 216 + d, zero from 225 on. Parameters
// and gradients outside have the raw features first (column d), then feature
// d's pairs at 9 + 24 d.
constexpr uint32_t kEncPairs = kEncoded - kFeatures; // 216
__host__ __device__ inline uint32_t outer_column(uint32_t k) {
  return k < kEncPairs ? k + kFeatures : k < kEncoded ? k - kEncPairs : k;
}

// Feature d with value x in one encoded row (16-byte aligned): the raw value
// and, per frequency k, sin and cos(pi 2^k x). Frequencies 0, 4 and 8 come
// from sincospi; the three after each are doubled (sin 2a = 2 sin a cos a,
// cos 2a = 1 - 2 sin^2 a), which adds at most ~1e-6 absolute error, below the
// bf16 rounding of the result.
__device__ __forceinline__ void encode_feature(float x, uint32_t d, uint16_t *row) {
  row[kEncPairs + d] = f2bf(x);
  uint4 *o = reinterpret_cast<uint4 *>(row + 2 * kFrequencies * d);
#pragma unroll
  for (uint32_t g = 0; g < kFrequencies / 4; ++g) {
    uint32_t v[4];
    float s = 0.f, c = 1.f;
    sincospif(ldexpf(x, int(4 * g)), &s, &c);
    v[0] = f2bf2(s, c);
#pragma unroll
    for (int k = 1; k < 4; ++k) {
      const float s2 = 2.f * s * c;
      c = fmaf(-2.f * s, s, 1.f);
      s = s2;
      v[k] = f2bf2(s, c);
    }
    o[g] = make_uint4(v[0], v[1], v[2], v[3]);
  }
}

} // namespace mlp
} // namespace pt
