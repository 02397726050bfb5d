// rad_mlp.h -- what the emulator's kernels share: BF16 operands, GELU, MFMA
// (rad_mlp.hip, rad_train.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

union V8 {
  bf16x8 v;
  uint16_t s[8];
  uint4 q;
};

__device__ __forceinline__ uint16_t f2bf(float x) {  // round to nearest even
  uint32_t u = __float_as_uint(x);
  if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)(u >> 16);  // inf / nan
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// GELU (erf form) and its derivative.  erf by Abramowitz & Stegun 7.1.26:
// erf(x) = 1 - (a1 t + ... + a5 t^5) exp(-x^2), t = 1 / (1 + p x) for x >= 0,
// absolute error <= 1.5e-7 -- below the bf16 rounding that follows every
// activation by four orders of magnitude, and a third of the cost of the
// correctly rounded erff.  The derivative shares exp(-z^2/2).
__device__ __forceinline__ float erf_as(float x, float& e) {
  const float ax = fabsf(x);
  const float t = __builtin_amdgcn_rcpf(fmaf(0.3275911f, ax, 1.0f));
  const float poly =
      t * fmaf(t, fmaf(t, fmaf(t, fmaf(t, 1.061405429f, -1.453152027f), 1.421413741f),
                       -0.284496736f),
               0.254829592f);
  e = __expf(-ax * ax);
  const float r = 1.0f - poly * e;
  return copysignf(r, x);
}
__device__ __forceinline__ float gelu(float z) {
  float e;
  return 0.5f * z * (1.0f + erf_as(z * 0.70710678118654752f, e));
}
__device__ __forceinline__ float gelu_d(float z) {
  float e;  // exp(-z^2 / 2)
  const float cdf = 0.5f * (1.0f + erf_as(z * 0.70710678118654752f, e));
  return cdf + z * 0.39894228040143268f * e;
}

__device__ __forceinline__ f32x4 mfma(const V8& a, const V8& b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, c, 0, 0, 0);
}

// this wave's weight fragments of one layer (output features [32w, 32w+32),
// K/32 x 2 x 16 bytes per lane), requested ahead of the layer that uses them
template <int K>
__device__ __forceinline__ void em_load(const uint16_t* W, V8 (&wa)[K / 32][2]) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int q = lane >> 4, c = lane & 15;
  const uint16_t* wr = W + (long)(wv * 32 + c) * K + q * 8;
#pragma unroll
  for (int ks = 0; ks < K / 32; ++ks)
#pragma unroll
    for (int i = 0; i < 2; ++i) wa[ks][i].q = *(const uint4*)(wr + (long)i * 16 * K + ks * 32);
}

}  // namespace
