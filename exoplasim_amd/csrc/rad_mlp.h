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

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// round to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint32_t f2bf2(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, bf16x2));
}
__device__ __forceinline__ uint16_t f2bf(float x) {
  return __builtin_bit_cast(uint16_t, (__bf16)x);
}

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

// Fragment order of a weight matrix W[N][K] (N a multiple of 16, K of 32): the
// 16 x 32 tiles (nt, ks) one after the other, ks fastest, each as the 64 lanes
// of v_mfma_f32_16x16x32_bf16 hold it, lane 16 q + c the 8 values k = 32 ks + 8 q
// .. + 7 of row n = 16 nt + c.  A wave's load of a tile is then 1 KB in a row;
// from row-major weights it is 64 bytes of each of 16 rows, and with every CU
// reading the same weights at once those loads, not the arithmetic, bounded
// the kernels (inference of 8192 columns 15.9 -> 10.0 us, of 65536 115 -> 65).
__device__ __forceinline__ void frag_nk(int e, int K, int& n, int& k) {
  const int j = e & 7, lane = (e >> 3) & 63, t = e >> 9, ks = t % (K / 32), nt = t / (K / 32);
  n = nt * 16 + (lane & 15);
  k = ks * 32 + (lane >> 4) * 8 + j;
}

// the K / 32 fragments of row tile nt, in fragment order or row-major
template <int K, bool PACKED = true>
__device__ __forceinline__ void load_tile(const uint16_t* W, int nt, V8 (&w)[K / 32]) {
  const int lane = threadIdx.x & 63, q = lane >> 4, c = lane & 15;
#pragma unroll
  for (int ks = 0; ks < K / 32; ++ks)
    w[ks].q = PACKED ? *(const uint4*)(W + (nt * (K / 32) + ks) * 512 + lane * 8)
                     : *(const uint4*)(W + (nt * 16 + c) * K + ks * 32 + q * 8);
}

// a wave's 32 output features x MT rows of one layer, transposed: acc[i][j]
// holds features 16 i + 4 q .. + 3 (of the wave's 32) of row 16 j + c; `in` are
// the rows in LDS, LDI values apart
template <int K, int LDI, int MT>
__device__ __forceinline__ void layer(const uint16_t* in, const V8 (&w)[2][K / 32],
                                      f32x4 (&acc)[2][MT / 16]) {
  const int lane = threadIdx.x & 63, q = lane >> 4, c = lane & 15;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < MT / 16; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int ks = 0; ks < K / 32; ++ks) {
    V8 h[MT / 16];
#pragma unroll
    for (int j = 0; j < MT / 16; ++j)
      h[j].q = *(const uint4*)(in + (j * 16 + c) * LDI + ks * 32 + q * 8);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < MT / 16; ++j) acc[i][j] = mfma(w[i][ks], h[j], acc[i][j]);
  }
}

}  // namespace
