// rad_train.hip -- the emulator network's training passes (43 -> 256 -> 256 ->
// 256 -> 21, GELU; include/exo_rad.h): forward with the activations the
// backward pass reads, and the gradients of all weights and biases.
//
//   k_cast_net   FP32 master weights -> padded bf16, all layers (forward: W,
//                backward: its transpose), one launch
//   k_train_fwd  the four layers of MT batch rows per block, activations in
//                LDS, z (FP32), h (bf16) and y written on the way
//   k_train_dx   the chain dz4 -> dz3 -> dz2 -> dz1 of MT rows per block, dz
//                (bf16) for the weight gradients and the block's bias sums
//   k_train_dw   the four dW = dZ^T X, split over the batch, one launch
//   k_train_sum  sums of the partial dW and bias gradients into the results
//
// At a batch of thousands of rows every one of these is bound by latency (a
// chain of three dependent layers, a few microseconds of matrix work), and a
// training step by its launches, so a pass is as few of them as its
// dependences allow: 2 and 4 launches and one workspace, where a kernel per
// layer and operand took 9 and 25 launches with the padded copies and fills
// between them.  (4096 rows, forward and backward pass with loss: 658 us per
// step with a kernel per layer, 340-360 us with these; kernel time 287 -> 45
// us.)  Every product and sum runs in the order of the per-layer kernels
// (rad_mlp.hip); only the bias sums are regrouped.
#include "../../include/exo_rad.h"
#include "rad_mlp.h"

namespace {

constexpr int TNIN = 43, TKIN = 64, TNH = 256, TNOUT = 21, TNOUTP = 32;
constexpr int TLD = TNH + 8, TLDX = TKIN + 8, TLDY = TNOUTP + 8;  // padded LDS rows (bf16)
constexpr int TNT = 512;                                          // 8 waves, 32 features each
// padded weights of the layers one after the other, and the bias sums of a
// block (layers 1..3, then 4)
constexpr int TW1 = 0, TW2 = TNH * TKIN, TW3 = TW2 + TNH * TNH, TW4 = TW3 + TNH * TNH;
constexpr int TWALL = TW4 + TNOUTP * TNH;
constexpr int TBALL = 3 * TNH + TNOUTP;

struct TrainW {
  const float* w[4];
};

// padded bf16 weights of layer l in fragment order, the layers one after the
// other: W[N][K], with TR its transpose Wt[K][N]
template <bool TR>
__global__ __launch_bounds__(256) void k_cast_net(TrainW p, uint16_t* out) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= TWALL) return;
  const int l = i < TW2 ? 0 : i < TW3 ? 1 : i < TW4 ? 2 : 3;
  const int e = i - (l == 0 ? TW1 : l == 1 ? TW2 : l == 2 ? TW3 : TW4);
  const int N = l == 3 ? TNOUTP : TNH, K = l == 0 ? TKIN : TNH;
  const int nout = l == 3 ? TNOUT : TNH, nin = l == 0 ? TNIN : TNH;
  int n, k;
  if (TR)
    frag_nk(e, N, k, n);
  else
    frag_nk(e, K, n, k);
  out[i] = (n < nout && k < nin) ? f2bf(p.w[l][n * nin + k]) : (uint16_t)0;
}

// the wave's two row tiles of one layer
template <int K>
__device__ __forceinline__ void load_pair(const uint16_t* W, V8 (&w)[2][K / 32]) {
  const int wv = threadIdx.x >> 6;
  load_tile<K>(W, 2 * wv, w[0]);
  load_tile<K>(W, 2 * wv + 1, w[1]);
}

// sum over the 16 lanes of a row, in every lane (DPP row rotations)
__device__ __forceinline__ float row16_sum(float x) {
  x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x128, 0xF, 0xF, false));
  x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x124, 0xF, 0xF, false));
  x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x122, 0xF, 0xF, false));
  x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x121, 0xF, 0xF, false));
  return x;
}

__device__ __forceinline__ uint2 pack4(const float (&v)[4]) {
  return uint2{f2bf2(v[0], v[1]), f2bf2(v[2], v[3])};
}

// the block's MT rows of 256 bf16 values, LDS -> global, whole lines
template <int MT>
__device__ __forceinline__ void rows_out(const uint16_t* s, uint16_t* g, int row0, int M) {
#pragma unroll
  for (int it = 0; it < MT / 16; ++it) {
    const int e = threadIdx.x + TNT * it, m = e >> 5, k = (e & 31) * 8;
    if (row0 + m < M) *(uint4*)(g + (long)(row0 + m) * TNH + k) = *(const uint4*)(s + m * TLD + k);
  }
}

struct TrainFwd {
  const float* x;      // [M][43]
  const uint16_t* wb;  // k_cast_net<false>
  const float* b[4];
  uint16_t* x0;        // [M][64]
  float* z[3];
  uint16_t* h[3];
  float* y;            // [M][21]
};

template <int MT>
__global__ __launch_bounds__(TNT, 2) void k_train_fwd(TrainFwd a, int M) {
  __shared__ __align__(16) uint16_t sx[MT * TLDX];
  __shared__ __align__(16) uint16_t sh[2][MT * TLD];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, q = lane >> 4, c = lane & 15;
  const int row0 = blockIdx.x * MT;
  // the inputs first, without a branch, so that the wait for them does not
  // include the weights; the weights of the layers ahead are on their way while
  // one is computed
  float xv[MT / 16][2];
#pragma unroll
  for (int it = 0; it < MT / 16; ++it) {
    const int e = tid + TNT * it, m = e >> 5, k = (e & 31) * 2;
    const float* xr = a.x + (long)min(row0 + m, M - 1) * TNIN;
    xv[it][0] = xr[min(k, TNIN - 1)];
    xv[it][1] = xr[min(k + 1, TNIN - 1)];
  }
  __builtin_amdgcn_sched_barrier(0);
  V8 w1[2][TKIN / 32], w2[2][TNH / 32], w3[2][TNH / 32], w4[TNH / 32];
  load_pair<TKIN>(a.wb + TW1, w1);
  load_pair<TNH>(a.wb + TW2, w2);
  float bias[3][2][4];
#pragma unroll
  for (int l = 0; l < 3; ++l)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) bias[l][i][r] = a.b[l][wv * 32 + i * 16 + 4 * q + r];
#pragma unroll
  for (int it = 0; it < MT / 16; ++it) {
    const int e = tid + TNT * it, m = e >> 5, k = (e & 31) * 2;
    const long row = row0 + m;
    const float v0 = row < M && k < TNIN ? xv[it][0] : 0.f;
    const float v1 = row < M && k + 1 < TNIN ? xv[it][1] : 0.f;
    const uint32_t p = f2bf2(v0, v1);
    *(uint32_t*)(sx + m * TLDX + k) = p;
    if (row < M) *(uint32_t*)(a.x0 + row * TKIN + k) = p;
  }
  __syncthreads();
  f32x4 acc[2][MT / 16];
  auto finish = [&](int l, uint16_t* hout) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int n = wv * 32 + i * 16 + 4 * q;
#pragma unroll
      for (int j = 0; j < MT / 16; ++j) {
        const int m = j * 16 + c;
        const float z[4] = {acc[i][j][0] + bias[l][i][0], acc[i][j][1] + bias[l][i][1],
                            acc[i][j][2] + bias[l][i][2], acc[i][j][3] + bias[l][i][3]};
        const float g[4] = {gelu(z[0]), gelu(z[1]), gelu(z[2]), gelu(z[3])};
        *(uint2*)(hout + m * TLD + n) = pack4(g);
        if (row0 + m < M)
          *(float4*)(a.z[l] + (long)(row0 + m) * TNH + n) = float4{z[0], z[1], z[2], z[3]};
      }
    }
    __syncthreads();
    rows_out<MT>(hout, a.h[l], row0, M);
  };
  layer<TKIN, TLDX, MT>(sx, w1, acc);
  load_pair<TNH>(a.wb + TW3, w3);
  finish(0, sh[0]);
  layer<TNH, TLD, MT>(sh[0], w2, acc);
  const int nt = wv & 1, mt = wv >> 1;  // output layer: feature tile, row tile
  if (mt < MT / 16) load_tile<TNH>(a.wb + TW4, nt, w4);
  finish(1, sh[1]);
  layer<TNH, TLD, MT>(sh[1], w3, acc);
  finish(2, sh[0]);
  if (mt >= MT / 16) return;
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < TNH / 32; ++k) {
    V8 h;
    h.q = *(const uint4*)(sh[0] + (mt * 16 + c) * TLD + 32 * k + q * 8);
    o = mfma(w4[k], h, o);
  }
  const long row = row0 + mt * 16 + c;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int n = nt * 16 + 4 * q + r;
    if (row < M && n < TNOUT) a.y[row * TNOUT + n] = o[r] + a.b[3][n];
  }
}

struct TrainDx {
  const float* gy;      // [M][21]
  const uint16_t* wt;   // k_cast_net<true>
  const float* z[3];
  uint16_t* dy;         // [M][32]
  uint16_t* dz[3];      // [M][256]
  float* bpart;         // [block][TBALL]
};

template <int MT>
__global__ __launch_bounds__(TNT, 2) void k_train_dx(TrainDx a, int M) {
  __shared__ __align__(16) uint16_t sy[MT * TLDY];
  __shared__ __align__(16) uint16_t sd[2][MT * TLD];
  __shared__ float sg[MT][TNOUTP + 1];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, q = lane >> 4, c = lane & 15;
  const int row0 = blockIdx.x * MT;
  float* bp = a.bpart + (long)blockIdx.x * TBALL;
  float gv[MT / 16];
#pragma unroll
  for (int it = 0; it < MT / 16; ++it) {
    const int e = tid + TNT * it, m = e >> 5, n = e & 31;
    gv[it] = a.gy[(long)min(row0 + m, M - 1) * TNOUT + min(n, TNOUT - 1)];
  }
  __builtin_amdgcn_sched_barrier(0);
  V8 w4[2][1], w3[2][TNH / 32], w2[2][TNH / 32];
  load_pair<TNOUTP>(a.wt + TW4, w4);
  load_pair<TNH>(a.wt + TW3, w3);
  float4 zv[3][2][MT / 16];
#pragma unroll
  for (int l = 2; l >= 0; --l)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < MT / 16; ++j) {
        const int row = row0 + j * 16 + c;
        zv[l][i][j] = *(const float4*)(a.z[l] + (long)(row < M ? row : M - 1) * TNH + wv * 32 +
                                       i * 16 + 4 * q);
      }
#pragma unroll
  for (int it = 0; it < MT / 16; ++it) {
    const int e = tid + TNT * it, m = e >> 5, n = e & 31;
    const long row = row0 + m;
    const float v = row < M && n < TNOUT ? gv[it] : 0.f;
    const uint16_t p = f2bf(v);
    sy[m * TLDY + n] = p;
    sg[m][n] = v;
    if (row < M) a.dy[row * TNOUTP + n] = p;
  }
  __syncthreads();
  if (tid < TNOUTP) {
    float s = 0.f;
#pragma unroll
    for (int m = 0; m < MT; ++m) s += sg[m][tid];
    bp[3 * TNH + tid] = s;
  }
  f32x4 acc[2][MT / 16];
  // dz of layer l = (dz of l + 1 . W) gelu'(z_l); rows past the batch are zero
  auto finish = [&](int l, uint16_t* out) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int n = wv * 32 + i * 16 + 4 * q;
      float bs[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < MT / 16; ++j) {
        const int m = j * 16 + c;
        const bool in = row0 + m < M;
        const float4 z = zv[l][i][j];
        const float g[4] = {in ? acc[i][j][0] * gelu_d(z.x) : 0.f,
                            in ? acc[i][j][1] * gelu_d(z.y) : 0.f,
                            in ? acc[i][j][2] * gelu_d(z.z) : 0.f,
                            in ? acc[i][j][3] * gelu_d(z.w) : 0.f};
        *(uint2*)(out + m * TLD + n) = pack4(g);
#pragma unroll
        for (int r = 0; r < 4; ++r) bs[r] += g[r];
      }
      // over the 16 rows of a lane quarter
#pragma unroll
      for (int r = 0; r < 4; ++r) bs[r] = row16_sum(bs[r]);
      if (c == 0) *(float4*)(bp + l * TNH + n) = float4{bs[0], bs[1], bs[2], bs[3]};
    }
    __syncthreads();
    rows_out<MT>(out, a.dz[l], row0, M);
  };
  layer<TNOUTP, TLDY, MT>(sy, w4, acc);
  load_pair<TNH>(a.wt + TW2, w2);
  finish(2, sd[0]);
  layer<TNH, TLD, MT>(sd[0], w3, acc);
  finish(1, sd[1]);
  layer<TNH, TLD, MT>(sd[1], w2, acc);
  finish(0, sd[0]);
}

// partial dW[N][K] of rows [mb, me) for one 64 x 64 tile of one layer: 64 rows
// a step, their dZ and X transposed in LDS (two rows of a column side by side
// in 32 bits), the next step's rows requested before the current one is used
struct TrainDw {
  const uint16_t* dz[4];
  const uint16_t* x[4];
  float* part;  // [split][TWALL]
};
constexpr int TDW_TILES = 40;  // 16 + 16 (layers 3, 2), 4 (layer 1), 4 (layer 4)
constexpr int TDW_P = 36;      // LDS row: 64 batch rows in 32 words and a pad

__global__ __launch_bounds__(256) void k_train_dw(TrainDw a, int M, int mchunk) {
  __shared__ __align__(16) uint32_t sz[64][TDW_P], sx[64][TDW_P];
  const int t = blockIdx.x % TDW_TILES, split = blockIdx.x / TDW_TILES;
  const int l = t < 16 ? 2 : t < 32 ? 1 : t < 36 ? 0 : 3;
  const int N = l == 3 ? TNOUTP : TNH, K = l == 0 ? TKIN : TNH;
  const int tl = l == 2 ? t : l == 1 ? t - 16 : l == 0 ? t - 32 : t - 36;
  const int n0 = (tl / (K / 64)) * 64, k0 = (tl % (K / 64)) * 64;
  const uint16_t *dz = a.dz[l], *x = a.x[l];
  const int mb = split * mchunk, me = min(M, mb + mchunk);
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, q = lane >> 4, c = lane & 15;
  const int wn = (wv >> 1) * 32, wk = (wv & 1) * 32;
  // thread -> row pair rp (of 32) and two quads of columns 4 cq, 4 (cq + 8)
  const int cq = tid & 7, rp = tid >> 3;
  uint2 vz[2][2], vx[2][2];  // [quad][row]
  auto load = [&](int m0) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const long m = m0 + 2 * rp + r;
        const int col = 4 * (cq + 8 * u);
        vz[u][r] = vx[u][r] = uint2{0u, 0u};
        if (m < me && n0 + col < N) vz[u][r] = *(const uint2*)(dz + m * N + n0 + col);
        if (m < me) vx[u][r] = *(const uint2*)(x + m * K + k0 + col);
      }
  };
  auto put = [&](uint32_t (*s)[TDW_P], const uint2 (&v)[2][2]) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int col = 4 * (cq + 8 * u);
      s[col][rp] = (v[u][0].x & 0xffffu) | (v[u][1].x << 16);
      s[col + 1][rp] = (v[u][0].x >> 16) | (v[u][1].x & 0xffff0000u);
      s[col + 2][rp] = (v[u][0].y & 0xffffu) | (v[u][1].y << 16);
      s[col + 3][rp] = (v[u][0].y >> 16) | (v[u][1].y & 0xffff0000u);
    }
  };
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  load(mb);
  for (int m0 = mb; m0 < me; m0 += 64) {
    put(sz, vz);
    put(sx, vx);
    __syncthreads();
    if (m0 + 64 < me) load(m0 + 64);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      V8 av[2], bv[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        av[i].q = *(const uint4*)&sz[wn + i * 16 + c][16 * ks + 4 * q];
        bv[i].q = *(const uint4*)&sx[wk + i * 16 + c][16 * ks + 4 * q];
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma(av[i], bv[j], acc[i][j]);
    }
    __syncthreads();
  }
  float* out = a.part + (long)split * TWALL + (l == 0 ? TW1 : l == 1 ? TW2 : l == 2 ? TW3 : TW4);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = n0 + wn + i * 16 + 4 * q + r, k = k0 + wk + j * 16 + c;
        if (n < N) out[n * K + k] = acc[i][j][r];
      }
}

struct TrainSum {
  const float *part, *bpart;
  float *dw[4], *db[4];
};
constexpr int TSUM_W = TWALL / 4 / 256;  // blocks of the weights, 4 values a thread
constexpr int TSUM_B = TBALL / 16;       // blocks of the biases, 16 each

__global__ __launch_bounds__(256) void k_train_sum(TrainSum a, int nsplit, int nblk) {
  static_assert(TWALL % 1024 == 0 && TBALL % 16 == 0, "whole blocks");
  if (blockIdx.x < TSUM_W) {
    const int i = (blockIdx.x * 256 + threadIdx.x) * 4;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
    for (int p = 0; p < nsplit; ++p) s += *(const f32x4*)(a.part + (long)p * TWALL + i);
    const int l = i < TW2 ? 0 : i < TW3 ? 1 : i < TW4 ? 2 : 3;
    const int e = i - (l == 0 ? TW1 : l == 1 ? TW2 : l == 2 ? TW3 : TW4);
    const int K = l == 0 ? TKIN : TNH, nin = l == 0 ? TNIN : TNH, nout = l == 3 ? TNOUT : TNH;
    const int n = e / K, k = e % K;
    if (n >= nout) return;
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (k + u < nin) a.dw[l][n * nin + k + u] = s[u];
    return;
  }
  __shared__ float red[16][17];
  const int col = threadIdx.x & 15, g = threadIdx.x >> 4;
  const int n = (blockIdx.x - TSUM_W) * 16 + col;
  float s = 0.f;
#pragma unroll 4
  for (int b = g; b < nblk; b += 16) s += a.bpart[(long)b * TBALL + n];
  red[g][col] = s;
  __syncthreads();
  if (g > 0) return;
  s = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) s += red[i][col];
  const int l = n / TNH, f = n % TNH;
  if (l < 3 || f < TNOUT) a.db[l][f] = s;
}

// batch rows per block: 16 while that leaves no CU more than one block, which
// halves a small batch's chain; else 32, each weight fragment serving twice the
// rows
int rows_per_block(int M) { return M <= 16 * 256 ? 16 : 32; }
int nsplit_of(int M) { return M / 256 < 1 ? 1 : M / 256 > 64 ? 64 : M / 256; }
long align256(long x) { return (x + 255) & ~255L; }

struct Layout {  // workspace of the backward pass, bytes
  long wt, dy, dz, bpart, part, total;
  explicit Layout(int M) {
    const long nblk = (M + 15) / 16;
    wt = 0;
    dy = align256(wt + 2L * TWALL);
    dz = align256(dy + 2L * M * TNOUTP);
    bpart = align256(dz + 6L * M * TNH);
    part = align256(bpart + 4L * nblk * TBALL);
    total = align256(part + 4L * nsplit_of(M) * TWALL);
  }
};

}  // namespace

extern "C" long exo_mlp_train_work(int M, int backward) {
  if (M < 0) return EXO_RAD_ERR_ARG;
  return backward ? Layout(M).total : 2L * TWALL;
}

extern "C" int exo_mlp_train_forward(int M, const float* x, const float* const* w,
                                     const float* const* b, void* x0, float* const* z,
                                     void* const* h, float* y, void* work, void* stream) {
  if (M < 0 || !w || !b || !z || !h) return EXO_RAD_ERR_ARG;
  if (M == 0) return EXO_RAD_OK;
  if (!x || !x0 || !y || !work) return EXO_RAD_ERR_ARG;
  TrainFwd a{};
  TrainW p{};
  for (int l = 0; l < 4; ++l) {
    if (!w[l] || !b[l] || (l < 3 && (!z[l] || !h[l]))) return EXO_RAD_ERR_ARG;
    p.w[l] = w[l];
    a.b[l] = b[l];
    if (l < 3) {
      a.z[l] = z[l];
      a.h[l] = (uint16_t*)h[l];
    }
  }
  a.x = x;
  a.wb = (const uint16_t*)work;
  a.x0 = (uint16_t*)x0;
  a.y = y;
  hipStream_t s = (hipStream_t)stream;
  k_cast_net<false><<<TWALL / 256, 256, 0, s>>>(p, (uint16_t*)work);
  const int mt = rows_per_block(M);
  const unsigned nblk = (unsigned)((M + mt - 1) / mt);
  if (mt == 16)
    k_train_fwd<16><<<nblk, TNT, 0, s>>>(a, M);
  else
    k_train_fwd<32><<<nblk, TNT, 0, s>>>(a, M);
  return hipGetLastError() == hipSuccess ? EXO_RAD_OK : EXO_RAD_ERR_HIP;
}

extern "C" int exo_mlp_train_backward(int M, const float* gy, const void* x0,
                                      const float* const* z, const void* const* h,
                                      const float* const* w, float* const* dw, float* const* db,
                                      void* work, void* stream) {
  if (M < 1 || !gy || !x0 || !z || !h || !w || !dw || !db || !work) return EXO_RAD_ERR_ARG;
  const Layout lay(M);
  char* base = (char*)work;
  uint16_t *wt = (uint16_t*)(base + lay.wt), *dy = (uint16_t*)(base + lay.dy);
  uint16_t* dz = (uint16_t*)(base + lay.dz);
  float *bpart = (float*)(base + lay.bpart), *part = (float*)(base + lay.part);
  TrainW p{};
  TrainDx d{};
  TrainDw g{};
  TrainSum t{};
  for (int l = 0; l < 4; ++l) {
    if (!w[l] || !dw[l] || !db[l] || (l < 3 && (!z[l] || !h[l]))) return EXO_RAD_ERR_ARG;
    p.w[l] = w[l];
    t.dw[l] = dw[l];
    t.db[l] = db[l];
    g.x[l] = (const uint16_t*)(l == 0 ? x0 : h[l - 1]);
    g.dz[l] = l == 3 ? dy : dz + (long)l * M * TNH;
    if (l < 3) {
      d.z[l] = z[l];
      d.dz[l] = dz + (long)l * M * TNH;
    }
  }
  d.gy = gy;
  d.wt = wt;
  d.dy = dy;
  d.bpart = bpart;
  t.bpart = bpart;
  g.part = part;
  t.part = part;
  hipStream_t s = (hipStream_t)stream;
  k_cast_net<true><<<TWALL / 256, 256, 0, s>>>(p, wt);
  const int mt = rows_per_block(M), nblk = (M + mt - 1) / mt;
  if (mt == 16)
    k_train_dx<16><<<nblk, TNT, 0, s>>>(d, M);
  else
    k_train_dx<32><<<nblk, TNT, 0, s>>>(d, M);
  int mchunk = (M + nsplit_of(M) - 1) / nsplit_of(M);
  mchunk = (mchunk + 31) / 32 * 32;
  const int ns = (M + mchunk - 1) / mchunk;
  k_train_dw<<<TDW_TILES * ns, 256, 0, s>>>(g, M, mchunk);
  k_train_sum<<<TSUM_W + TSUM_B, 256, 0, s>>>(t, ns, nblk);
  return hipGetLastError() == hipSuccess ? EXO_RAD_OK : EXO_RAD_ERR_HIP;
}
