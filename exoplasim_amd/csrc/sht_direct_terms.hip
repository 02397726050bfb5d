// sht_direct_terms.hip -- folded direct Legendre transforms with several
// Fourier inputs and tables (src/legmod.f90 folded branches):
//   uv2dv  (:391-422)   (u, v)                       -> (D, zeta)
//   qtend  (:468-496)   (qn, uq, vq)                 -> q
//   mktend (:555-602)   (tn, fu, fv, ke, ut, vt)     -> (D, T, zeta)
// Each output field is a sum of terms  sign * t[pair][w] * X_i[m][cls][pair][c]
// where X_i is input i folded into E = N+S (class sym) / O = N-S (class anti)
// and the class of table t at (m,n) is sym iff (n-m even) != (t is Q-type).
//
// Per zonal wavenumber m and parity p of n - m, each output is a GEMM over
// the latitude pairs:  C[n][lev, oc] = sum_t sum_pair A_t[n][pair] B_t[pair][lev, oc]
// with A_t the table t at the rows n = m + p + 2j and B_t[pair][lev, oc] =
// sign * X_in[cls][pair][m][lev][ic] for the term of table t and output
// component oc.  One 16x16x4 MFMA (v_mfma_f32_16x16x4_f32, in the FP64 mode
// v_mfma_f64_16x16x4_f64) takes 16 rows n x 4 pairs of A and 4 pairs x 16
// columns (8 levels x re/im) of B, so each table value serves 8 levels.
//
// A block owns one member, 8 levels and MR wavenumbers of one job: up to 3
// inputs (one table each) and up to 2 outputs that share them.  It walks the
// latitude pairs KC at a time: the folded Fourier values of those pairs
// (all inputs, its levels and wavenumbers) are staged in LDS, and the tables
// and inputs of the steps ahead are in flight through the MFMAs; every
// (output, m, p, row tile) accumulates in registers across all pairs, so the
// sum over latitudes is complete in the block (no partial sums).  Wave w takes
// m = m0 + w.
//
// What bounds it is the latency of those steps (stage, barrier, tables), not
// bytes or flops, so the jobs of one call run in one launch: the blocks of
// mktend's and gridpointa's four outputs overlap, and divergence and
// vorticity, which share two of their inputs and tables, are one job (one
// launch per output before: mktend of T42 L20, 32 members, FP32, 69.6 -> 51
// us; T63, 16 members, 81 -> 57; T127 L40, 4 members, 242 -> 184).  In FP64
// the vector and matrix peaks are equal; the matrix form wins over one thread
// per coefficient, which read each table value once per level, by that reuse
// (mktend T42 251 -> 95 us, T63 388 -> 101, T127 2320 -> 273), and needs no
// partial sums in scratch.
#include <type_traits>

#include "sht_internal.h"

namespace exo {

constexpr int DIRX_MR = 8;  // wavenumbers per block, one per wave
constexpr int DIRX_NT = 512, DIRX_LG = 8;  // threads, levels per block

template <int T, typename R, int NIN>
struct DirxCfg {
  static constexpr int NMR = (TS<T>::NM + DIRX_MR - 1) / DIRX_MR;
  // Pairs per step: as many as the step's table operands allow in registers
  // (fewer inputs, more pairs).  FP64 operands take twice the registers and
  // the LDS.
  static constexpr int KC = (sizeof(R) == 8) ? ((NIN == 1) ? 8 : 4)
                            : (NIN == 1)     ? ((T == 127) ? 8 : 16)
                            : (NIN == 2 && T == 63) ? 16
                                                    : 8;
  static constexpr int KS = DIRX_LG * 2 * DIRX_MR + 2;  // reals per (input, class, pair), padded
  // FP32: two staged steps in LDS and two steps' tables in registers; FP64's
  // registers leave no room for the second (T127 L10 gridpointa 233 -> 283 us)
  static constexpr bool AHEAD = sizeof(R) == 4;
  static constexpr int STEP = NIN * 2 * KC * KS;  // reals of one staged step
  static constexpr size_t LDS = sizeof(R) * STEP * (AHEAD ? 2 : 1);
};

// one job: the term list regrouped by table.  Slot s multiplies table tab[s]
// by, for output o and component oc, sign[o][s][oc] * X_in[o][s][oc] component
// ic[o][s][oc] (sign 0: no term); every list here has one table per input.
template <typename R>
struct DirxJob {
  const R* in[3];
  R* out[2];
  const R* tab[3];  // FP32: the packed table (k_pack_dir); FP64: [pair][w]
  int nin, nout, nlev, nlg;
  long in_stride, out_stride;
  int8_t sign[2][3][2], src[2][3][2], ic[2][3][2], isq[3];
};
constexpr int DIRX_JOBS = 4;
template <typename R>
struct DirxJobs {
  int njob, nmem, per;        // per: blocks per member
  int start[DIRX_JOBS + 1];   // first block of each job within a member
  DirxJob<R> job[DIRX_JOBS];
};

// RB: row tiles of 16 per parity that the block's wavenumbers need (dirx_run)
template <int T, typename R, int NIN, int NOUT, int RB>
__device__ __forceinline__ void dirx_body(const DirxJob<R>& a, int mem, int lg, int mr,
                                          char* lds) {
  using S = TS<T>;
  using C = DirxCfg<T, R, NIN>;
  using R2 = R __attribute__((ext_vector_type(2)));
  using Acc = typename std::conditional<sizeof(R) == 8, f64x4, f32x4>::type;
  constexpr bool F64 = sizeof(R) == 8;
  constexpr int N = S::NLON, NLAT = S::NLAT, NPAIR = S::NPAIR, NCSP = S::NCSP;
  constexpr int MR = DIRX_MR, LG = DIRX_LG, KC = C::KC, KS = C::KS, NT = DIRX_NT;
  constexpr int NKS = KC / 4;  // MFMA K steps (4 pairs each) per staged step
  constexpr int NJ = 2 * MR;   // reals of one staged row segment
  static_assert(NPAIR % KC == 0, "pairs per step");
  static_assert(MR == NT / 64, "one wavenumber per wave");
  // staged values per step: (input, level, pair, 4 reals) with the reals
  // fastest, 16-byte loads
  constexpr int NJ4 = NJ / 4;
  constexpr int NITEM = NIN * LG * KC * NJ4;
  constexpr int MAXIT = (NITEM + NT - 1) / NT;
  R* const X0 = (R*)lds;  // [step % 2 (AHEAD)][input][class][pair][level][m][re/im]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m0 = mr * MR, lev0 = lg * LG;
  const int nl = a.nlev - lev0 < LG ? a.nlev - lev0 : LG;  // levels of this block

  // A wave stages items of one input: its levels of this block as one buffer,
  // so that levels past the last load zeros (2 m0 + NJ <= N: the 16-byte runs
  // stay inside their rows; reals past the truncation are staged and not used).
  // The loads have no branch and no arithmetic on their results, which would
  // wait for them here instead of at the next step's fold.
  static_assert(NJ4 * KC * LG % 64 == 0, "one input per wave");
  static_assert(2 * ((TS<T>::NM - 1) / MR * MR) + NJ <= N, "staged runs inside a row");
  constexpr int ES = (int)sizeof(R), NC = NPAIR / KC;
  __amdgpu_buffer_rsrc_t rsi[MAXIT];
  int vn[MAXIT], vs[MAXIT];  // byte offsets of the northern run of step 0, the southern of step NC - 1
#pragma unroll
  for (int it = 0; it < MAXIT; ++it) {
    const int e = tid + NT * it;
    const int j4 = e % NJ4, k = (e / NJ4) % KC, l = (e / (NJ4 * KC)) % LG;
    const int i = (64 * wv + NT * it) / (NJ4 * KC * LG);
    const R* in = NIN > 2 && i == 2 ? a.in[NIN > 2 ? 2 : 0] : NIN > 1 && i == 1 ? a.in[1] : a.in[0];
    rsi[it] = buffer_rsrc(in + mem * a.in_stride + (long)lev0 * NLAT * N, nl * NLAT * N * ES);
    const int o = l * NLAT * N + 2 * m0 + 4 * j4;
    vn[it] = e < NITEM ? (o + k * N) * ES : BUF_NONE;
    vs[it] = e < NITEM ? (o + (NLAT - NPAIR + KC - 1 - k) * N) * ES : BUF_NONE;
  }
  auto quad = [&](__amdgpu_buffer_rsrc_t rs, int off, int soff, R* v) {
    uint4 u[sizeof(R) / 4];
#pragma unroll
    for (int h = 0; h < (int)sizeof(R) / 4; ++h) u[h] = buffer_load_x4(rs, off + 16 * h, soff);
    __builtin_memcpy(v, u, 4 * sizeof(R));
  };
  R rn[MAXIT][4], rs[MAXIT][4];
  auto load = [&](int c) {
#pragma unroll
    for (int it = 0; it < MAXIT; ++it) {
      quad(rsi[it], vn[it], c * KC * N * ES, rn[it]);
      quad(rsi[it], vs[it], (NC - 1 - c) * KC * N * ES, rs[it]);
    }
  };
  // fold into E = N + S (class 0) and O = N - S (class 1)
  auto store = [&](R* X) {
#pragma unroll
    for (int it = 0; it < MAXIT; ++it) {
      const int e = tid + NT * it;
      if (64 * wv + NT * it < NITEM) {
        const int j4 = e % NJ4, k = (e / NJ4) % KC, l = (e / (NJ4 * KC)) % LG,
                  i = e / (NJ4 * KC * LG);
        const int o = l * NJ + 4 * j4;  // even, and KS is even: pairs of reals are aligned
        R2* xe = (R2*)&X[((i * 2 + 0) * KC + k) * KS + o];
        R2* xo = (R2*)&X[((i * 2 + 1) * KC + k) * KS + o];
        xe[0] = R2{rn[it][0] + rs[it][0], rn[it][1] + rs[it][1]};
        xe[1] = R2{rn[it][2] + rs[it][2], rn[it][3] + rs[it][3]};
        xo[0] = R2{rn[it][0] - rs[it][0], rn[it][1] - rs[it][1]};
        xo[1] = R2{rn[it][2] - rs[it][2], rn[it][3] - rs[it][3]};
      }
    }
  };

  // A operand: row r = lane & 15, pair 4 ks + (lane >> 4) of the step; B
  // operand: column lane & 15 = (level l, component oc), the same pair
  const int r = lane & 15, kq = lane >> 4, l = (lane & 15) >> 1, oc = lane & 1;
  // (the waves past the truncation repeat the last wavenumber's tables and
  // store nothing)
  const int m = m0 + wv < T ? m0 + wv : T;
  const int w0 = w0_of(T, m);
  Acc acc[NOUT][2][RB];
#pragma unroll
  for (int o = 0; o < NOUT; ++o)
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int rt = 0; rt < RB; ++rt) acc[o][p][rt] = Acc{0, 0, 0, 0};
  // this lane's B source per output, slot and parity: offset of (input, class,
  // pair kq, level l, component ic) in X, and the sign bit.  Of the folded
  // input the symmetric class (E) iff (n - m even) != Q-type table.
  auto term = [](int o, int s) { return !(NIN == 3 && NOUT == 2 && o == 1 && s == 0); };
  int boff[NOUT][NIN][2];
  uint32_t bsg[NOUT][NIN];
#pragma unroll
  for (int o = 0; o < NOUT; ++o)
#pragma unroll
    for (int s = 0; s < NIN; ++s) {
      const int src = oc ? a.src[o][s][1] : a.src[o][s][0];
      const int ic = oc ? a.ic[o][s][1] : a.ic[o][s][0];
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int cls = (p == 0) == (a.isq[s] != 0) ? 1 : 0;
        boff[o][s][p] = ((src * 2 + cls) * KC + kq) * KS + l * NJ + ic + 2 * wv;
      }
      bsg[o][s] = (oc ? a.sign[o][s][1] : a.sign[o][s][0]) < 0 ? 0x80000000u : 0u;
    }
  // FP64 tables are read as they are, [pair][w]: the pair of reals at w0 +
  // 2 (16 rt + r) holds the rows n of both parities, so one 16-byte load
  // feeds both parities' MFMAs; rows past the truncation hold other
  // coefficients, and their results are not stored
  __amdgpu_buffer_rsrc_t rst[NIN];
  if constexpr (F64) {
#pragma unroll
    for (int s = 0; s < NIN; ++s) rst[s] = buffer_rsrc(a.tab[s], NPAIR * NCSP * 8);
  }

  auto tables = [&](int c, R (&av)[NIN][2][RB][NKS]) {
#pragma unroll
    for (int s = 0; s < NIN; ++s)
#pragma unroll
      for (int rt = 0; rt < RB; ++rt) {
        if constexpr (F64) {
#pragma unroll
          for (int ks = 0; ks < NKS; ++ks) {
            const uint4 v = buffer_load_x4(rst[s], (kq * NCSP + 2 * r) * 8,
                                           ((c * KC + 4 * ks) * NCSP + w0 + 32 * rt) * 8);
            R d[2];
            __builtin_memcpy(d, &v, 16);
            av[s][0][rt][ks] = d[0];
            av[s][1][rt][ks] = d[1];
          }
        } else {
          // one 16-byte load per 8 pairs and row tile: 2 K steps of both parities
#pragma unroll
          for (int g = 0; g < KC / 8; ++g) {
            const f32x4 v = ((const f32x4*)a.tab[s])[((m * S::RB + rt) * (NPAIR / 8) +
                                                      c * (KC / 8) + g) * 64 + lane];
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
              for (int h = 0; h < 2; ++h) av[s][p][rt][2 * g + h] = v[2 * p + h];
          }
        }
      }
  };
  auto products = [&](const R* X, const R (&av)[NIN][2][RB][NKS]) {
#pragma unroll
    for (int s = 0; s < NIN; ++s)
#pragma unroll
      for (int o = 0; o < NOUT; ++o) {
        if (!term(o, s)) continue;
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
          for (int p = 0; p < 2; ++p) {
            const R bv = flip_sign(X[boff[o][s][p] + 4 * ks * KS], bsg[o][s]);
#pragma unroll
            for (int rt = 0; rt < RB; ++rt) {
              if constexpr (F64)
                acc[o][p][rt] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[s][p][rt][ks], bv,
                                                                     acc[o][p][rt], 0, 0, 0);
              else
                acc[o][p][rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[s][p][rt][ks], bv,
                                                                     acc[o][p][rt], 0, 0, 0);
            }
          }
      }
  };
  load(0);
  if constexpr (C::AHEAD) {
    // While step c is multiplied, the tables of step c + 1 and the inputs of
    // step c + 2 are on their way, and the inputs of step c + 1 are folded into
    // the other half of LDS.  One barrier per step: behind it the half of step c
    // is complete, and that of step c - 1 no longer read.  (One step and two
    // barriers: T42 L20, 32 members, gridpointa 241 us against 237, T127 L20, 2
    // members, 312 against 290, the T127 round trip 722 against 713.)
    R av[2][NIN][2][RB][NKS];
    tables(0, av[0]);
    store(X0);
    if (NC > 1) load(1);
    auto step = [&](int c, const R (&cur)[NIN][2][RB][NKS], R (&next)[NIN][2][RB][NKS]) {
      __syncthreads();
      if (c + 1 < NC) tables(c + 1, next);
      products(X0 + (c & 1) * C::STEP, cur);
      if (c + 1 < NC) store(X0 + ((c + 1) & 1) * C::STEP);
      if (c + 2 < NC) load(c + 2);
    };
    for (int c = 0; c < NC; c += 2) {
      step(c, av[0], av[1]);
      if (NC % 2 == 0 || c + 1 < NC) step(c + 1, av[1], av[0]);
    }
  } else {
    for (int c = 0; c < NC; ++c) {
      __syncthreads();  // the previous step's MFMAs have read X
      store(X0);
      __syncthreads();
      // every A operand of this step first, so that their latencies overlap;
      // then the next step's inputs, whose loads stay in flight through the
      // MFMAs
      R av[NIN][2][RB][NKS];
      tables(c, av);
      if (c + 1 < NC) load(c + 1);
      products(X0, av);
    }
  }
  // item v of a lane is row 4 kq + v of column (l, oc); in the FP64 form row
  // 4 v + kq
  if (l >= nl || m0 + wv > T) return;
#pragma unroll
  for (int o = 0; o < NOUT; ++o) {
    R* out = a.out[o] + mem * a.out_stride + (long)(lev0 + l) * S::NRSP;
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int rt = 0; rt < RB; ++rt)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int dn = p + 2 * (16 * rt + (F64 ? 4 * v + kq : 4 * kq + v));
          if (m + dn <= T) out[2 * (w0 + dn) + oc] = acc[o][p][rt][v];
        }
  }
}

// The block's wavenumbers m0 .. m0 + 7 need the row tiles of m0 (n - m = 0 .. T
// - m0); the tile count is a template argument of the body, so that its products
// have no branches between them.  (A branch per product, on the wavenumber's
// own tile count, and one per operand for terms that a list does not have, kept
// the compiler from overlapping any of a step's loads: T42 L20, 32 members,
// gridpointa 241 us against 258, T21 L10 FP64, one member, 28.5 against 31.9, T127
// L40 round trip of 8 members 722 against 736.)
template <int T, typename R, int NIN, int NOUT, int RB = 1>
__device__ __forceinline__ void dirx_run(const DirxJob<R>& a, int mem, int lg, int mr, char* lds) {
  if constexpr (RB < TS<T>::RB) {
    if ((T - mr * DIRX_MR) / 2 >= 16 * RB) {
      dirx_run<T, R, NIN, NOUT, RB + 1>(a, mem, lg, mr, lds);
      return;
    }
  }
  dirx_body<T, R, NIN, NOUT, RB>(a, mem, lg, mr, lds);
}

// Minimum waves per SIMD asked of the compiler: two blocks per CU instead of
// one where the FP64 registers come down to 128 with at most 18 of them
// spilled (T42 L20, 32 members: mktend 95 against 100 us, uv2dv 38 against 46;
// T63 mktend spills as much for 103 against 100 us, and T127 more: those keep
// their registers)
template <int T, typename R, int NOUT, int NIN>
constexpr int dirx_waves() {
  return sizeof(R) == 8 && (T == 42 || (T == 63 && NIN == 2)) ? 4 : 2;
}

// One job alone: fc2sp of Fourier fields, uv2dv, qtend.  (qtend in the kernel
// below, which holds the two-output body's registers: T127 L40, 4 members,
// 112 us against 89.)
template <int T, typename R, int NIN, int NOUT>
__global__ __launch_bounds__(DIRX_NT, (dirx_waves<T, R, NOUT, NIN>())) void k_dirx_one(
    DirxJob<R> a, int per) {
  __shared__ __align__(16) char lds[DirxCfg<T, R, NIN>::LDS];
  constexpr int NMR = DirxCfg<T, R, NIN>::NMR;
  // neighbouring wavenumber ranges stage the two halves of the same 128-byte
  // lines of a Fourier row: renumbered so that they run on one XCD's L2
  const int b = xcd_block(blockIdx.x, gridDim.x);
  const int mem = b / per, i = b - mem * per;
  dirx_run<T, R, NIN, NOUT>(a, mem, i / NMR, i % NMR, lds);
}

// mktend, gridpointa: jobs of three inputs and one or two outputs, and of one
// input, in one launch (blocks as above, a member's jobs side by side)
template <int T, typename R>
__global__ __launch_bounds__(DIRX_NT, (dirx_waves<T, R, 2, 3>())) void k_dirx_mf(DirxJobs<R> j) {
  __shared__ __align__(16) char lds[DirxCfg<T, R, 3>::LDS > DirxCfg<T, R, 1>::LDS
                                        ? DirxCfg<T, R, 3>::LDS
                                        : DirxCfg<T, R, 1>::LDS];
  constexpr int NMR = DirxCfg<T, R, 1>::NMR;
  const int b = xcd_block(blockIdx.x, gridDim.x);
  const int mem = b / j.per;
  const int q = b - mem * j.per;
  int k = 0;
#pragma unroll
  for (int i = 1; i < DIRX_JOBS; ++i)
    if (i < j.njob && q >= j.start[i]) k = i;
  k = __builtin_amdgcn_readfirstlane(k);
  const DirxJob<R>& a = j.job[k];
  const int i = q - j.start[k];
  const int mr = i % NMR, lg = i / NMR;
  if (a.nin == 1)
    dirx_run<T, R, 1, 1>(a, mem, lg, mr, lds);
  else if (a.nout == 1)
    dirx_run<T, R, 3, 1>(a, mem, lg, mr, lds);
  else
    dirx_run<T, R, 3, 2>(a, mem, lg, mr, lds);
}

template <int T, typename R>
static int dirx_t(const Tables& tb, const DirxArgs* args, int njob, hipStream_t s) {
  if (njob < 1 || njob > DIRX_JOBS) return -2;
  DirxJobs<R> jobs{};
  jobs.nmem = args[0].nmem;
  bool wide = false;  // a job with three inputs
  for (int k = 0; k < njob; ++k) {
    const DirxArgs& a = args[k];
    DirxJob<R>& g = jobs.job[jobs.njob];
    if (a.nmem != jobs.nmem || a.nin < 1 || a.nin > 3 || a.nout < 1 || a.nout > 2) return -2;
    if (a.nlev <= 0) continue;
    const R* tabs[3] = {};
    int nslot = 0;
    for (int t = 0; t < a.nterm; ++t) {
      const DirxTerm& tm = a.terms[t];
      const R* tab;
      if constexpr (sizeof(R) == 8)
        tab = tb.filt64 + (long)tm.table * tb.npair * tb.ncsp;
      else
        tab = tb.dir_f32[tm.table];
      int i = 0;
      while (i < nslot && tabs[i] != tab) ++i;
      if (i == nslot) {
        if (i == 3 || !tab) return -2;
        tabs[nslot++] = tab;
        g.tab[i] = tab;
        g.isq[i] = table_is_q(tm.table) ? 1 : 0;
      }
      if (g.sign[tm.o][i][tm.oc] != 0) return -2;  // one term per (output, table, component)
      g.sign[tm.o][i][tm.oc] = tm.sign;
      g.src[tm.o][i][tm.oc] = tm.in;
      g.ic[tm.o][i][tm.oc] = tm.ic;
    }
    if (nslot != a.nin) return -2;  // one table per input
    if (a.nin < 3 && a.nin != a.nout) return -2;
    // every output has a term of every table, but the second of three inputs'
    // (mktend's vorticity) none of the first
    for (int o = 0; o < a.nout; ++o)
      for (int i = 0; i < a.nin; ++i)
        for (int c = 0; c < 2; ++c)
          if ((g.sign[o][i][c] != 0) != !(a.nin == 3 && a.nout == 2 && o == 1 && i == 0)) return -2;
    wide = wide || a.nin == 3;
    for (int i = 0; i < a.nin; ++i) g.in[i] = (const R*)a.in[i];
    for (int o = 0; o < a.nout; ++o) g.out[o] = (R*)a.out[o];
    g.nin = a.nin;
    g.nout = a.nout;
    g.nlev = a.nlev;
    g.nlg = (a.nlev + DIRX_LG - 1) / DIRX_LG;
    g.in_stride = a.in_stride;
    g.out_stride = a.out_stride;
    jobs.per += DirxCfg<T, R, 1>::NMR * g.nlg;
    jobs.start[++jobs.njob] = jobs.per;
  }
  const long nblk = (long)jobs.nmem * jobs.per;
  if (nblk <= 0) return 0;
  const int nin = jobs.job[0].nin, nout = jobs.job[0].nout;
  const dim3 grid((unsigned)nblk);
  if (jobs.njob > 1 || (nin == 3 && nout == 2)) {
    for (int k = 0; k < jobs.njob; ++k)
      if (!wide || jobs.job[k].nin == 2) return -2;
    k_dirx_mf<T, R><<<grid, DIRX_NT, 0, s>>>(jobs);
  } else if (nin == 3) {
    k_dirx_one<T, R, 3, 1><<<grid, DIRX_NT, 0, s>>>(jobs.job[0], jobs.per);
  } else if (nin == 2) {
    k_dirx_one<T, R, 2, 2><<<grid, DIRX_NT, 0, s>>>(jobs.job[0], jobs.per);
  } else {
    k_dirx_one<T, R, 1, 1><<<grid, DIRX_NT, 0, s>>>(jobs.job[0], jobs.per);
  }
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int launch_dirx(const Tables& tb, int mode, const DirxArgs* args, int njob, hipStream_t s) {
  const bool d = (mode == MODE_F64);
  switch (tb.ntru) {
    case 21: return d ? dirx_t<21, double>(tb, args, njob, s) : dirx_t<21, float>(tb, args, njob, s);
    case 42: return d ? dirx_t<42, double>(tb, args, njob, s) : dirx_t<42, float>(tb, args, njob, s);
    case 63: return d ? dirx_t<63, double>(tb, args, njob, s) : dirx_t<63, float>(tb, args, njob, s);
    case 127:
      return d ? dirx_t<127, double>(tb, args, njob, s) : dirx_t<127, float>(tb, args, njob, s);
    default: return -2;
  }
}

}  // namespace exo
