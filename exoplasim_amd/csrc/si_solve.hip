// si_solve.hip -- the semi-implicit spectral solve in FP64 on the GPU.
//
//   k_makebm      bm1(:,:,n) = inverse(delt^2 (t0 dsigma + g.tau) + I/(n(n+1)))
//                 for n = 1..NTRU (src/plasim.f90:1683-1703), one workgroup
//                 per n, Gauss-Jordan elimination with partial pivoting in LDS.
//   k_si_apply    divergence at time t from eq. 17 of Hoskins & Simmons
//                 (1975) and the ln(ps) and temperature updates
//                 (src/plasim.f90:2817-2876), 16 spectral reals x 16 levels
//                 per block.
// Matrices are column-major NLEV x NLEV as in the reference.
#include <hip/hip_runtime.h>

#include "../../include/exo_si.h"

namespace {

constexpr int MAXLEV = 64;

__global__ void k_makebm(int nlev, int ntru, double delt, const double* t0,
                         const double* dsigma, const double* g, const double* tau,
                         double* bm1, int* status) {
  const int jn = blockIdx.x + 1;  // total wavenumber 1..ntru
  if (jn > ntru) return;
  __shared__ double a[MAXLEV][2 * MAXLEV + 1];  // [row][col], augmented [A | I]
  __shared__ int piv;
  const int tid = threadIdx.x;
  const int n2 = 2 * nlev;
  const double zdeltsq = delt * delt;
  // A(j2, j1) = delt^2 (t0(j1) dsigma(j2) + g(:,j1).tau(j2,:)) + delta/(n(n+1))
  for (int idx = tid; idx < nlev * nlev; idx += blockDim.x) {
    const int j2 = idx % nlev, j1 = idx / nlev;
    double dp = 0.0;
    for (int k = 0; k < nlev; ++k) dp += g[j1 * nlev + k] * tau[k * nlev + j2];
    double v = zdeltsq * (t0[j1] * dsigma[j2] + dp);
    if (j1 == j2) v += 1.0 / (double)(jn * (jn + 1));
    a[j2][j1] = v;
    a[j2][nlev + j1] = (j1 == j2) ? 1.0 : 0.0;
  }
  __syncthreads();
  for (int col = 0; col < nlev; ++col) {
    if (tid == 0) {
      int p = col;
      double best = fabs(a[col][col]);
      for (int r = col + 1; r < nlev; ++r)
        if (fabs(a[r][col]) > best) {
          best = fabs(a[r][col]);
          p = r;
        }
      piv = p;
      if (best == 0.0) atomicExch(status, 1);
    }
    __syncthreads();
    const int p = piv;
    if (p != col)
      for (int c = tid; c < n2; c += blockDim.x) {
        const double t = a[col][c];
        a[col][c] = a[p][c];
        a[p][c] = t;
      }
    __syncthreads();
    const double inv = 1.0 / a[col][col];
    __syncthreads();
    for (int c = tid; c < n2; c += blockDim.x) a[col][c] *= inv;
    __syncthreads();
    for (int idx = tid; idx < nlev * n2; idx += blockDim.x) {
      const int r = idx / n2, c = idx % n2;
      if (r != col && c != col) a[r][c] -= a[r][col] * a[col][c];
    }
    __syncthreads();
    for (int r = tid; r < nlev; r += blockDim.x)
      if (r != col) a[r][col] = 0.0;
    __syncthreads();
  }
  double* out = bm1 + (long)(jn - 1) * nlev * nlev;
  for (int idx = tid; idx < nlev * nlev; idx += blockDim.x) {
    const int r = idx % nlev, c = idx / nlev;
    out[c * nlev + r] = a[r][nlev + c];
  }
}

// Interface arrays of type R (the model's real kind); arithmetic in FP64.
// A block takes SI_CB consecutive spectral reals and all levels: thread (c, l0)
// owns column c and the levels l0, l0 + SI_LB, ..., so that a single member
// fills the chip and the spectral arrays are read in whole 128-byte lines.
// The column's temperatures and the right-hand side of eq. 17 meet in LDS
// between the three matrix products (g, bm1 of the column's total
// wavenumber, tau), whose rows are contiguous per thread and come from L2;
// every sum runs in the order of the levels.  (One thread per column, with
// its level arrays in per-lane memory, kept 4 of 256 CUs busy at T21: the
// call took 34.9 us at T21 L10, 141 us at T42 L20 and 621 us at T127 L40 in
// FP64, against 4.8, 7.9 and 45.8 us.)
constexpr int SI_CB = 16, SI_LB = 16;

template <typename R>
__global__ __launch_bounds__(SI_CB* SI_LB) void k_si_apply(
    int nlev, int nsp, const int* nindex, double delt, const double* t0, const double* dsigma,
    const double* g, const double* tau, const double* bm1, const R* sop, const R* spm,
    const R* atm, const R* adm, R* stt, R* sdt, R* spt) {
  __shared__ double st[MAXLEV][SI_CB], at[MAXLEV][SI_CB];
  __shared__ double zz[MAXLEV][SI_CB], d[MAXLEV][SI_CB];
  const int c = threadIdx.x % SI_CB, l0 = threadIdx.x / SI_CB;
  const int jsp = blockIdx.x * SI_CB + c;
  const bool live = jsp < nsp;  // no early return: the block meets at barriers
  const int jn = live ? nindex[jsp] : 0;
  const double zq = jn > 0 ? 1.0 / (double)(jn * (jn + 1)) : 0.0;
  for (int l = l0; l < nlev; l += SI_LB) {
    st[l][c] = live ? (double)stt[(long)l * nsp + jsp] : 0.0;
    at[l][c] = live ? (double)atm[(long)l * nsp + jsp] : 0.0;
  }
  const double sp_t = live ? (double)spt[jsp] : 0.0, sp_m = live ? (double)spm[jsp] : 0.0;
  const double so = live ? (double)sop[jsp] : 0.0;
  __syncthreads();
  // rhs of eq. 17 of level l
  for (int l = l0; l < nlev; l += SI_LB) {
    const double ds = live ? (double)sdt[(long)l * nsp + jsp] : 0.0;
    const double dm = live ? (double)adm[(long)l * nsp + jsp] : 0.0;
    double zgt = 0, zgm = 0;
#pragma unroll 4
    for (int k = 0; k < nlev; ++k) {
      const double gk = g[l * nlev + k];
      zgt += gk * st[k][c];
      zgm += gk * at[k][c];
    }
    const double z0 = t0[l];
    const double zt = zgt - z0 * sp_t;
    const double zm = zgm + z0 * sp_m;
    const double za = ds * zq + so;
    const double zb = dm * zq;
    zz[l][c] = zb + delt * (zm + za + delt * zt);
  }
  __syncthreads();
  for (int l = l0; l < nlev; l += SI_LB) {
    double zsum = 0;
    if (jn > 0) {
      const double* b = bm1 + (long)(jn - 1) * nlev * nlev + (long)l * nlev;
#pragma unroll 4
      for (int l2 = 0; l2 < nlev; ++l2) zsum += zz[l2][c] * b[l2];
    }
    d[l][c] = (jsp < 2) ? 0.0 : zsum;  // first mode is zero (src/plasim.f90:2860)
  }
  __syncthreads();
  if (!live) return;
  if (l0 == 0) {
    double ps = sp_t;
    for (int l = 0; l < nlev; ++l) ps += dsigma[l] * d[l][c];
    spt[jsp] = (R)ps;
  }
  for (int l = l0; l < nlev; l += SI_LB) {
    double s = 0;
#pragma unroll 4
    for (int k = 0; k < nlev; ++k) s += tau[l * nlev + k] * d[k][c];
    stt[(long)l * nsp + jsp] = (R)(st[l][c] - s);
    sdt[(long)l * nsp + jsp] = (R)d[l][c];
  }
}

}  // namespace

struct exo_si_s {
  int nlev = 0, ntru = 0, nsp = 0;
  double *t0 = nullptr, *dsigma = nullptr, *g = nullptr, *tau = nullptr, *bm1 = nullptr;
  int* nindex = nullptr;
  int* status = nullptr;
};

#define HIPCK(x)                              \
  do {                                        \
    if ((x) != hipSuccess) return EXO_SI_ERR_HIP; \
  } while (0)

extern "C" int exo_si_create(exo_si_t* si, int nlev, int ntru, const double* t0,
                             const double* dsigma, const double* g, const double* tau) {
  if (!si || nlev < 1 || nlev > MAXLEV || ntru < 1 || !t0 || !dsigma || !g || !tau)
    return EXO_SI_ERR_ARG;
  exo_si_s* s = new exo_si_s();
  s->nlev = nlev;
  s->ntru = ntru;
  s->nsp = (ntru + 1) * (ntru + 2);
  const size_t m2 = sizeof(double) * nlev * nlev;
  HIPCK(hipMalloc(&s->t0, sizeof(double) * nlev));
  HIPCK(hipMalloc(&s->dsigma, sizeof(double) * nlev));
  HIPCK(hipMalloc(&s->g, m2));
  HIPCK(hipMalloc(&s->tau, m2));
  HIPCK(hipMalloc(&s->bm1, m2 * ntru));
  HIPCK(hipMalloc(&s->nindex, sizeof(int) * s->nsp));
  HIPCK(hipMalloc(&s->status, sizeof(int)));
  HIPCK(hipMemcpy(s->t0, t0, sizeof(double) * nlev, hipMemcpyHostToDevice));
  HIPCK(hipMemcpy(s->dsigma, dsigma, sizeof(double) * nlev, hipMemcpyHostToDevice));
  HIPCK(hipMemcpy(s->g, g, m2, hipMemcpyHostToDevice));
  HIPCK(hipMemcpy(s->tau, tau, m2, hipMemcpyHostToDevice));
  // total wavenumber of each spectral real (src/plasim.f90:1640-1646)
  int* ni = new int[s->nsp];
  for (int m = 0, jr = 0; m <= ntru; ++m)
    for (int n = m; n <= ntru; ++n, jr += 2) ni[jr] = ni[jr + 1] = n;
  hipError_t e = hipMemcpy(s->nindex, ni, sizeof(int) * s->nsp, hipMemcpyHostToDevice);
  delete[] ni;
  if (e != hipSuccess) return EXO_SI_ERR_HIP;
  *si = s;
  return EXO_SI_OK;
}

extern "C" int exo_si_destroy(exo_si_t s) {
  if (!s) return EXO_SI_ERR_ARG;
  void* ps[] = {s->t0, s->dsigma, s->g, s->tau, s->bm1, s->nindex, s->status};
  for (void* p : ps)
    if (p) (void)hipFree(p);
  delete s;
  return EXO_SI_OK;
}

extern "C" int exo_si_makebm(exo_si_t s, double delt, void* stream) {
  if (!s) return EXO_SI_ERR_ARG;
  hipStream_t st = (hipStream_t)stream;
  HIPCK(hipMemsetAsync(s->status, 0, sizeof(int), st));
  k_makebm<<<s->ntru, 64, 0, st>>>(s->nlev, s->ntru, delt, s->t0, s->dsigma, s->g, s->tau,
                                   s->bm1, s->status);
  HIPCK(hipGetLastError());
  int h = 0;
  HIPCK(hipMemcpyAsync(&h, s->status, sizeof(int), hipMemcpyDeviceToHost, st));
  HIPCK(hipStreamSynchronize(st));
  return h ? EXO_SI_ERR_SINGULAR : EXO_SI_OK;
}

extern "C" int exo_si_bm1(exo_si_t s, double* bm1) {
  if (!s || !bm1) return EXO_SI_ERR_ARG;
  HIPCK(hipMemcpy(bm1, s->bm1, sizeof(double) * s->nlev * s->nlev * s->ntru,
                  hipMemcpyDeviceToHost));
  return EXO_SI_OK;
}

template <typename R>
static int apply_t(exo_si_t s, double delt, const R* sop, const R* spm, const R* atm,
                   const R* adm, R* stt, R* sdt, R* spt, hipStream_t st) {
  k_si_apply<R><<<(s->nsp + SI_CB - 1) / SI_CB, SI_CB * SI_LB, 0, st>>>(
      s->nlev, s->nsp, s->nindex, delt, s->t0, s->dsigma, s->g, s->tau, s->bm1, sop, spm, atm,
      adm, stt, sdt, spt);
  return hipGetLastError() == hipSuccess ? EXO_SI_OK : EXO_SI_ERR_HIP;
}

extern "C" int exo_si_apply(exo_si_t s, int fp64, double delt, const void* sop, const void* spm,
                            const void* atm, const void* adm, void* stt, void* sdt, void* spt,
                            void* stream) {
  if (!s || !sop || !spm || !atm || !adm || !stt || !sdt || !spt) return EXO_SI_ERR_ARG;
  hipStream_t st = (hipStream_t)stream;
  if (fp64)
    return apply_t<double>(s, delt, (const double*)sop, (const double*)spm, (const double*)atm,
                           (const double*)adm, (double*)stt, (double*)sdt, (double*)spt, st);
  return apply_t<float>(s, delt, (const float*)sop, (const float*)spm, (const float*)atm,
                        (const float*)adm, (float*)stt, (float*)sdt, (float*)spt, st);
}
