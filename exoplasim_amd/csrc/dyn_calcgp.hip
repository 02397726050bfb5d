// dyn_calcgp.hip -- the grid-point dynamics of PlaSim between the inverse and
// the direct transforms, on the GPU (declared in include/exo_dyn.h):
//
//   k_calcgp  calcgp (src/plasim.f90:2587-2750): virtual temperatures,
//             vertical velocity (sigma-dot), the nonlinear tendencies gtn,
//             gqn, guz, gvz, the geopotential term gphi and dw; with it the
//             products of gridpointa (src/plasim.f90:2436-2446) and, on
//             request, gp = exp(gp) (:2434); in gridpointa also gp2fc of the
//             fields that go to the direct transforms
//   k_gpmt    the Fourier-space d/dlambda of ln(ps) (src/plasim.f90:2425-2430)
//
// calcgp is a column computation of pointwise terms, prefix sums over the
// levels and two matrix products over the levels (c and g).  A block takes 64
// grid points, or one latitude row in gridpointa, and all levels; its 4 to 10 waves
// share the levels, a lane owning the same points at each.  What a level needs
// of the others -- v . grad ln ps, the divergence and the humidity term --
// meets in LDS, and c and g are read through scalar loads (a wave's lanes all
// work on one level).  6 fields are read and 11 written per level.  On large
// calls the vector ALUs (65% busy at T42 L20, 32 members, FP32) and HBM (3.7 TB/s
// there) bound it together, on small ones the chain of a wave's levels.
//
// (One thread per column with its level arrays in registers held 202 VGPRs at
// L20 in FP32 and spilled at L40 in FP64; level counts without an
// instantiation of their own kept the arrays in scratch.  gridpointa of T42
// L20, 32 members, FP32: 336 us with it and the row FFT as a launch, 318 with
// this kernel on the grid, 273 with the rows transformed in it, and 239 -> 222 by a
// lane's points side by side and rows of half the length; T21 L10, one member,
// FP64: 49, 39.5, 37.5 us; T63 L20, 3 members, FP64: 294 and 253 us on the grid.)
#include "../../include/exo_dyn.h"
#include "sht_plan.h"

namespace exo {

template <typename R>
struct DynVert {
  const R *sigmah, *dsigma, *rdsig, *t0, *t01s2, *tkp, *c, *g;
  R akap, rdbrv, adv, psurf, ww;
};

template <typename R>
struct CalcgpPtrs {
  const R *gu, *gv, *gt, *gd, *gz, *gq, *dq;
  R* gp;
  const R *gpj, *gpm, *rcsq;
  R *gtn, *gqn, *guz, *gvz, *gphi, *dw, *gvp;
  R *gut, *gvt, *gke, *guq, *gvq;
};

// ROW = 0: calcgp on the grid, 64 points per block.  ROW = N (64, 128):
// gridpointa on rows of N longitudes, one row per block; the nine tendency fields of a
// level and gvp then leave as the Fourier coefficients of their rows (gp2fc):
// the wave that computed a level transforms it in LDS rows of its own,
// GpCfg::NFB rows at a time, so the grid values of those fields never reach
// HBM.  Each real row is one complex FFT of half its length, its even points
// the real and its odd points the imaginary parts: the rounding of a field is
// then that of its own row.  (Two fields of a level in one FFT of full length
// left the smaller one the rounding of the larger: the moisture tendency of
// levels with 1e-4 of the humidity 3 digits, and a NaN in it reached the
// temperature's.)
template <typename R, int ROW, int WAVES = 8>
struct GpCfg {
  static constexpr int PPL = ROW ? ROW / 64 : 1;  // points per lane
  static constexpr int P = 64 * PPL;              // points per block
  static constexpr int W = WAVES;                 // waves per block
  // rows at a time: all ten of a level, but four in FP64 on rows of 128, whose
  // ten would leave the level arrays too little LDS
  static constexpr int NFB = sizeof(R) == 4 || ROW <= 64 ? 10 : 4;
  static constexpr int H = ROW / 2, NP = H + H / 32;  // FFT length, padded FFT row
  static constexpr int R0 = H == 64 && NFB == 10 ? 16 : 8;  // first radix: fewest idle lanes
  // waves per SIMD asked for
  static constexpr int WPS = W > 8 ? 3 : (sizeof(R) == 4 || ROW <= 64) ? 4 : 2;
  static size_t lds(int nlev) {
    return sizeof(R) * 3 * nlev * P + (ROW ? sizeof(C2<R>) * (W * NFB * NP + ROW) : 0);
  }
};

// A wave-uniform vector of the vertical set-up, read through scalar loads
template <typename R>
using Uni = __attribute__((address_space(4))) const R*;

// With sid (gridpointa) rcsq = 1 / cos^2 comes from the Gaussian abscissas, as
// the model sets it up (src/plasim.f90:1897 csq = 1 - sid^2 in the real kind,
// :205), and is written to rcsq_out; else it is read.
template <typename R, int ROW, int WAVES>
__global__ __launch_bounds__(64 * WAVES, (GpCfg<R, ROW, WAVES>::WPS)) void k_calcgp(CalcgpPtrs<R> f, DynVert<R> v, int n, int nhor,
                                                long mstride, int nqspec, int exp_gp,
                                                const double* sid, int nlon, R* rcsq_out,
                                                const C2<R>* tw) {
  using C = GpCfg<R, ROW, WAVES>;
  using R2 = R __attribute__((ext_vector_type(2)));
  constexpr int PPL = C::PPL, P = C::P, W = C::W;
  extern __shared__ __align__(16) char smem[];
  R2* zg = (R2*)smem;          // [level][point]: (zvgpg, gd)
  R* cr = (R*)(zg + n * P);    // [level][point]: humidity term of the virtual temperature
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // where a lane's points lie in a level of zg and cr: side by side, but a wave
  // apart where 32 bytes per lane would put two lanes on each LDS bank
  const int l0 = PPL > 1 && sizeof(R) == 4 ? PPL * lane : lane;
  constexpr int LS = PPL > 1 && sizeof(R) == 4 ? 1 : 64;
  // Every field is addressed by a wave-uniform base (member, level, block) and
  // the lane's PPL consecutive points within the block, so that the address
  // arithmetic is scalar.  The lanes past the last point repeat it and store
  // nothing.
  const int h0 = blockIdx.x * P;
  const long mo = (long)blockIdx.y * mstride + h0;
  unsigned pt = lane;
  bool live = true;
  if constexpr (ROW == 0) {
    live = h0 + lane < nhor;
    if (!live) pt = nhor - 1 - h0;
  }
  struct V {
    R v[PPL];
  } __attribute__((packed, aligned(sizeof(R))));
  auto at = [&](const R* p, int j, R (&x)[PPL]) {
    const V u = ((const V*)(p + (mo + (long)j * nhor)))[pt];
#pragma unroll
    for (int i = 0; i < PPL; ++i) x[i] = u.v[i];
  };
  auto put = [&](R* p, int j, const R (&x)[PPL]) {
    V u;
#pragma unroll
    for (int i = 0; i < PPL; ++i) u.v[i] = x[i];
    if (live) ((V*)(p + (mo + (long)j * nhor)))[pt] = u;
  };
  const Uni<R> dsig = (Uni<R>)v.dsigma, sigh = (Uni<R>)v.sigmah, rdsig = (Uni<R>)v.rdsig;
  const Uni<R> t0v = (Uni<R>)v.t0, t01 = (Uni<R>)v.t01s2, tkp = (Uni<R>)v.tkp;
  const R qfac = R(1) / v.rdbrv - R(1);

  // ---- surface fields ----
  R gpm[PPL], gpj[PPL], rcsq[PPL], gp[PPL];
  at(f.gpm, 0, gpm);
  at(f.gpj, 0, gpj);
  at(f.gp, 0, gp);
  if (!sid) at(f.rcsq, 0, rcsq);
#pragma unroll
  for (int i = 0; i < PPL; ++i) {
    if (sid) {
      const double x = sid[(h0 + PPL * (int)pt + i) / nlon];
      rcsq[i] = R(1) / (R)(1.0 - x * x);
    }
    if (exp_gp) gp[i] = exp(gp[i]);
  }
  if constexpr (ROW > 0) {
    C2<R>* tws = (C2<R>*)(cr + n * P) + W * C::NFB * C::NP;
    for (int k = threadIdx.x; k < ROW; k += 64 * W) tws[k] = C2<R>{tw[k].x, -tw[k].y};
  }

  // ---- zvgpg = rcsq (u d/dlambda + v d/dmu) ln ps, the divergence, and the
  // virtual temperature's humidity term.  The reference forms (gt + t0)(1 +
  // (1/rdbrv - 1) zq) - t0 and then subtracts gt again for gphi
  // (src/plasim.f90:2617-2622, 2742): t0 is large against the humidity term,
  // and the subtractions cancel it.  The same quantities in the form without
  // the cancellation: corr = (gt + t0)(1/rdbrv - 1) zq, ztv1 = gt + corr, ztv1
  // - gt = corr and ztv2 = (gt + corr - t0 adv zq) / (1 + adv zq). ----
  for (int j = w; j < n; j += W) {
    R gu[PPL], gv[PPL], gd[PPL], gt[PPL], zq[PPL];
    at(f.gu, j, gu), at(f.gv, j, gv), at(f.gd, j, gd), at(f.gt, j, gt);
    at(nqspec == 1 ? f.gq : f.dq, j, zq);
#pragma unroll
    for (int i = 0; i < PPL; ++i) {
      if (nqspec == 1) zq[i] = zq[i] / gp[i];
      zq[i] = zq[i] > R(0) ? zq[i] : R(0);
      zg[j * P + l0 + LS * i] = R2{rcsq[i] * (gu[i] * gpm[i] + gv[i] * gpj[i]), gd[i]};
      cr[j * P + l0 + LS * i] = (gt[i] + t0v[j]) * (qfac * zq[i]);
    }
  }
  __syncthreads();
  if (w == 0) {  // (after the barrier: every wave has read gp)
    if (exp_gp) put(f.gp, 0, gp);
    if (sid) put(rcsq_out, 0, rcsq);
  }

  // ---- this wave's levels [j0, j1) ----
  const int j0 = w * (n / W) + (w < n % W ? w : n % W);
  const int j1 = j0 + n / W + (w < n % W ? 1 : 0);
  if (j0 >= j1) return;  // no barrier follows
  // the sums of the sigma-dot integral in the reference's order: over all
  // levels (zsumd, vp), and over the levels above j0 (rz, rv)
  R tot[PPL], vp[PPL], rz[PPL], rv[PPL];
#pragma unroll
  for (int i = 0; i < PPL; ++i) tot[i] = vp[i] = rz[i] = rv[i] = R(0);
#pragma unroll 4
  for (int k = 0; k < n; ++k) {
    const R dk = dsig[k];
#pragma unroll
    for (int i = 0; i < PPL; ++i) {
      if (k == j0) rz[i] = tot[i], rv[i] = vp[i];
      const R2 x = zg[k * P + l0 + LS * i];
      tot[i] = tot[i] + dk * x.y;
      vp[i] = vp[i] + dk * x.x;
    }
  }
#pragma unroll
  for (int i = 0; i < PPL; ++i) tot[i] = tot[i] + vp[i];
  if (ROW == 0 && w == 0) put(f.gvp, 0, vp);
  // the terms at the interface above level j (gtd, gqm, gud, gvd of level
  // j - 1, and tim = t01s2 (sigmah gvp - the sum of zvgpg dsigma)), carried one
  // level on; zero above the top and below the bottom
  R gt[PPL], gq[PPL], gu[PPL], gv[PPL];
  R gtd_m[PPL], gqm_m[PPL], gud_m[PPL], gvd_m[PPL], tim[PPL];
  {
    const int jm = j0 > 0 ? j0 - 1 : 0;
    R gtm[PPL], gqm[PPL], gum[PPL], gvm[PPL];
    at(f.gt, j0, gt), at(f.gq, j0, gq), at(f.gu, j0, gu), at(f.gv, j0, gv);
    at(f.gt, jm, gtm), at(f.gq, jm, gqm), at(f.gu, jm, gum), at(f.gv, jm, gvm);
#pragma unroll
    for (int i = 0; i < PPL; ++i) {
      const R zsdotp = sigh[jm] * tot[i] - (rz[i] + rv[i]);
      const R a = zsdotp * (gt[i] - gtm[i]), b = zsdotp * (gq[i] + gqm[i]);
      const R c = zsdotp * (gu[i] - gum[i]), d = zsdotp * (gv[i] - gvm[i]);
      const R e = t01[jm] * (sigh[jm] * vp[i] - rv[i]);
      gtd_m[i] = j0 > 0 ? a : R(0), gqm_m[i] = j0 > 0 ? b : R(0);
      gud_m[i] = j0 > 0 ? c : R(0), gvd_m[i] = j0 > 0 ? d : R(0);
      tim[i] = j0 > 0 ? e : R(0);
    }
  }
  C2<R>* fb = (C2<R>*)(cr + n * P) + w * C::NFB * C::NP;  // this wave's FFT rows
  struct V2 {
    R v[2];
  } __attribute__((packed, aligned(sizeof(R))));
  for (int j = j0; j < j1; ++j) {
    const bool top = j == 0, bottom = j == n - 1;
    // this level's inputs first, so that they arrive during the sums below
    const int jp = bottom ? j : j + 1;
    R gz[PPL], gt1[PPL], gq1[PPL], gu1[PPL], gv1[PPL], dq[PPL];
    at(f.gz, j, gz), at(f.gt, jp, gt1), at(f.gq, jp, gq1), at(f.gu, jp, gu1), at(f.gv, jp, gv1);
    if (nqspec != 1) at(f.dq, j, dq);
    // c(k, j) for k <= j: column j of c; ztptb = ztpta + the same sum over the
    // divergence
    R ztpta[PPL], ztptb[PPL], gphi[PPL];
#pragma unroll
    for (int i = 0; i < PPL; ++i) ztpta[i] = ztptb[i] = gphi[i] = R(0);
    const Uni<R> cj = (Uni<R>)v.c + j * n, gj = (Uni<R>)v.g + j * n;
#pragma unroll 4
    for (int k = 0; k <= j; ++k) {
      const R ck = cj[k];
#pragma unroll
      for (int i = 0; i < PPL; ++i) {
        const R2 x = zg[k * P + l0 + LS * i];
        ztpta[i] = ztpta[i] + ck * x.x;
        ztptb[i] = ztptb[i] + ck * x.y;
      }
    }
    // gphi(j) = 2 / rcsq * sum_k g(k, j) (ztv1 - gt)(k)
#pragma unroll 4
    for (int k = 0; k < n; ++k) {
      const R gk = gj[k];
#pragma unroll
      for (int i = 0; i < PPL; ++i) gphi[i] = gphi[i] + gk * cr[k * P + l0 + LS * i];
    }
    R out[10][PPL];  // gtn gqn guz gvz gut gvt guq gvq gke, and gvp at the top
    R dw[PPL];
    const R rd = rdsig[j], dsj = bottom ? R(0) : dsig[j], shj = sigh[j], t01j = t01[j];
#pragma unroll
    for (int i = 0; i < PPL; ++i) {
      const R2 x = zg[j * P + l0 + LS * i];
      const R zv = x.x, gd = x.y, corr = cr[j * P + l0 + LS * i];
      R zq = (nqspec == 1) ? gq[i] / gp[i] : dq[i];
      zq = zq > R(0) ? zq : R(0);
      ztptb[i] = ztpta[i] + ztptb[i];
      const R ztv1 = gt[i] + corr;
      const R ztv2 = (gt[i] + corr - t0v[j] * (v.adv * zq)) / (R(1) + v.adv * zq);
      gphi[i] = gphi[i] * R(2) / rcsq[i];
      // (sigma-dot times the differences across the interface below j)
      rz[i] = rz[i] + dsj * gd;
      rv[i] = rv[i] + dsj * zv;
      const R zsdotp = shj * tot[i] - (rz[i] + rv[i]);
      const R gtd = bottom ? R(0) : zsdotp * (gt1[i] - gt[i]);
      const R gqm = bottom ? R(0) : zsdotp * (gq1[i] + gq[i]);
      const R gud = bottom ? R(0) : zsdotp * (gu1[i] - gu[i]);
      const R gvd = bottom ? R(0) : zsdotp * (gv1[i] - gv[i]);
      const R ti = bottom ? R(0) : t01j * (shj * vp[i] - rv[i]);
      const R za = top ? -gd : zv - ztptb[i], zt = top ? R(0) : tkp[j] * (zv - ztpta[i]);
      dw[i] = (top ? gd : za) * gp[i] * v.psurf * v.ww;
      out[0][i] = gt[i] * gd + v.akap * ztv2 * za + zt - rd * (gtd + gtd_m[i] + ti + tim[i]);
      out[1][i] = -rd * (gqm - gqm_m[i]);
      out[2][i] = -gu[i] * gz[i] - gpj[i] * ztv1 - rd * (gvd + gvd_m[i]);
      out[3][i] = gv[i] * gz[i] - gpm[i] * ztv1 - rd * (gud + gud_m[i]);
      out[4][i] = gu[i] * gt[i];
      out[5][i] = gv[i] * gt[i];
      out[6][i] = gu[i] * gq[i];
      out[7][i] = gv[i] * gq[i];
      out[8][i] = gu[i] * gu[i] + gv[i] * gv[i] + gphi[i];
      out[9][i] = top ? vp[i] : R(0);
      gtd_m[i] = gtd, gqm_m[i] = gqm, gud_m[i] = gud, gvd_m[i] = gvd, tim[i] = ti;
      gt[i] = gt1[i], gq[i] = gq1[i], gu[i] = gu1[i], gv[i] = gv1[i];
    }
    put(f.dw, j, dw);
    put(f.gphi, j, gphi);
    R* const dst[10] = {f.gtn, f.gqn, f.guz, f.gvz, f.gut, f.gvt, f.guq, f.gvq, f.gke, f.gvp};
    if constexpr (ROW == 0) {
#pragma unroll
      for (int q = 0; q < 9; ++q)
        if (dst[q] && (q < 6 || q > 7 || nqspec == 1)) put(dst[q], j, out[q]);
    } else {
      // gp2fc: Z = FFT(x[2k] + i x[2k + 1]) of half the length holds the sums E
      // over the even and O over the odd points, E = (Z[k] + conj Z[H - k]) / 2,
      // O = (Z[k] - conj Z[H - k]) / 2i, and with w = e^{-2 pi i k / N} X[k] = E +
      // w O, X[H - k] = conj(E - w O); X[0] = Re Z[0] + Im Z[0], X[H / 2] = conj
      // Z[H / 2].  RPI rows side by side in a wave.
      constexpr int NFB = C::NFB, NP = C::NP, N = ROW, H = C::H, RPI = 128 / H;
      const C2<R>* tws = (const C2<R>*)(cr + n * P) + W * NFB * NP;
      const R sc = R(0.5) / R(N);
      const int k = lane % (H / 2), kn = k ? H - k : H / 2, sub = lane / (H / 2);
#pragma unroll
      for (int q0 = 0; q0 < 10; q0 += NFB) {
#pragma unroll
        for (int q = q0; q < q0 + NFB && q < 10; ++q) {
          C2<R>* row = fb + (q - q0) * NP;
          if constexpr (PPL == 2)
            row[wix<C::H, R>(lane)] = C2<R>{out[q][0], out[q][PPL - 1]};
          else
            ((R*)(row + wix<C::H, R>(lane >> 1)))[lane & 1] = out[q][0];
        }
        if (q0 + NFB <= 10)
          fft_wave_rows<H, C::R0, NFB, -1, 2>(fb, tws, lane);
        else
          fft_wave_rows<H, C::R0, (10 % NFB ? 10 % NFB : 1), -1, 2>(fb, tws, lane);
#pragma unroll
        for (int q = q0; q < q0 + NFB && q < 10; q += RPI) {
          const int r = q + sub;
          R* d = dst[q];
#pragma unroll
          for (int u = 1; u < RPI; ++u) {
            R* const du = dst[q + u < 10 ? q + u : 9];
            d = sub == u ? du : d;
          }
          if (r >= q0 + NFB || r > 9 || (r == 9 && !top) || (r / 2 == 3 && nqspec != 1)) continue;
          const C2<R>* row = fb + (r - q0) * NP;
          const C2<R> zk = row[wix<C::H, R>(k)], zn = row[wix<C::H, R>(kn)];
          const R ex = zk.x + zn.x, ey = zk.y - zn.y;
          const C2<R> t = cmul(tws[k], C2<R>{zk.x - zn.x, zk.y + zn.y});
          V2* o = (V2*)(d + (mo + (long)j * nhor));
          o[k] = V2{{(k ? ex + t.y : R(2) * (zk.x + zk.y)) * sc, (k ? ey - t.x : R(0)) * sc}};
          o[kn] = V2{{(k ? ex - t.y : R(2) * zn.x) * sc, (k ? -(ey + t.x) : R(-2) * zn.y) * sc}};
        }
        wave_lds_sync();  // the rows are read before the next ones are written
      }
    }
  }
}

// Fourier-space d/dlambda: one complex coefficient (m) per thread
template <typename R>
__global__ void k_gpmt(const R* in, R* out, int nlon, long total) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i >= total) return;
  const int m = (int)(i % (nlon / 2));
  const R re = in[2 * i], im = in[2 * i + 1];
  out[2 * i] = -im * (R)m;
  out[2 * i + 1] = re * (R)m;
}

}  // namespace exo

using namespace exo;

struct exo_dyn_s {
  int nlev = 0;
  double* d64 = nullptr;  // sigmah dsigma rdsig t0 t01s2 tkp (nlev each), c, g (nlev^2 each)
  float* d32 = nullptr;
  double sc[5] = {0, 0, 0, 0, 0};  // akap rdbrv adv psurf ww
};

template <typename R>
static DynVert<R> vert_of(const exo_dyn_s* d) {
  const int n = d->nlev;
  const R* b;
  if constexpr (sizeof(R) == 8)
    b = d->d64;
  else
    b = d->d32;
  DynVert<R> v;
  v.sigmah = b;
  v.dsigma = b + n;
  v.rdsig = b + 2 * n;
  v.t0 = b + 3 * n;
  v.t01s2 = b + 4 * n;
  v.tkp = b + 5 * n;
  v.c = b + 6 * n;
  v.g = b + 6 * n + n * n;
  v.akap = (R)d->sc[0];
  v.rdbrv = (R)d->sc[1];
  v.adv = (R)d->sc[2];
  v.psurf = (R)d->sc[3];
  v.ww = (R)d->sc[4];
  return v;
}

extern "C" int exo_dyn_create(exo_dyn_t* dyn, int nlev, const double* sigmah,
                              const double* dsigma, const double* rdsig, const double* t0,
                              const double* t01s2, const double* tkp, const double* c,
                              const double* g, double akap, double rdbrv, double adv,
                              double psurf, double ww) {
  if (!dyn) return EXO_ERR_ARG;
  *dyn = nullptr;
  if (nlev < 2 || nlev > 64 || !sigmah || !dsigma || !rdsig || !t0 || !t01s2 || !tkp || !c ||
      !g)
    return EXO_ERR_ARG;
  exo_dyn_s* d = new exo_dyn_s();
  d->nlev = nlev;
  d->sc[0] = akap;
  d->sc[1] = rdbrv;
  d->sc[2] = adv;
  d->sc[3] = psurf;
  d->sc[4] = ww;
  const int tot = 6 * nlev + 2 * nlev * nlev;
  double* host = new double[tot];
  const double* parts[6] = {sigmah, dsigma, rdsig, t0, t01s2, tkp};
  for (int k = 0; k < 6; ++k)
    for (int i = 0; i < nlev; ++i) host[k * nlev + i] = parts[k][i];
  for (int i = 0; i < nlev * nlev; ++i) {
    host[6 * nlev + i] = c[i];
    host[6 * nlev + nlev * nlev + i] = g[i];
  }
  float* host32 = new float[tot];
  for (int i = 0; i < tot; ++i) host32[i] = (float)host[i];
  int rc = EXO_OK;
  if (hipMalloc(&d->d64, sizeof(double) * tot) != hipSuccess ||
      hipMalloc(&d->d32, sizeof(float) * tot) != hipSuccess ||
      hipMemcpy(d->d64, host, sizeof(double) * tot, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(d->d32, host32, sizeof(float) * tot, hipMemcpyHostToDevice) != hipSuccess)
    rc = EXO_ERR_HIP;
  delete[] host;
  delete[] host32;
  if (rc != EXO_OK) {
    exo_dyn_destroy(d);
    return rc;
  }
  *dyn = d;
  return EXO_OK;
}

extern "C" int exo_dyn_destroy(exo_dyn_t d) {
  if (!d) return EXO_ERR_ARG;
  (void)hipDeviceSynchronize();
  if (d->d64) (void)hipFree(d->d64);
  if (d->d32) (void)hipFree(d->d32);
  delete d;
  return EXO_OK;
}

template <typename R>
static int calcgp_t(exo_dyn_t d, int nmem, long ms, int nhor, int nqspec, int exp_gp,
                    const exo_calcgp_fields* f, hipStream_t s, const double* sid = nullptr,
                    int nlon = 1, void* rcsq_out = nullptr, const void* tw = nullptr,
                    bool in_place = false) {
  CalcgpPtrs<R> p;
  p.gu = (const R*)f->gu;
  p.gv = (const R*)f->gv;
  p.gt = (const R*)f->gt;
  p.gd = (const R*)f->gd;
  p.gz = (const R*)f->gz;
  p.gq = (const R*)f->gq;
  p.dq = (const R*)f->dq;
  p.gp = (R*)f->gp;
  p.gpj = (const R*)f->gpj;
  p.gpm = (const R*)f->gpm;
  p.rcsq = (const R*)f->rcsq;
  p.gtn = (R*)f->gtn;
  p.gqn = (R*)f->gqn;
  p.guz = (R*)f->guz;
  p.gvz = (R*)f->gvz;
  p.gphi = (R*)f->gphi;
  p.dw = (R*)f->dw;
  p.gvp = (R*)f->gvp;
  p.gut = (R*)f->gut;
  p.gvt = (R*)f->gvt;
  p.gke = (R*)f->gke;
  p.guq = (R*)f->guq;
  p.gvq = (R*)f->gvq;
  const DynVert<R> v = vert_of<R>(d);
  auto launch = [&](auto kern, int points, int waves, size_t lds) -> int {
    if (lds > 65536 &&
        hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)lds) != hipSuccess)
      return EXO_ERR_LAUNCH;
    const dim3 grid((unsigned)((nhor + points - 1) / points), (unsigned)nmem);
    kern<<<grid, 64 * waves, lds, s>>>(p, v, d->nlev, nhor, ms, nqspec, exp_gp, sid, nlon, (R*)rcsq_out,
                                (const C2<R>*)tw);
    return hipGetLastError() == hipSuccess ? EXO_OK : EXO_ERR_LAUNCH;
  };
  const int n = d->nlev;
  // Waves per block of a row kernel.  Up to one block per CU its own chain of
  // levels is the time, and 10 waves shorten it (gridpointa, 10 against 8 and 4
  // waves: T21 L10 FP64, one member, 26.6, 26.9, 29.4 us; T42 L10 FP32 38.3, 39.4,
  // 42.1), but in FP64 on rows of 128, whose registers do not allow it (T42 L10
  // 54.3, 46.7, 50.7).  Above, FP64 takes 4, two of whose blocks fit a CU's LDS (8
  // against 4: T42 L20, 8 members, 126.3, 119.7; T21 L10, 32 members, 68.5, 65.4;
  // from L20 on 8 would do better at T21: 103, 111), FP32 8 (T42 L20, 32 members,
  // 10, 8 and 4: 278.7, 247.9, 255.7).
  const bool few = (long)(nhor / (nlon > 0 ? nlon : 1)) * nmem <= 256;
  switch (tw ? nlon : 0) {
    case 64:
      if (few) return launch(k_calcgp<R, 64, 10>, 64, 10, GpCfg<R, 64, 10>::lds(n));
      if constexpr (sizeof(R) == 8)
        return launch(k_calcgp<R, 64, 4>, 64, 4, GpCfg<R, 64, 4>::lds(n));
      else
        return launch(k_calcgp<R, 64, 8>, 64, 8, GpCfg<R, 64>::lds(n));
    case 128:
      if constexpr (sizeof(R) == 4) {
        if (few) return launch(k_calcgp<R, 128, 10>, 128, 10, GpCfg<R, 128, 10>::lds(n));
      } else {
        if (!few) return launch(k_calcgp<R, 128, 4>, 128, 4, GpCfg<R, 128, 4>::lds(n));
      }
      return launch(k_calcgp<R, 128, 8>, 128, 8, GpCfg<R, 128>::lds(n));
    default:
      // An output in the place of an input: a wave reads its neighbours' levels
      // next to its own, so one wave takes them all, which has read a level and
      // the next one before it writes the first.
      if (in_place) return launch(k_calcgp<R, 0, 1>, 64, 1, GpCfg<R, 0, 1>::lds(n));
      // Few levels on many points: with 8 waves each has one or two levels to
      // pay for its sums over all of them (L10, 294912 points, FP64 131 us against
      // 116 with 4 waves, FP32 48 against 41; 73728 points 24.9 and 24.8, 16.3 and
      // 14.5; 18432 points 10.5 and 10.9; L20, 147456 points, FP32 43.9 and 45.1).
      if (n <= 16 && ((nhor + 63L) / 64) * nmem > 1024)
        return launch(k_calcgp<R, 0, 4>, 64, 4, GpCfg<R, 0, 4>::lds(n));
      return launch(k_calcgp<R, 0, 8>, 64, 8, GpCfg<R, 0>::lds(n));
  }
}

// Does an output of a member overlap an input that is read level by level?
static bool calcgp_in_place(const exo_calcgp_fields* f, size_t bytes) {
  const void* in[] = {f->gu, f->gv, f->gt, f->gq, f->gz, f->dq};
  const void* out[] = {f->gtn, f->gqn, f->guz, f->gvz, f->gphi, f->dw,
                       f->gut, f->gvt, f->gke, f->guq, f->gvq};
  for (const void* i : in)
    for (const void* o : out)
      if (i && o && (uintptr_t)i < (uintptr_t)o + bytes && (uintptr_t)o < (uintptr_t)i + bytes)
        return true;
  return false;
}

// Does gridpointa's calcgp transform its rows itself?  On rows of 64 and 128
// whose level arrays fit a CU's LDS (all levels but FP64 above L41 on 128).
// Three points per lane on rows of 192 spilled (T63 L20, 16 members, FP32: 479 us
// against 390 with calcgp on the grid and the row FFT as a launch; FP64, 3
// members: 289 against 253).
constexpr size_t GP_LDS = 160 * 1024;
static bool calcgp_rows(int mode, int nlon, int nlev) {
  const bool d = mode == MODE_F64;
  switch (nlon) {
    case 64: return (d ? GpCfg<double, 64>::lds(nlev) : GpCfg<float, 64>::lds(nlev)) <= GP_LDS;
    case 128: return (d ? GpCfg<double, 128>::lds(nlev) : GpCfg<float, 128>::lds(nlev)) <= GP_LDS;
    default: return false;
  }
}

extern "C" int exo_dyn_calcgp(exo_dyn_t d, int mode, int nmem, long member_stride, int nhor,
                              int nqspec, int exp_gp, const exo_calcgp_fields* f,
                              void* stream) {
  if (!d || !f || mode < EXO_F64 || mode > EXO_BF16X3 || nmem < 0 || nhor < 0 ||
      (nqspec != 0 && nqspec != 1))
    return EXO_ERR_ARG;
  if (nmem == 0 || nhor == 0) return EXO_OK;
  if (nmem > 1 && member_stride <= 0) return EXO_ERR_ARG;
  const void* need[] = {f->gu, f->gv, f->gt, f->gd, f->gz, f->gq, f->gp, f->gpj, f->gpm,
                        f->rcsq, f->gtn, f->gqn, f->guz, f->gvz, f->gphi, f->dw, f->gvp};
  for (const void* q : need)
    if (!q) return EXO_ERR_ARG;
  if (nqspec == 0 && !f->dq) return EXO_ERR_ARG;
  hipStream_t s = (hipStream_t)stream;
  const size_t es = mode == EXO_F64 ? 8 : 4;
  const bool in_place = calcgp_in_place(f, es * d->nlev * nhor);
  return mode == EXO_F64 ? calcgp_t<double>(d, nmem, member_stride, nhor, nqspec, exp_gp, f, s,
                                            nullptr, 1, nullptr, nullptr, in_place)
                         : calcgp_t<float>(d, nmem, member_stride, nhor, nqspec, exp_gp, f, s,
                                           nullptr, 1, nullptr, nullptr, in_place);
}

extern "C" int exo_dyn_gpmt(int mode, int nlon, long nrow, const void* in, void* out,
                            void* stream) {
  if (mode < EXO_F64 || mode > EXO_BF16X3 || nlon < 2 || (nlon & 1) || nrow < 0 ||
      (nrow > 0 && (!in || !out)))
    return EXO_ERR_ARG;
  const long total = nrow * (nlon / 2);
  if (total == 0) return EXO_OK;
  const unsigned nb = (unsigned)((total + 255) / 256);
  hipStream_t s = (hipStream_t)stream;
  if (mode == EXO_F64)
    k_gpmt<double><<<nb, 256, 0, s>>>((const double*)in, (double*)out, nlon, total);
  else
    k_gpmt<float><<<nb, 256, 0, s>>>((const float*)in, (float*)out, nlon, total);
  return hipGetLastError() == hipSuccess ? EXO_OK : EXO_ERR_LAUNCH;
}

// ---------------------------------------------------------------------------
// the device-resident gridpointa transform group
// ---------------------------------------------------------------------------
// work slots (units of NHOR values) of one member
namespace {
struct GpaSlots {
  int gz, gd, gt, gq, gp, gpj, gpm, gu, gv, dq, rcsq;
  int a;  // first FFT slot: gtn gqn guz gvz gut gvt gke guq gvq (nlev each), gvp
  int gtn, gqn, guz, gvz, gut, gvt, gke, guq, gvq, gvp, gphi, dw, total;
  explicit GpaSlots(int n) {
    gz = 0, gd = n, gt = 2 * n, gq = 3 * n, gp = 4 * n, gpj = 4 * n + 1, gpm = 4 * n + 2;
    gu = 4 * n + 3, gv = 5 * n + 3, dq = 6 * n + 3, rcsq = 7 * n + 3;
    a = 7 * n + 4;
    gtn = a, gqn = a + n, guz = a + 2 * n, gvz = a + 3 * n, gut = a + 4 * n, gvt = a + 5 * n;
    gke = a + 6 * n, guq = a + 7 * n, gvq = a + 8 * n, gvp = a + 9 * n;
    gphi = a + 9 * n + 1, dw = a + 10 * n + 1, total = a + 11 * n + 1;
  }
};
}  // namespace

extern "C" int exo_gridpointa_fields(int nlev) {
  return nlev < 2 ? EXO_ERR_ARG : GpaSlots(nlev).total;
}

extern "C" int exo_gridpointa(exo_sht_plan_t p, exo_dyn_t d, int mode, int nmem, int nqspec,
                              const void* sp_state, long sp_stride, void* work, long work_stride,
                              void* sp_tend, long tend_stride, void* stream) {
  if (!p || !d || mode < EXO_F64 || mode > EXO_BF16X3 || nmem < 0 ||
      (nqspec != 0 && nqspec != 1))
    return EXO_ERR_ARG;
  if (nmem == 0) return EXO_OK;
  const Tables& tb = p->tb;
  const int n = d->nlev, nsp = 4 * n + 1;
  const long nhor = (long)tb.nlat * tb.nlon;
  const GpaSlots sl(n);
  if (!sp_state || !work || !sp_tend || sp_stride < (long)nsp * 2 * tb.ncsp ||
      tend_stride < (long)nsp * 2 * tb.ncsp || work_stride < (long)sl.total * nhor)
    return EXO_ERR_ARG;
  std::lock_guard<std::mutex> lk(p->mu);
  hipStream_t s = (hipStream_t)stream;
  const size_t es = (mode == MODE_F64) ? 8 : 4;
  char* wk = (char*)work;
  auto slot = [&](int k) { return (void*)(wk + es * nhor * k); };

  // invlega (src/legmod.f90:635-656) fused with fc2gp, and gpmt
  InvArgs base{};
  base.sp = sp_state;
  base.out = work;
  base.sp_stride = sp_stride;
  base.out_stride = work_stride;
  base.nmem = nmem;
  base.plavor = tb.plavor;
  base.var = p->inv_var[mode];
  if (mode == MODE_BF16X3) {
    const int rc = plan_grow(&p->pk, &p->pk_bytes, pack_bytes(tb, nmem, nsp));
    if (rc) return rc;
    if (launch_pack(tb, (const float*)sp_state, sp_stride, 0, nsp, nmem, (float*)p->pk, s))
      return EXO_ERR_LAUNCH;
    base.bpk = p->pk;
    base.bpk_stride = (long)nsp * pk_field(tb.ntru);
    base.bpk_f0 = 0;
  }
  auto scalar = [&](int table, int src0, int dst0, int nfield, int dlam) {
    InvArgs a = base;
    a.kind = INV_SCALAR;
    a.table = table;
    a.src0 = src0;
    a.dst0 = dst0;
    a.nfield = nfield;
    a.dlam = dlam;
    return a;
  };
  // sz sd st (sq, sp) -> gz gd gt (gq, gp); with nqspec = 0 gq is the caller's
  const InvArgs wide = scalar(TQI, 0, sl.gz, nqspec ? nsp : 3 * n, 0);
  const InvArgs one[3] = {scalar(TQJ, 4 * n, sl.gpj, 1, 0), scalar(TQI, 4 * n, sl.gpm, 1, 1),
                          scalar(TQI, 4 * n, sl.gp, 1, 0)};
  InvArgs uv = base;
  uv.kind = INV_UV;
  uv.vor0 = 0;
  uv.div0 = n;
  uv.u0 = sl.gu;
  uv.v0 = sl.gv;
  uv.nlev = n;
  if (launch_inverse_rt(tb, mode, wide, one, nqspec ? 2 : 3, uv, s)) return EXO_ERR_LAUNCH;

  // gp = exp(gp), calcgp and the products (src/plasim.f90:2434-2446)
  exo_calcgp_fields f{};
  f.gu = slot(sl.gu);
  f.gv = slot(sl.gv);
  f.gt = slot(sl.gt);
  f.gd = slot(sl.gd);
  f.gz = slot(sl.gz);
  f.gq = slot(sl.gq);
  f.dq = slot(sl.dq);
  f.gp = slot(sl.gp);
  f.gpj = slot(sl.gpj);
  f.gpm = slot(sl.gpm);
  f.rcsq = slot(sl.rcsq);
  f.gtn = slot(sl.gtn);
  f.gqn = slot(sl.gqn);
  f.guz = slot(sl.guz);
  f.gvz = slot(sl.gvz);
  f.gphi = slot(sl.gphi);
  f.dw = slot(sl.dw);
  f.gvp = slot(sl.gvp);
  f.gut = slot(sl.gut);
  f.gvt = slot(sl.gvt);
  f.gke = slot(sl.gke);
  f.guq = nqspec ? slot(sl.guq) : nullptr;
  f.gvq = nqspec ? slot(sl.gvq) : nullptr;
  const bool rows = calcgp_rows(mode, tb.nlon, n);
  const void* tw = !rows ? nullptr : mode == MODE_F64 ? (const void*)tb.tw64 : (const void*)tb.tw32;
  int rc = mode == MODE_F64 ? calcgp_t<double>(d, nmem, work_stride, (int)nhor, nqspec, 1, &f, s,
                                               tb.sid, tb.nlon, slot(sl.rcsq), tw)
                            : calcgp_t<float>(d, nmem, work_stride, (int)nhor, nqspec, 1, &f, s,
                                              tb.sid, tb.nlon, slot(sl.rcsq), tw);
  if (rc) return rc;

  // gp2fc of the nine tendency fields and gvpp, in place, where calcgp has
  // not done it
  if (!rows && launch_fft(tb, mode, -1, slot(sl.a), tb.nlon, (long)(9 * n + 1) * tb.nlat, s, nmem,
                          work_stride))
    return EXO_ERR_LAUNCH;

  // mktend -> szt, sdt, stt; qtend -> sqt; fc2sp(gvpp) -> spt (src/plasim.f90:2473-2486)
  auto out = [&](int k) { return (void*)((char*)sp_tend + es * 2 * tb.ncsp * k); };
  const DirxArgs jobs[4] = {
      mktend_dz(slot(sl.gke), slot(sl.guz), slot(sl.gvz), out(n), out(0), n, nmem, work_stride,
                tend_stride),
      mktend_t(slot(sl.gvt), slot(sl.gtn), slot(sl.gut), out(2 * n), n, nmem, work_stride,
               tend_stride),
      fc2sp_job(slot(sl.gvp), out(4 * n), TQC, 1, nmem, work_stride, tend_stride),
      mktend_t(slot(sl.gvq), slot(sl.gqn), slot(sl.guq), out(3 * n), n, nmem, work_stride,
               tend_stride)};
  if (launch_dirx(tb, mode, jobs, nqspec ? 4 : 3, s)) return EXO_ERR_LAUNCH;
  return EXO_OK;
}
