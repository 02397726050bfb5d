// sht_transforms_impl.h -- the per-truncation transform kernels and their
// launchers for one precision mode.  Each sht_transforms_m<mode>.hip
// includes this file and instantiates one mode, so the four modes compile in
// parallel; sht_transforms.hip dispatches on the mode.
#pragma once
#include "sht_bodies.h"
#include "sht_launch.h"

namespace exo {

template <int T, int MODE, int KIND, bool FUSED, int V>
__global__ __launch_bounds__((InvCfg<T, MODE, V>::NT)) void k_inv(InvArgs a, const void* tabA0, const void* tabA1,
                                             const void* tabv, const void* twp) {
  __shared__ __align__(16) char lds[InvLds<T, MODE, FUSED, V>::BYTES];
  inv_body<T, MODE, KIND, FUSED, V>(a, xcd_block(blockIdx.x, gridDim.x), tabA0, tabA1, tabv,
                                    twp, lds);
}

// The inverse transforms of a round trip or of a dynamics step in one launch:
// per member, the sp2fc blocks (aq, table qi), the blocks of the one-field
// jobs (aj with the table, destination and d/dlambda switch of job k: a round
// trip's sp2fcdmu; a dynamics step's sp2fcdmu, d/dlambda and, without
// spectral humidity, ln ps) and the dv2uv blocks (au), each block the same
// work item as in its own kernel.  One launch instead of one per transform
// removes their ramp-up/drain tails, and the blocks of one member (which read
// the same spectral coefficients) run close together.  (gridpointa with one
// launch per transform: T21 L10 FP64, one member, 42 us of inverse launches
// against 15 us; T42 L20, 32 members, 107 us against 74 us.  All scalar jobs
// as an array of arguments picked by index made the T42 round trip of 128
// members 1.8% slower: every block then waits for one more scalar load
// before its arguments.)
template <int T, int MODE, int V>
__global__ __launch_bounds__((InvCfg<T, MODE, V>::NT)) void k_inv_rt(InvArgs aq, InvArgs aj, InvArgs au, const void* tq,
                                                InvOneJobs one, const void* tv0, const void* tu,
                                                const void* tabv, const void* twp,
                                                int gq, int gj, int gu) {
  __shared__ __align__(16) char lds[InvLds<T, MODE, true, V>::BYTES];
  constexpr int NPB = TS<T>::NPAIR / InvCfg<T, MODE, V>::LP;
  const int per = NPB * (gq + gj + gu);
  int mem, r;
  if (T == 127 && aq.nmem % 8 == 0) {
    // T127: workgroups go round-robin to the 8 XCDs, and XCD x =
    // blockIdx.x % 8 runs members x M .. x M + M - 1 (M = nmem / 8), first
    // all their dv2uv items, then all their scalar items: the round trip of
    // 8 members at L40 1% faster than the member-major order below (which
    // stays faster at T42, by about as much)
    const int x = blockIdx.x % 8, i = blockIdx.x / 8, M = aq.nmem / 8;
    const int nu = M * NPB * gu, ns = NPB * (gq + gj);
    if (i < nu) {
      mem = x * M + i / (NPB * gu);
      r = ns + i % (NPB * gu);
    } else {
      mem = x * M + (i - nu) / ns;
      r = (i - nu) % ns;
    }
  } else if (T == 127 && aq.nmem < 8) {
    // fewer members than XCDs: contiguous ranges of a member's blocks would give
    // some XCDs only dv2uv items (two terms), others only scalar ones.  The long
    // dv2uv items first, dealt out over all XCDs (round trips: FP64 L15, 2
    // members, 262 -> 242 us; BF16X3 L40, 3 members, 248 -> 237; gridpointa FP64
    // L10, one member, 232 -> 218.  At T63 and T42, whose launches last a few
    // rounds of blocks at most, the ranges' locality counts for more: T63 L30
    // FP64, 5 members, 159 against 165.)
    const int i = blockIdx.x, nu = NPB * gu, ns = NPB * (gq + gj);
    const bool uv = i < aq.nmem * nu;
    const int k = uv ? i : i - aq.nmem * nu, n = uv ? nu : ns;
    mem = k / n;
    r = k - mem * n + (uv ? ns : 0);
  } else {
    const int b = xcd_block(blockIdx.x, gridDim.x);
    mem = b / per;
    r = b - mem * per;
  }
  if (r < NPB * gq)
    inv_body<T, MODE, INV_SCALAR, true, V>(aq, mem * NPB * gq + r, tq, tu, tabv, twp, lds);
  else if (r < NPB * (gq + gj)) {
    const int k = __builtin_amdgcn_readfirstlane((r - NPB * gq) / NPB);
    aj.table = one.table[k];
    aj.dst0 = one.dst0[k];
    aj.dlam = one.dlam[k];
    inv_body<T, MODE, INV_SCALAR, true, V>(aj, mem * NPB + (r - NPB * (gq + k)), one.tab[k], tu,
                                           tabv, twp, lds);
  }
  else
    inv_body<T, MODE, INV_UV, true, V>(au, mem * NPB * gu + (r - NPB * (gq + gj)), tv0, tu,
                                       tabv, twp, lds);
}

template <int T, int MODE, bool FUSED, int V>
__global__ __launch_bounds__((FwdCfg<T, MODE, V>::NT)) void k_fwd(FwdArgs a, const void* tabv, const void* twp,
                                             void* scratch) {
  __shared__ __align__(16) char lds[FwdLds<T, MODE, FUSED, V>::BYTES];
  fwd_body<T, MODE, FUSED, V>(a, xcd_block(blockIdx.x, gridDim.x), tabv, twp, scratch, lds);
}

// sum of the per-pair-block partial direct transforms in a fixed order
template <typename R>
__global__ void k_reduce_partials(const R* scratch, R* sp, int npb, int nmem, int nfield,
                                  int nrsp, long sp_stride, int dst0) {
  const long total = (long)nmem * nfield * nrsp;
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i >= total) return;
  const int x = (int)(i % nrsp);
  const int f = (int)((i / nrsp) % nfield);
  const int mem = (int)(i / ((long)nrsp * nfield));
  R s = 0;
  for (int b = 0; b < npb; ++b) s += scratch[(long)b * total + i];
  sp[mem * sp_stride + (long)(dst0 + f) * nrsp + x] = s;
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
template <int T, int MODE, int V>
static int inv_tv(const Tables& tb, bool fused, const InvArgs& a, hipStream_t s) {
  const long nblk = inv_items<T, MODE, V>(a);
  if (nblk <= 0) return 0;
  const void *A0 = nullptr, *A1 = nullptr;
  const int t0 = (a.kind == INV_UV) ? TQV : a.table;
  if (MODE == MODE_BF16X3) {
    A0 = tb.inv_bf[t0];
    A1 = tb.inv_bf[TQU];
  } else if (MODE == MODE_F32MFMA) {
    A0 = tb.inv_f32[t0];
    A1 = tb.inv_f32[TQU];
  } else if (MODE == MODE_F64) {
    A0 = tb.inv_f64[t0];
    A1 = tb.inv_f64[TQU];
  }
  const void* tv = (MODE == MODE_F64) ? (const void*)tb.filt64 : (const void*)tb.filt32;
  const void* tw = (MODE == MODE_F64) ? (const void*)tb.tw64 : (const void*)tb.tw32;
  dim3 grid((unsigned)nblk), block(InvCfg<T, MODE, V>::NT);
  if (a.kind == INV_UV) {
    if (fused)
      k_inv<T, MODE, INV_UV, true, V><<<grid, block, 0, s>>>(a, A0, A1, tv, tw);
    else
      k_inv<T, MODE, INV_UV, false, V><<<grid, block, 0, s>>>(a, A0, A1, tv, tw);
  } else {
    if (fused)
      k_inv<T, MODE, INV_SCALAR, true, V><<<grid, block, 0, s>>>(a, A0, A1, tv, tw);
    else
      k_inv<T, MODE, INV_SCALAR, false, V><<<grid, block, 0, s>>>(a, A0, A1, tv, tw);
  }
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

// The tile variant of a fused inverse on a plan that was not tuned, from the
// blocks it would have with half the fields per block (V = 3).  While those
// have a CU each (256) they only engage idle CUs; above, whole blocks on 512
// threads, whose matrix tiles are full.  Round trip inverses in us, V = 0, 2, 3, by
// those blocks: T42 BF16X3 108: 18.2, 13.5, 12.4; 224: 18.7, 14.1, 13.1; 280:
// 19.0, 14.6, 16.8; 432: 19.9, 15.7, 18.5; FP32MFMA 216: 24.9, 17.4, 15.8; 280: 25.0, 17.6,
// 19.2; T21 BF16X3 224: 11.8, 10.6, 10.2; 270: 12.2, 10.9, 12.1; T63 BF16X3 252: 26.6,
// 19.1, 17.5; 264: 26.6, 19.1, 23.0.  Exceptions: FP64 at T21, whose short rows
// keep 256 threads busy (L20, 16 members 18.7, 21.0, 29.9); FP32, which has no
// matrix tiles and whose vector sums want the most waves, up to T42 (L20, 16
// members 233, 145, 111) and to two and a half blocks per CU at T63 (sp2fc alone
// 504: 95, 75, 57; 630: 94, 75, 73; 756: 95, 76, 82; the round trip's inverse 528:
// 218, 145, 118; 1008: 278, 177, 196).
template <int T, int MODE>
static int inv_auto(long nblk3) {
  if (MODE == MODE_F64 && T == 21) return 0;
  if (MODE == MODE_F32 && T <= 42) return 3;
  return nblk3 <= (MODE == MODE_F32 && T == 63 ? 640 : 256) ? 3 : 2;
}

// blocks at V = 3 of the call that a launch belongs to: a call that runs its
// members in chunks uses the tiles of one launch of them all
template <int T, int MODE>
static long inv_rule(InvArgs a) {
  if (a.nrule > 0) a.nmem = a.nrule;
  return inv_items<T, MODE, 3>(a);
}
template <int T, int MODE>
static long fwd_rule(FwdArgs a) {
  if (a.nrule > 0) a.nmem = a.nrule;
  return fwd_items<T, MODE, 3>(a);
}

// the unfused (drop-in) transforms always use the default tiles
template <int T, int MODE>
static int inv_t(const Tables& tb, bool fused, const InvArgs& a, hipStream_t s) {
  const int v = !fused ? 0 : a.var >= 0 ? a.var : inv_auto<T, MODE>(inv_rule<T, MODE>(a));
  if (v == 1) return inv_tv<T, MODE, 1>(tb, fused, a, s);
  if (v == 2) return inv_tv<T, MODE, 2>(tb, fused, a, s);
  if (v == 3) return inv_tv<T, MODE, 3>(tb, fused, a, s);
  return inv_tv<T, MODE, 0>(tb, fused, a, s);
}

template <int T, int MODE, int V>
static int inv_rt_tv(const Tables& tb, const InvArgs& aq, const InvArgs* aj, int nj,
                     const InvArgs& au, hipStream_t s) {
  using C = InvCfg<T, MODE, V>;
  constexpr int NPB = TS<T>::NPAIR / C::LP;
  if (nj < 1 || nj > INV_ONE_MAX || aq.nmem != au.nmem) return -1;
  const int gq = (aq.nfield + C::FB - 1) / C::FB;
  const int gu = (au.nlev + C::FB / 2 - 1) / (C::FB / 2);
  const long nblk = (long)aq.nmem * NPB * (gq + nj + gu);
  if (nblk <= 0) return 0;
  InvOneJobs one{};
  for (int k = 0; k < nj; ++k) {
    const InvArgs& a = aj[k];
    if (a.nmem != aq.nmem || a.nfield != 1 || a.src0 != aj[0].src0) return -1;
    one.tab[k] = MODE == MODE_BF16X3    ? (const void*)tb.inv_bf[a.table]
                 : MODE == MODE_F32MFMA ? (const void*)tb.inv_f32[a.table]
                                        : (const void*)tb.inv_f64[a.table];
    one.table[k] = a.table;
    one.dst0[k] = a.dst0;
    one.dlam[k] = a.dlam;
  }
  const void *tq = nullptr, *tv0 = nullptr, *tu = nullptr;
  if (MODE == MODE_BF16X3) {
    tq = tb.inv_bf[TQI];
    tv0 = tb.inv_bf[TQV];
    tu = tb.inv_bf[TQU];
  } else if (MODE == MODE_F32MFMA) {
    tq = tb.inv_f32[TQI];
    tv0 = tb.inv_f32[TQV];
    tu = tb.inv_f32[TQU];
  } else if (MODE == MODE_F64) {
    tq = tb.inv_f64[TQI];
    tv0 = tb.inv_f64[TQV];
    tu = tb.inv_f64[TQU];
  }
  const void* tv = (MODE == MODE_F64) ? (const void*)tb.filt64 : (const void*)tb.filt32;
  const void* tw = (MODE == MODE_F64) ? (const void*)tb.tw64 : (const void*)tb.tw32;
  k_inv_rt<T, MODE, V><<<(unsigned)nblk, C::NT, 0, s>>>(aq, aj[0], au, tq, one, tv0, tu,
                                                       tv, tw, gq, nj, gu);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

template <int T, int MODE>
static int inv_rt_t(const Tables& tb, const InvArgs& aq, const InvArgs* aj, int nj,
                    const InvArgs& au, hipStream_t s) {
  const int v = aq.var >= 0 ? aq.var
                            : inv_auto<T, MODE>(inv_rule<T, MODE>(aq) +
                                                nj * inv_rule<T, MODE>(aj[0]) +
                                                inv_rule<T, MODE>(au));
  if (v == 1) return inv_rt_tv<T, MODE, 1>(tb, aq, aj, nj, au, s);
  if (v == 2) return inv_rt_tv<T, MODE, 2>(tb, aq, aj, nj, au, s);
  if (v == 3) return inv_rt_tv<T, MODE, 3>(tb, aq, aj, nj, au, s);
  return inv_rt_tv<T, MODE, 0>(tb, aq, aj, nj, au, s);
}

template <int T, int MODE>
static size_t fwd_scratch_t(int nmem, int nfield) {
  using C = FwdCfg<T, MODE>;
  if (C::NPB == 1) return 0;
  return (size_t)C::NPB * nmem * nfield * TS<T>::NRSP * sizeof(RealT<MODE>);
}

template <int T, int MODE, int V>
static int fwd_tv(const Tables& tb, bool fused, const FwdArgs& a, void* scratch, size_t sbytes,
                  hipStream_t s) {
  using C = FwdCfg<T, MODE, V>;
  using R = RealT<MODE>;
  const long nblk = fwd_items<T, MODE, V>(a);
  if (nblk <= 0) return 0;
  if (C::NPB > 1 && (scratch == nullptr || sbytes < fwd_scratch_t<T, MODE>(a.nmem, a.nfield)))
    return -4;
  if (a.table != TQC) return -2;  // the table whose pairs lie side by side by 16 bytes
  const void* tv = (MODE == MODE_F64) ? (const void*)tb.fwd2 : (const void*)tb.fwd4;
  const void* tw = (MODE == MODE_F64) ? (const void*)tb.tw64 : (const void*)tb.tw32;
  dim3 grid((unsigned)nblk), block(C::NT);
  if (fused)
    k_fwd<T, MODE, true, V><<<grid, block, 0, s>>>(a, tv, tw, scratch);
  else
    k_fwd<T, MODE, false, V><<<grid, block, 0, s>>>(a, tv, tw, scratch);
  if (C::NPB > 1) {
    const long total = (long)a.nmem * a.nfield * TS<T>::NRSP;
    k_reduce_partials<R><<<(unsigned)((total + 255) / 256), 256, 0, s>>>(
        (const R*)scratch, (R*)a.sp, C::NPB, a.nmem, a.nfield, TS<T>::NRSP, a.sp_stride, a.dst0);
  }
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

// The tile variant of a fused direct transform on a plan that was not tuned,
// from the blocks of V = 3 (half the fields, 512 threads): as long as those fit
// the CUs (FP32: two per CU), a block's own time counts and the smallest block
// is the fastest; above, 512 threads on all fields, but 256 in FP64 at T42,
// where two such blocks share a CU's LDS and a wide one does not fit twice.
// Round trip directs in us, V = 0, 2, 3: T42 L20 BF16X3, 1 member 15.1, 9.0,
// 5.3; 16 members 15.4, 13.5, 16.2; FP64, 1 member 11.4, 9.6, 9.9; 16 members
// 32.4, 41.0, 42.6; T63 L20 BF16X3, 16 members 66.9, 42.7, 43.4.
template <int T, int MODE>
static int fwd_auto(long nblk3) {
  if (nblk3 <= (MODE == MODE_F64 ? 256 : 512)) return 3;
  return (MODE == MODE_F64 && T == 42) ? 0 : 2;
}

template <int T, int MODE>
static int fwd_t(const Tables& tb, bool fused, const FwdArgs& a, void* scratch, size_t sbytes,
                 hipStream_t s) {
  const int v = !fused ? 0 : a.var >= 0 ? a.var : fwd_auto<T, MODE>(fwd_rule<T, MODE>(a));
  if (v == 1) return fwd_tv<T, MODE, 1>(tb, fused, a, scratch, sbytes, s);
  if (v == 2) return fwd_tv<T, MODE, 2>(tb, fused, a, scratch, sbytes, s);
  if (v == 3) return fwd_tv<T, MODE, 3>(tb, fused, a, scratch, sbytes, s);
  return fwd_tv<T, MODE, 0>(tb, fused, a, scratch, sbytes, s);
}

#define EXO_DISPATCH_T(fn, ...)                                   \
  switch (tb.ntru) {                                              \
    case 21: return fn<21, MODE_X>(__VA_ARGS__);                  \
    case 42: return fn<42, MODE_X>(__VA_ARGS__);                  \
    case 63: return fn<63, MODE_X>(__VA_ARGS__);                  \
    case 127: return fn<127, MODE_X>(__VA_ARGS__);                \
    default: return -2;                                           \
  }

template <int MODE_X>
int inv_mode(const Tables& tb, bool fused, const InvArgs& a, hipStream_t s) {
  EXO_DISPATCH_T(inv_t, tb, fused, a, s)
}
template <int MODE_X>
int inv_rt_mode(const Tables& tb, const InvArgs& aq, const InvArgs* aj, int nj,
                const InvArgs& au, hipStream_t s) {
  EXO_DISPATCH_T(inv_rt_t, tb, aq, aj, nj, au, s)
}
template <int MODE_X>
int fwd_mode(const Tables& tb, bool fused, const FwdArgs& a, void* scr, size_t sb,
                    hipStream_t s) {
  EXO_DISPATCH_T(fwd_t, tb, fused, a, scr, sb, s)
}
template <int MODE_X>
size_t scr_mode(const Tables& tb, int nmem, int nfield) {
  switch (tb.ntru) {
    case 21: return fwd_scratch_t<21, MODE_X>(nmem, nfield);
    case 42: return fwd_scratch_t<42, MODE_X>(nmem, nfield);
    case 63: return fwd_scratch_t<63, MODE_X>(nmem, nfield);
    case 127: return fwd_scratch_t<127, MODE_X>(nmem, nfield);
    default: return 0;
  }
}

}  // namespace exo
