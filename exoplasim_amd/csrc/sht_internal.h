// sht_internal.h -- library-internal declarations (plan object, kernels,
// launch helpers).  Not part of the C ABI.
#pragma once
#include <hip/hip_runtime.h>

#include <initializer_list>

#include "sht_common.h"

struct exo_sht_plan_s;

namespace exo {

__global__ void k_inigau(int klat, double* pz0, double* pzw);
__global__ void k_legini(int ntru, int npair, const double* sid, const double* gwd, double* tab);
__global__ void k_filtered(int ntru, int npair, const double* tab, const double* skgpsp,
                           const double* skspgp, double* out64, float* out32);
__global__ void k_pack_inv(int ntru, int npair, int kbmax, int t, const double* filt64,
                           float* f32, double* f64);
__global__ void k_pack_inv_bf(int ntru, int npair, int t, const double* filt64, uint16_t* bf);
__global__ void k_pack_dir(int ntru, int npair, int rb, int t, const double* filt64, float* out);
template <typename R>
__global__ void k_pack_fwd(int npair, int ncsp, const R* filt, R* out);
__global__ void k_twiddle(int n, double* tw64, float* tw32);

// Which inverse transform a launch performs.
enum InvKind : int {
  INV_SCALAR = 0,  // sp2fc with qi (or sp2fcdmu with qj) of a run of fields
  INV_UV = 1,      // dv2uv: (D, zeta) -> (u cos, v cos), terms qv and qu
};

// Device tables of one truncation (all FP64 values computed on the GPU).
struct Tables {
  int ntru = 0, nlat = 0, nlon = 0, npair = 0, ncsp = 0;
  int kbmax = 0;
  double* sid = nullptr;      // [nlat]
  double* gwd = nullptr;      // [nlat]
  double* tab = nullptr;      // [8][npair][ncsp] unfiltered
  double* filt64 = nullptr;   // [8][npair][ncsp] filter folded in
  float* filt32 = nullptr;
  // the direct transform's table qc, its pairs of 16 bytes together side by side
  float* fwd4 = nullptr;      // [npair/4][ncsp][4] of filt32
  double* fwd2 = nullptr;     // [npair/2][ncsp][2] of filt64
  double* skgpsp = nullptr;   // [ntru+1]
  double* skspgp = nullptr;
  // split-BF16 inverse table operands (3 planes): qi, qj, and under TQV qv and
  // qu together
  uint16_t* inv_bf[NTAB] = {};
  float* inv_f32[NTAB] = {};    // FP32-MFMA inverse table operands
  double* inv_f64[NTAB] = {};   // FP64-MFMA inverse table operands
  float* dir_f32[NTAB] = {};    // MFMA direct table operands (qc, qe, qm, qq)
  int dir_rb = 0;               // row tiles of 16 per (m, parity)
  double* tw64 = nullptr;     // [nlon] complex
  float* tw32 = nullptr;
  double plavor = 0.0;
};

// Launch arguments of the fused/unfused inverse and direct transforms.
struct InvArgs {
  const void* sp;   // spectral input (member stride sp_stride reals)
  void* out;        // grid (fused) or Fourier (unfused) output
  long sp_stride, out_stride;
  int nmem;
  int kind;
  int table;        // INV_SCALAR: TQI or TQJ
  int src0, dst0, nfield;               // INV_SCALAR field runs
  int vor0, div0, u0, v0, nlev;         // INV_UV
  double plavor;
  int var;          // tile variant (InvCfg / FwdCfg), -1: by the size of the call
  int nrule;        // members of the whole call, of which this launch runs nmem (0: nmem)
  int dlam;         // INV_SCALAR: times i m before the FFT (d/dlambda)
  // MODE_BF16X3: the parity-ordered spectral operand (launch_pack) of
  // fields [bpk_f0, ...), bpk_stride floats per member
  const void* bpk;
  long bpk_stride;
  int bpk_f0;
};

// what differs between the one-field jobs of launch_inverse_rt
constexpr int INV_ONE_MAX = 3;
struct InvOneJobs {
  const void* tab[INV_ONE_MAX];  // packed table
  int table[INV_ONE_MAX], dst0[INV_ONE_MAX], dlam[INV_ONE_MAX];
};

struct FwdArgs {
  const void* in;   // grid (fused) or Fourier (unfused) input
  void* sp;         // spectral output (or partial sums when npb > 1)
  long in_stride, sp_stride;
  int nmem;
  int src0, dst0, nfield;
  int table;        // TQC
  int var;          // tile variant (InvCfg / FwdCfg), -1: by the size of the call
  int nrule;        // members of the whole call, of which this launch runs nmem (0: nmem)
};

// One term of a multi-input direct transform: out_o[oc] += sign * t * X_in[ic]
struct DirxTerm {
  int8_t in, ic, oc, sign;
  int8_t table;
  int8_t o = 0;
};
// One job of the multi-input direct transforms: nout spectral outputs (2*NCSP,
// nlev) of nin Fourier inputs fc(2, NLON/2, NLAT, nlev), per member
struct DirxArgs {
  const void* in[3];
  void* out[2];
  int nin, nout, nlev, nterm;
  DirxTerm terms[10];
  int nmem;                   // members (>= 1)
  long in_stride, out_stride; // member strides of the inputs / the output, in reals
};
inline DirxArgs dirx_job(std::initializer_list<const void*> in, std::initializer_list<void*> out,
                         std::initializer_list<DirxTerm> terms, int nlev, int nmem,
                         long in_stride, long out_stride) {
  DirxArgs a{};
  for (const void* x : in) a.in[a.nin++] = x;
  for (void* x : out) a.out[a.nout++] = x;
  for (const DirxTerm& t : terms) a.terms[a.nterm++] = t;
  a.nlev = nlev;
  a.nmem = nmem;
  a.in_stride = in_stride;
  a.out_stride = out_stride;
  return a;
}
// The jobs of the folded branches of src/legmod.f90; a term is {input, input
// component, output component, sign, table[, output]}.
// mktend (:538-549): D = qq.ke - qe.fv + i qm.fu and Z = qe.fu + i qm.fv,
// which share their inputs
inline DirxArgs mktend_dz(const void* ke, const void* fv, const void* fu, void* d, void* z,
                          int nlev, int nmem, long fs, long ss) {
  return dirx_job({ke, fv, fu}, {d, z},
                  {{0, 0, 0, +1, TQQ}, {1, 0, 0, -1, TQE}, {2, 1, 0, -1, TQM},
                   {0, 1, 1, +1, TQQ}, {1, 1, 1, -1, TQE}, {2, 0, 1, +1, TQM},
                   {2, 0, 0, +1, TQE, 1}, {1, 1, 0, -1, TQM, 1},
                   {2, 1, 1, +1, TQE, 1}, {1, 0, 1, +1, TQM, 1}},
                  nlev, nmem, fs, ss);
}
// and T = qe.vt + qc.tn - i qm.ut; qtend (:468-496) is the same sum with (q;
// vq, qn, uq) for (T; vt, tn, ut)
inline DirxArgs mktend_t(const void* vt, const void* tn, const void* ut, void* t, int nlev,
                         int nmem, long fs, long ss) {
  return dirx_job({vt, tn, ut}, {t},
                  {{0, 0, 0, +1, TQE}, {1, 0, 0, +1, TQC}, {2, 1, 0, +1, TQM},
                   {0, 1, 1, +1, TQE}, {1, 1, 1, +1, TQC}, {2, 0, 1, -1, TQM}},
                  nlev, nmem, fs, ss);
}
// uv2dv (:391-422): D = -qe.v + i qm.u, Z = qe.u + i qm.v
inline DirxArgs uv2dv_dz(const void* u, const void* v, void* d, void* z, int nlev, int nmem,
                         long fs, long ss) {
  return dirx_job({u, v}, {d, z},
                  {{1, 0, 0, -1, TQE}, {0, 1, 0, -1, TQM}, {1, 1, 1, -1, TQE}, {0, 0, 1, +1, TQM},
                   {0, 0, 0, +1, TQE, 1}, {1, 1, 0, -1, TQM, 1},
                   {0, 1, 1, +1, TQE, 1}, {1, 0, 1, +1, TQM, 1}},
                  nlev, nmem, fs, ss);
}
// fc2sp (:178-223) of nlev fields with table t
inline DirxArgs fc2sp_job(const void* fc, void* sp, int t, int nlev, int nmem, long fs, long ss) {
  return dirx_job({fc}, {sp}, {{0, 0, 0, +1, (int8_t)t}, {0, 1, 1, +1, (int8_t)t}}, nlev, nmem,
                  fs, ss);
}

// all jobs (over the same members) in one launch: uv2dv_dz or an fc2sp_job
// alone, or up to four of mktend_dz, mktend_t and fc2sp_job with at least
// one of the former
int launch_dirx(const Tables& T, int mode, const DirxArgs* jobs, int njob, hipStream_t s);

int launch_inverse(const Tables& T, int mode, bool fused, const InvArgs& a, hipStream_t s);
// the sp2fc run (aq), nj <= INV_ONE_MAX one-field scalar jobs (aj: sp2fc,
// sp2fcdmu or d/dlambda of one and the same field) and the dv2uv (au) of a
// round trip or a dynamics step, fused with fc2gp, in one launch; tile
// variant aq.var
int launch_inverse_rt(const Tables& T, int mode, const InvArgs& aq, const InvArgs* aj, int nj,
                      const InvArgs& au, hipStream_t s);
int launch_forward(const Tables& T, int mode, bool fused, const FwdArgs& a, void* scratch,
                   size_t scratch_bytes, hipStream_t s);
size_t forward_scratch_bytes(const Tables& T, int mode, int nmem, int nfield);
// Fourier rows of the T127 FP32 direct transform of grid input
size_t fwd_fft_scratch_bytes(const Tables& T, int nmem, int nfield);
// in-place FFTs of lot rows of n values, for nmem members mstride values
// apart; the forward FFT (dir -1) may read its rows from src instead
// (smstride per member) and write only the first kmax complex coefficients
// of each row (0: all n/2)
int launch_fft(const Tables& T, int mode, int dir, void* a, int n, long lot, hipStream_t s,
               int nmem = 1, long mstride = 0, const void* src = nullptr, long smstride = 0,
               int kmax = 0);
// parity-ordered copy (PK layout, sht_common.h) of fp32 spectral fields
// [f0, f0+nf) of nmem members for the split-BF16 inverse; out holds nmem *
// nf * pk_field(ntru) floats
int launch_pack(const Tables& T, const float* sp, long sp_stride, int f0, int nf, int nmem,
                float* out, hipStream_t s);
inline size_t pack_bytes(const Tables& T, int nmem, int nf) {
  return sizeof(float) * (size_t)nmem * nf * pk_field(T.ntru);
}

// the device tables of a plan (defined with the plan object)
const Tables& plan_tables(const exo_sht_plan_s* p);

}  // namespace exo
