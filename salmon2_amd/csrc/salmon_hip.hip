// MI355X (gfx950) real-time Kohn-Sham propagation hot path: device state,
// kernels and the C ABI declared in include/salmon_hip.h.
//
// Kernels (one launch each, all deterministic: no floating-point atomics):
//   k_update_kvector  phase table zekr_uV and per-k stencil terms
//                     (update_kvector_nonlocalpt, src/common/hamiltonian.f90:847-903)
//   k_proj<NW>        batched projector x orbital contraction on FP64 MFMA
//                     (v_mfma_f64_16x16x4f64): uVpsi of zpseudo
//                     (src/common/nonlocal_potential.f90:360-369) for NW = 1 and the
//                     four moments of calc_current_nonlocal (density_matrix.f90:532-591)
//                     for NW = 4 (NW = 5: with the next step's projection)
//   k_proj_scatter    the KB term of a Taylor term with the projection of its result
//   k_stencilz, k_stencil8, k_stencil<HC,NC>  25-point stencil + V_local + k+A gradient
//                     (zstencil_typical_seq, zstencil_core/typical/seq.f90:17-127) fed by
//                     direct global->LDS DMA rings; in the last Taylor term it also forms
//                     the sum of taylor.f90:53-114
//   k_nl_scatter      the KB scatter of zpseudo (nonlocal_potential.f90:370-378) as a
//                     deterministic per-point gather over a point->(atom, j) inverse map
//   k_taylor_small    a whole orbital per block for small grids: the Taylor step (or H psi) from LDS;
//   k_current_small   its current (small_grid.h)
//   k_density_*       calc_density (density_matrix.f90:150-230)
//   k_current_*       stencil_current + calc_current (density_matrix.f90:240-530)
//   k_dipole_part/_sum calc_dip (src/rt/dip.f90:114-225)
//   k_dft_*           Hartree potential (poisson_ft, src/poisson/poisson_periodic.f90:23-242)
//   k_xc_pz           PZ81 LDA (src/xc/builtin_pz.f90:23-83) and its spin-polarised form
//                     (src/xc/builtin_pz_sp.f90:23-98)
//   k_update_vlocal   update_vlocal (src/common/hamiltonian.f90:813-843) with the
//                     predictor-corrector average (src/rt/time_evolution_step.f90:404)
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <algorithm>
#include <atomic>
#include <climits>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "salmon_hip.h"

namespace {

thread_local std::string g_err;

int fail(int code, const char *fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_err = buf;
  return code;
}

#define HIPCHK(x)                                                                            \
  do {                                                                                       \
    hipError_t e_ = (x);                                                                     \
    if (e_ != hipSuccess) return fail(SALMON_HIP_EHIP, "%s: %s", #x, hipGetErrorString(e_)); \
  } while (0)

#define LAUNCHCHK(name)                                                                          \
  do {                                                                                           \
    hipError_t e_ = hipGetLastError();                                                           \
    if (e_ != hipSuccess) return fail(SALMON_HIP_EHIP, "launch %s: %s", name, hipGetErrorString(e_)); \
  } while (0)

constexpr int kBlock = 256;
constexpr int kProjJC = 32;      // sphere points staged per LDS chunk in k_proj
constexpr int kProjOrb = 64;     // orbitals per k_proj block (4 waves x 16)
constexpr int kMaxLmaPerAtom = 16;
constexpr int kDensGroup = 32;   // orbitals per density partial

__device__ __forceinline__ int wrapi(int v, int n) { return (v + 8 * n) % n; }

// Complex element types: double2 (FP64) or float2 (FP32, mixed-precision chain).
// A float2 element is moved by two dword DMAs per 64-point wave chunk (lane i ->
// point 32k + i/2, half i%2), a double2 element by one dwordx4 DMA (lane i -> point i).
template <typename R> struct Cx;
template <> struct Cx<double> { using T = double2; };
template <> struct Cx<float> { using T = float2; };
template <typename E> struct DmaW;
template <> struct DmaW<double2> { static constexpr int W = 1; };
template <> struct DmaW<float2> { static constexpr int W = 2; };

template <typename D, typename S>
__device__ __forceinline__ D cvt2(const S &v) {
  D r;
  r.x = v.x;
  r.y = v.y;
  return r;
}

// ---------------------------------------------------------------------------
// Phase table and per-k stencil coefficients
// ---------------------------------------------------------------------------
struct KvecArgs {
  const double *veck;    // (3, nk)
  const double *rxyz;    // (3, nps, natom)
  const double *uv;      // (nps, nlma)
  const int *mps;        // (natom)
  const int2 *atom_lma;  // (natom): first ilma, count
  const int *entof;      // (nps, natom): CSR entry of each sphere point
  double2 *zekr;         // (nps, nlma, nk)
  double2 *zent;         // (cmax, nent, nk)
  double *kpar;          // (16, nk): k_lap0, k_nabt(12), kAc(3)
  double coef_nab[12];
  double coef_lap0;
  double ax, ay, az;
  // with actab: A = (actab(:, itt) + actab(:, itt-1)) / 2 at the device step counter *itt
  const double *actab;
  const int *itt;
  int tmax;              // last row of actab (nt + 1); the step counter is clamped to 1..tmax
  int natom, nlma, nps, nk, nent, cmax;
  int split;             // blocks per atom and k: 1, or cmax of one projector each
};

// the midpoint field of the current step from the device table, else the by-value field
__device__ __forceinline__ void kvec_field(const KvecArgs &a, double &ax, double &ay, double &az) {
  if (a.actab) {
    const int t = min(max(*a.itt, 1), a.tmax);
    ax = 0.5 * (a.actab[3 * t + 0] + a.actab[3 * (t - 1) + 0]);
    ay = 0.5 * (a.actab[3 * t + 1] + a.actab[3 * (t - 1) + 1]);
    az = 0.5 * (a.actab[3 * t + 2] + a.actab[3 * (t - 1) + 2]);
  } else {
    ax = a.ax;
    ay = a.ay;
    az = a.az;
  }
}

// A block takes all projectors of an atom at one k (a point's phase serves them all) or, in launches of
// few atoms and k-points, one of them (kvec_split).
__device__ __forceinline__ void update_kvector_body(const KvecArgs &a, int ib, int ik) {
  double ax, ay, az;
  kvec_field(a, ax, ay, az);
  const double kx = a.veck[3 * ik + 0] + ax;
  const double ky = a.veck[3 * ik + 1] + ay;
  const double kz = a.veck[3 * ik + 2] + az;
  if (ib == 0 && threadIdx.x == 0) {
    double *kp = a.kpar + 16 * ik;
    double ss = kx * kx;
    ss = ss + ky * ky;
    ss = ss + kz * kz;
    kp[0] = a.coef_lap0 + 0.5 * ss;
    for (int n = 0; n < 4; ++n) {
      kp[1 + n] = kx * a.coef_nab[n];
      kp[5 + n] = ky * a.coef_nab[4 + n];
      kp[9 + n] = kz * a.coef_nab[8 + n];
    }
    kp[13] = kx;
    kp[14] = ky;
    kp[15] = kz;
  }
  const int ia = ib / a.split;
  if (ia >= a.natom) return;
  const int2 al = a.atom_lma[ia];
  const int l0 = ib - ia * a.split;
  const int nl = a.split > 1 ? min(1, al.y - l0) : al.y;  // the block's projectors: l0 .. l0 + nl - 1
  if (nl < 1) return;
  const int m = a.mps[ia];
  for (int j = threadIdx.x; j < m; j += blockDim.x) {
    const double *uv = a.uv + (size_t)j + (size_t)a.nps * (al.x + l0);
    double u[4];  // the first projectors' values beside the phase's latency
#pragma unroll
    for (int l = 0; l < 4; ++l) u[l] = l < nl ? uv[(size_t)a.nps * l] : 0.0;
    const int e = a.entof[(size_t)j + (size_t)a.nps * ia];
    const double *r = a.rxyz + 3 * ((size_t)j + (size_t)a.nps * ia);
    const double th = kx * r[0] + ky * r[1] + kz * r[2];
    double s, c;
    sincos(th, &s, &c);
    double2 *ze = a.zent + (size_t)a.cmax * ((size_t)e + (size_t)a.nent * ik) + l0;
    double2 *zk = a.zekr + (size_t)j + (size_t)a.nps * ((size_t)(al.x + l0) + (size_t)a.nlma * ik);
#pragma unroll
    for (int l = 0; l < 4; ++l)
      if (l < nl) zk[(size_t)a.nps * l] = ze[l] = make_double2(c * u[l], -s * u[l]);
    for (int l = 4; l < nl; ++l) {
      const double ul = uv[(size_t)a.nps * l];
      zk[(size_t)a.nps * l] = ze[l] = make_double2(c * ul, -s * ul);
    }
  }
}

__global__ __launch_bounds__(kBlock) void k_update_kvector(KvecArgs a) { update_kvector_body(a, blockIdx.x, blockIdx.y); }

// Per-k stencil terms only (hpsi reads system%vec_Ac at every call,
// src/common/hamiltonian.f90:146-155; the phase table is left untouched).
__global__ void k_set_kpar(KvecArgs a) {
  const int ik = threadIdx.x;
  if (ik >= a.nk) return;
  double ax, ay, az;
  kvec_field(a, ax, ay, az);
  const double kx = a.veck[3 * ik + 0] + ax;
  const double ky = a.veck[3 * ik + 1] + ay;
  const double kz = a.veck[3 * ik + 2] + az;
  double *kp = a.kpar + 16 * ik;
  double ss = kx * kx;
  ss = ss + ky * ky;
  ss = ss + kz * kz;
  kp[0] = a.coef_lap0 + 0.5 * ss;
  for (int n = 0; n < 4; ++n) {
    kp[1 + n] = kx * a.coef_nab[n];
    kp[5 + n] = ky * a.coef_nab[4 + n];
    kp[9 + n] = kz * a.coef_nab[8 + n];
  }
  kp[13] = kx;
  kp[14] = ky;
  kp[15] = kz;
}

// ---------------------------------------------------------------------------
// Projector x orbital contraction on FP64 MFMA (v_mfma_f64_16x16x4f64).
// D[n][o] = sum_K A[n][K] B[K][o] with K = (sphere point j, re/im),
// o = 16 orbitals per wave, n = (lma-weight index lw, re/im part).
//   part re:  Re(conj(Z) r_w psi) = Zr r_w psi_re + Zi r_w psi_im
//   part im:  Im(conj(Z) r_w psi) = Zr r_w psi_im - Zi r_w psi_re
// r_0 = 1 (plain projection), r_1..3 = rxyz components (current moments).
// Operand layout: lane L holds A[L%16][L/16] and B[L/16][L%16]; the result
// lands as D[L/16 + 4r][L%16] in register r.  Rows are therefore assigned as
// n = 8h + 4p + q (q = 0..3, p = part, h = half) <-> lw = 8t + 4h + q, so the
// re and im rows of one lw sit in registers (2h, 2h+1) of the same lane.
// ---------------------------------------------------------------------------
struct ProjArgs {
  const void *psi;        // orbital block base (double2, or float2 in the mixed-precision chain)
  const double2 *zekr;    // (nps, nlma, nk)
  const double *rxyz;     // (3, nps, natom)
  const int *jidx;        // (nps, natom) offsets within an orbital block
  const int *mps;         // (natom)
  const int2 *atom_lma;   // (natom): first ilma, count
  const double *rinv;     // (nlma)
  double2 *out;           // NW=1: c(nb, nlma, nk) scaled by rinv; NW=4, 5: (4, nlma, nb, nk) raw
  size_t osz;
  int nb, nk, natom, nps, nlma, ngrp;
  const int *skip;        // device flag: the launch does nothing when it is set (null: never)
  // NW=5: weight 4 is the plain projection under a second phase table (the next step's), written
  // as c(nb, nlma, nk) scaled by rinv
  const double2 *zekr2;
  double2 *out2;
};

// XCD-aware order of a launch of nblk blocks (block b runs on XCD b % 8): the blocks of one XCD
// take a contiguous range of the work items, so the cache lines that neighbouring items share
// are read through one L2
__device__ __forceinline__ int xcd_order(int b, int nblk) {
  const int nfull = (nblk / 8) * 8;
  return b < nfull ? (b % 8) * (nblk / 8) + b / 8 : b;
}

// Waves of a block on parts of the sphere (ProjStage's S): 4 where the operand staging is small, 1 where
// four private stagings of it would cost more than they spread (d projectors under five weights,
// 512 orbitals at 96 x 14 x 12: 79 us split, 57 us not; s+p projectors, 1024 orbitals at 32^3: 187 us split
// and 202 us not for the fused pass, 128 orbitals there 14 us and 21 us for the projection).  Handles of
// the mixed precision keep the points in one sequence (fused pass of 216 atoms, 1728 orbitals 985 us, 953 us
// split), for reproducibility: what is rounded to FP32 after the sum then stays bit for bit what it was before
// the split (either way 5e-8 from FP64 on that case).  One handle's
// forms all sum a projection in one order (the chunks of S = 4 are of one length).
constexpr int proj_split(int lm, bool mixed) { return lm <= 4 && !mixed ? 4 : 1; }
constexpr int proj_orb(int split) { return split == 4 ? 16 : kProjOrb; }

// Staging of the contraction.  S = 1: a block takes 64 orbitals, 16 per wave, and the waves share the
// projectors of a chunk of JC sphere points; S = 4: a block takes 16 orbitals and its waves every
// fourth chunk each, with the partial sums added in wave order at the end (launches of few blocks).
// The A operand lies in LDS as MT tiles of 8 weighted projectors (complex) per point, unused ones
// zero, so that a lane's value for an MFMA is one 8-byte read and a sign; the orbitals as 16 per
// wave and point.  Both are XOR-swizzled: writes (lanes on points) and reads (lanes on projectors or
// orbitals) both spread over the banks.
template <int NW, int LMX, int S>
struct ProjStage {
  static constexpr int JC = NW == 1 && S == 1 ? kProjJC : kProjJC / 2;
  static constexpr int MT = (NW * LMX + 7) / 8;
  static constexpr int OB = proj_orb(S);           // orbitals per block
  static constexpr int kPer = JC / 4;                 // orbital values per lane and chunk
  static constexpr int kT = S == 4 ? 64 : kBlock;     // threads that stage one chunk's projectors
  static constexpr int kZPer = (JC * LMX + kT - 1) / kT;
  double2 sp[4][JC * 16];
  double2 z[S][JC * 8 * MT];
  static __device__ __forceinline__ int zs(int jj, int lw) {
    return jj * 8 * MT + (lw ^ (((jj >> 1) & 7) | (MT % 2 == 0 ? (jj & 1) << 3 : 0)));
  }
  static __device__ __forceinline__ int so(int jj, int o) { return jj * 16 + (o ^ (jj & 15)); }
};
typedef double __attribute__((ext_vector_type(4))) d4;

template <int S>
__device__ __forceinline__ void stage_sync() {
  if constexpr (S == 1) {
    __syncthreads();
  } else {  // wave-private staging: LDS accesses of one wave stay in order
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

// acc += A B over one staged chunk
template <int NW, int LMX, int S>
__device__ __forceinline__ void stage_mfma(const double2 *sp, const double2 *z, int lane, int ntile, d4 *acc) {
  using P = ProjStage<NW, LMX, S>;
  const int h = (lane >> 4) >> 1, comp = (lane >> 4) & 1;  // K row: point 2 ks + h, re/im of psi
  const int oc = lane & 15;                                // orbital column (B) / output row (A)
  const int part = (oc >> 2) & 1, lw0 = (oc >> 3) * 4 + (oc & 3);
  const double *spd = (const double *)sp + comp, *zd = (const double *)z + (part ^ comp);
  const unsigned neg = part && !comp ? 0x80000000u : 0u;
#pragma unroll 4
  for (int ks = 0; ks < P::JC / 2; ++ks) {
    const int jp = 2 * ks + h;
    const double bval = spd[2 * P::so(jp, oc)];
#pragma unroll
    for (int tt = 0; tt < P::MT; ++tt) {
      if (tt < ntile) {
        const double v = zd[2 * P::zs(jp, tt * 8 + lw0)];
        const double aval = __hiloint2double(__double2hiint(v) ^ neg, __double2loint(v));
        acc[tt] = __builtin_amdgcn_mfma_f64_16x16x4f64(aval, bval, acc[tt], 0, 0, 0);
      }
    }
  }
}

// S = 4: the waves' sums into wave 0's, in wave order (red: 3 x MT x 64 d4, over the staging)
template <int MT>
__device__ __forceinline__ void stage_reduce(d4 *red, int wave, int lane, d4 *acc) {
  __syncthreads();
  if (wave > 0)
#pragma unroll
    for (int tt = 0; tt < MT; ++tt) red[((wave - 1) * MT + tt) * 64 + lane] = acc[tt];
  __syncthreads();
  if (wave == 0)
#pragma unroll
    for (int tt = 0; tt < MT; ++tt)
      for (int w = 0; w < 3; ++w) acc[tt] += red[(w * MT + tt) * 64 + lane];
}

// LMX bounds the projectors of one atom (the tile and staging sizes).  Bound by the gathers: a sphere's
// points of one orbital are runs of a few points, and nearly every 128-byte line of the orbitals is
// read.  With the A values formed per wave from unswizzled tables (45 vector instructions an MFMA) NW = 5 took
// 264 us for 64 atoms, 32^3 and 1024 orbitals, 131 us so (0.6 GB of lines, 4.6 TB/s), and 1183 and 692 us for
// 216 atoms, 48^3 and 1728 orbitals (5.1 TB/s); NW = 1 for 64 atoms and 128 orbitals 37 and 14 us.
template <int NW, typename TP, int LMX, int S>
__device__ __forceinline__ void proj_body(const ProjArgs &a, int bid) {
  static_assert(LMX <= kMaxLmaPerAtom, "LMX bounds the projectors of one atom");
  using P = ProjStage<NW, LMX, S>;
  constexpr int JC = P::JC, MT = P::MT;
  constexpr size_t kRed = S == 4 ? sizeof(d4) * 3 * MT * 64 : 0;
  __shared__ __attribute__((aligned(32))) char lds[sizeof(P) > kRed ? sizeof(P) : kRed];
  P &st = *(P *)lds;
  const int grp = bid % a.ngrp;
  const int t = bid / a.ngrp;
  const int ia = t % a.natom;
  const int ik = t / a.natom;
  const int2 al = a.atom_lma[ia];
  const int m = a.mps[ia];
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int nlw = NW * al.y;            // (lma, weight) pairs of this atom
  const int ntile = (nlw + 7) >> 3;     // 8 lw (16 rows) per MFMA tile
  const size_t kbase = (size_t)ik * a.nb;
  const int ob0 = grp * P::OB + (S == 4 ? 0 : 16 * wave);  // first orbital of this wave
  double2 *sp = st.sp[wave], *z = st.z[S == 4 ? wave : 0];
  const int zt = S == 4 ? lane : (int)threadIdx.x;

  d4 acc[MT];
#pragma unroll
  for (int tt = 0; tt < MT; ++tt) acc[tt] = d4{0.0, 0.0, 0.0, 0.0};
  for (int e = zt; e < JC * 8 * ntile; e += P::kT)
    if (e / JC >= nlw) z[P::zs(e % JC, e / JC)] = make_double2(0.0, 0.0);

  // the next chunk is loaded into registers while the MFMAs consume the staged one
  TP pre[P::kPer];
  double2 zpre[P::kZPer], zpre2[NW == 5 ? P::kZPer : 1];
  double rpre[3] = {0.0, 0.0, 0.0};
  const TP *psi = (const TP *)a.psi;
  const int *jx = a.jidx + (size_t)a.nps * ia;
  const double2 *zk = a.zekr + (size_t)a.nps * ((size_t)al.x + (size_t)a.nlma * ik);
  const double2 *zk2 = NW == 5 ? a.zekr2 + (size_t)a.nps * ((size_t)al.x + (size_t)a.nlma * ik) : nullptr;
  // every thread loads the same sphere point of each chunk; its grid index is fetched one chunk
  // ahead, so the psi gathers wait on one load, not two
  const int jt = lane % JC, o0 = lane / JC, l0 = zt / JC;
  constexpr int kStep = S * JC;
  const int jb = S == 4 ? wave * JC : 0;
  int jnext = jb + jt < m ? jx[jb + jt] : 0;
  auto load_chunk = [&](int j0) {
    const int jv = jnext;
    const int j = j0 + jt;
    jnext = j + kStep < m ? jx[j + kStep] : 0;
#pragma unroll
    for (int r = 0; r < P::kZPer; ++r) {
      const int l = l0 + (P::kT / JC) * r;
      zpre[r] = (j < m && l < al.y) ? zk[(size_t)j + (size_t)a.nps * l] : make_double2(0.0, 0.0);
      if constexpr (NW == 5)
        zpre2[r] = (j < m && l < al.y) ? zk2[(size_t)j + (size_t)a.nps * l] : make_double2(0.0, 0.0);
    }
    if constexpr (NW > 1) {
#pragma unroll
      for (int i = 0; i < 3; ++i) rpre[i] = j < m ? a.rxyz[3 * ((size_t)j + (size_t)a.nps * ia) + i] : 0.0;
    }
#pragma unroll
    for (int r = 0; r < P::kPer; ++r) {
      const int ob = ob0 + o0 + (64 / JC) * r;
      TP v;
      v.x = 0;
      v.y = 0;
      if (j < m && ob < a.nb) v = psi[(kbase + ob) * a.osz + jv];
      pre[r] = v;
    }
  };
  load_chunk(jb);
  for (int j0 = jb; j0 < m; j0 += kStep) {
#pragma unroll
    for (int r = 0; r < P::kPer; ++r) sp[P::so(jt, o0 + (64 / JC) * r)] = cvt2<double2>(pre[r]);
#pragma unroll
    for (int r = 0; r < P::kZPer; ++r) {
      const int l = l0 + (P::kT / JC) * r;
      if (l < al.y) {
        if constexpr (NW == 1) {
          z[P::zs(jt, l)] = zpre[r];
        } else {
          z[P::zs(jt, l * NW)] = zpre[r];
#pragma unroll
          for (int i = 0; i < 3; ++i) z[P::zs(jt, l * NW + 1 + i)] = make_double2(zpre[r].x * rpre[i], zpre[r].y * rpre[i]);
          if constexpr (NW == 5) z[P::zs(jt, l * NW + 4)] = zpre2[r];
        }
      }
    }
    stage_sync<S>();
    if (j0 + kStep < m) load_chunk(j0 + kStep);
    stage_mfma<NW, LMX, S>(sp, z, lane, ntile, acc);
    stage_sync<S>();
  }
  if constexpr (S == 4) {
    stage_reduce<MT>((d4 *)lds, wave, lane, acc);
    if (wave > 0) return;
  }
  // lane (kq, oc) holds rows kq + 4r: r = 2h -> re of lw = 8t + 4h + kq, r = 2h+1 -> its im
  const int kq = lane >> 4;
  const int ob = ob0 + (lane & 15);
  if (ob >= a.nb) return;
#pragma unroll
  for (int tt = 0; tt < MT; ++tt) {
    if (tt >= ntile) break;
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const int lw = tt * 8 + hh * 4 + kq;
      if (lw >= nlw) continue;
      const int w = lw % NW;
      const int l = lw / NW;
      const int ilma = al.x + l;
      const double re = acc[tt][2 * hh], im = acc[tt][2 * hh + 1];
      if (NW == 1) {
        const double s = a.rinv[ilma];
        a.out[((size_t)ik * a.nlma + ilma) * a.nb + ob] = make_double2(re * s, im * s);
      } else if (NW == 5 && w == 4) {
        const double s = a.rinv[ilma];
        a.out2[((size_t)ik * a.nlma + ilma) * a.nb + ob] = make_double2(re * s, im * s);
      } else {
        a.out[((kbase + ob) * a.nlma + ilma) * 4 + w] = make_double2(re, im);
      }
    }
  }
}

// up to 4 projectors per atom the registers leave four waves per SIMD
template <int NW, typename TP, int LMX, int S>
__global__ __launch_bounds__(kBlock, LMX == 4 ? 4 : 2) void k_proj(ProjArgs a) {
  if (a.skip && *a.skip) return;  // a device-side gate switched this launch off
  proj_body<NW, TP, LMX, S>(a, xcd_order(blockIdx.x, gridDim.x));
}

// ---------------------------------------------------------------------------
// KB term of one H application fused with the projection of its result: for a Taylor term
// h = H h_prev the pass adds s * sum_lma c_prev(lma) zekr(j, lma) at the sphere points that one
// (atom, point) pair covers alone and projects the completed h onto the atom's projectors (the
// c of the next term), reading h once.  Block = (k, atom, orbitals) as in k_proj<1>: each
// lane owns one sphere point of every chunk and part of the orbitals; after the chunk is
// staged in LDS it completes its points (exclusive ones: KB sum in ascending ilma, in FP64, then
// rounded to TP as k_nl_scatter stores it), writes them back and puts the rounded values into the
// LDS tile the MFMAs read.  Points covered by several pairs are completed beforehand by
// k_nl_scatter over their list, and no point is written by two blocks (an exclusive point
// belongs to one atom, and the blocks of one atom split the orbitals), so the pass is
// deterministic and race-free.  c_prev for the block's orbitals is staged in dynamic LDS
// (cmax x orbitals of the block).  Bound by the lines read and written back: 64 atoms, 32^3, 1024
// orbitals 213 us before the A values were staged and the points split over the waves, 187 us so
// (0.9 GB, 4.8 TB/s); 216 atoms, 48^3, 1728 orbitals in complex FP32 990 and 953 us (4 GB).
// ---------------------------------------------------------------------------
struct ProjScatArgs {
  ProjArgs p;              // projection of h (p.psi = h, p.out = its c, scaled by rinv)
  const double2 *cin;      // c of h_prev (nb, nlma, nk), scaled by rinv
  const int *jexcl;        // (nps, natom): offset within an orbital block if one pair covers the point, else -1
  double2 s;               // h += s * sum (1 for the terms without the Taylor sum)
  int cmax;                // projectors per atom, at most (the row count of the staged c)
};

template <typename TP, int LM, int S>
__device__ __forceinline__ void proj_scatter_body(const ProjScatArgs &A, int bid) {
  static_assert(LM <= kMaxLmaPerAtom, "LM bounds the projectors of one atom");
  const ProjArgs &a = A.p;
  using P = ProjStage<1, LM, S>;
  constexpr int JC = P::JC, MT = P::MT;
  constexpr size_t kRed = S == 4 ? sizeof(d4) * 3 * MT * 64 : 0;
  __shared__ __attribute__((aligned(32))) char lds[sizeof(P) > kRed ? sizeof(P) : kRed];
  P &st = *(P *)lds;
  extern __shared__ double2 csh[];  // cmax x OB
  const int grp = bid % a.ngrp;
  const int t = bid / a.ngrp;
  const int ia = t % a.natom;
  const int ik = t / a.natom;
  const int2 al = a.atom_lma[ia];
  const int m = a.mps[ia];
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int nlw = al.y;
  const int ntile = (nlw + 7) >> 3;
  const size_t kbase = (size_t)ik * a.nb;
  const int ow = S == 4 ? 0 : 16 * wave;  // first orbital of this wave within the block
  double2 *sp = st.sp[wave], *z = st.z[S == 4 ? wave : 0];
  const int zt = S == 4 ? lane : (int)threadIdx.x;

  for (int e = threadIdx.x; e < al.y * P::OB; e += kBlock) {
    const int l = e / P::OB, ob = grp * P::OB + e % P::OB;
    csh[e] = ob < a.nb ? A.cin[((size_t)ik * a.nlma + al.x + l) * a.nb + ob] : make_double2(0.0, 0.0);
  }
  for (int e = zt; e < JC * 8 * ntile; e += P::kT)
    if (e / JC >= nlw) z[P::zs(e % JC, e / JC)] = make_double2(0.0, 0.0);
  __syncthreads();

  d4 acc[MT];
#pragma unroll
  for (int tt = 0; tt < MT; ++tt) acc[tt] = d4{0.0, 0.0, 0.0, 0.0};
  TP pre[P::kPer];
  double2 zpre[P::kZPer];
  const int *jx = a.jidx + (size_t)a.nps * ia;
  const int *jxe = A.jexcl + (size_t)a.nps * ia;
  const double2 *zk = a.zekr + (size_t)a.nps * ((size_t)al.x + (size_t)a.nlma * ik);
  // This thread's point of a chunk and its orbitals o0 + kOs r.  S = 1: over the whole block, so that all waves
  // complete points where the orbitals fill one wave's MFMA columns only (16 orbitals of 20 x 26 x 28, 8 atoms of 9
  // projectors, mixed: Taylor step 619 us, 813 us with each wave on its own 16; 64 orbitals the same).
  constexpr int kOs = P::kT / JC;
  const int jt = zt % JC, o0 = zt / JC, l0 = o0;
  TP *h = (TP *)a.psi + (kbase + grp * P::OB + o0) * a.osz;
  const size_t hs = kOs * a.osz;
  const int nor = a.nb - grp * P::OB - o0;  // orbitals of this thread: r with kOs r < nor
  constexpr int kStep = S * JC;
  const int jb = S == 4 ? wave * JC : 0;
  int jnext = jb + jt < m ? jx[jb + jt] : 0;
  int xnext = jb + jt < m ? jxe[jb + jt] : -1;
  int jload = 0, xload = -1;  // point offset and exclusive offset of the chunk last loaded
  double2 zown[LM];           // zekr of this thread's point of that chunk (exclusive points only)
  auto load_chunk = [&](int j0) {
    jload = jnext;
    xload = xnext;
    const int j = j0 + jt;
#pragma unroll
    for (int l = 0; l < LM; ++l)
      zown[l] = (xload >= 0 && l < al.y) ? zk[(size_t)j + (size_t)a.nps * l] : make_double2(0.0, 0.0);
    const bool more = j + kStep < m;
    jnext = more ? jx[j + kStep] : 0;
    xnext = more ? jxe[j + kStep] : -1;
#pragma unroll
    for (int r = 0; r < P::kZPer; ++r) {
      const int l = l0 + (P::kT / JC) * r;
      zpre[r] = (j < m && l < al.y) ? zk[(size_t)j + (size_t)a.nps * l] : make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int r = 0; r < P::kPer; ++r) {
      TP v;
      v.x = 0;
      v.y = 0;
      if (j < m && kOs * r < nor) v = h[r * hs + jload];
      pre[r] = v;
    }
  };
  load_chunk(jb);
  for (int j0 = jb; j0 < m; j0 += kStep) {
    // complete this thread's point if one pair covers it (xload >= 0 implies j0 + jt < m) while
    // staging the chunk
#pragma unroll
    for (int r = 0; r < P::kPer; ++r) {
      const int o = o0 + kOs * r;
      double2 v = cvt2<double2>(pre[r]);
      if (xload >= 0 && kOs * r < nor) {
        double2 sum = make_double2(0.0, 0.0);
#pragma unroll
        for (int l = 0; l < LM; ++l) {
          if (l < al.y) {
            const double2 cv = csh[l * P::OB + o];
            sum.x += cv.x * zown[l].x - cv.y * zown[l].y;
            sum.y += cv.x * zown[l].y + cv.y * zown[l].x;
          }
        }
        v.x += A.s.x * sum.x - A.s.y * sum.y;
        v.y += A.s.x * sum.y + A.s.y * sum.x;
        const TP vt = cvt2<TP>(v);
        h[r * hs + jload] = vt;
        v = cvt2<double2>(vt);
      }
      (S == 4 ? sp : st.sp[o >> 4])[P::so(jt, o & 15)] = v;
    }
#pragma unroll
    for (int r = 0; r < P::kZPer; ++r) {
      const int l = l0 + (P::kT / JC) * r;
      if (l < al.y) z[P::zs(jt, l)] = zpre[r];
    }
    stage_sync<S>();
    if (j0 + kStep < m) load_chunk(j0 + kStep);
    stage_mfma<1, LM, S>(sp, z, lane, ntile, acc);
    stage_sync<S>();
  }
  if constexpr (S == 4) {
    stage_reduce<MT>((d4 *)lds, wave, lane, acc);
    if (wave > 0) return;
  }
  const int kq = lane >> 4;
  const int ob = grp * P::OB + ow + (lane & 15);
  if (ob >= a.nb) return;
#pragma unroll
  for (int tt = 0; tt < MT; ++tt) {
    if (tt >= ntile) break;
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const int lw = tt * 8 + hh * 4 + kq;
      if (lw >= nlw) continue;
      const int ilma = al.x + lw;
      const double re = acc[tt][2 * hh], im = acc[tt][2 * hh + 1];
      const double sc = a.rinv[ilma];
      a.out[((size_t)ik * a.nlma + ilma) * a.nb + ob] = make_double2(re * sc, im * sc);
    }
  }
}

template <typename TP, int LM, int S>
__global__ __launch_bounds__(kBlock, LM == 4 ? 4 : 2) void k_proj_scatter(ProjScatArgs A) {
  if (A.p.skip && *A.p.skip) return;  // a device-side gate switched this launch off
  proj_scatter_body<TP, LM, S>(A, xcd_order(blockIdx.x, gridDim.x));
}

constexpr int kMaxComb = 5;   // Taylor order up to 6

// ---------------------------------------------------------------------------
// Local hpsi: 25-point stencil + V + k.grad (zstencil_typical_seq,
// zstencil_core/typical/seq.f90:17-127), with the Taylor combination folded
// into the last term.  The KB term is added afterwards by k_nl_scatter.
//
// Block = full x rows (nx) x TY rows in y (one point per thread), streaming z
// over [z0, z0+TZ).  Every per-plane input arrives by direct global->LDS DMA
// (global_load_lds, issued through inline asm so that only explicit
// s_waitcnt vmcnt(N) waits gate it) kDmaDepth planes ahead:
//   tile ring  (kRingT slots): psi rows of planes z .. z+4+D  (x/y neighbours, queue head)
//   halo ring  (D+1 slots):    the 4+4 y-halo rows of planes z .. z+D
//   V ring     (D+1 slots):    V_local of planes z .. z+D
//   comb ring  (2 slots, last term only): psi, h1 .. h_{N-2} of planes z, z+1
// z neighbours come from a 9-deep register queue fed from the tile ring.  The
// only compiler-visible global memory operation in the loop is the store, so
// the in-order vmcnt counter never forces an early wait on the ring.
// NC < 0:  hout = H_loc in
// NC >= 0: hout = (((psi + c1 h1) + ... + c_{N-1} in) + c_N H_loc in), N = NC + 1
// ---------------------------------------------------------------------------
constexpr int kDmaDepth = 2;
// The per-plane wait lets the DMAs issued in the previous iteration stay in flight: the data a
// plane needs must have been issued at least two iterations earlier.
static_assert(kDmaDepth >= 2, "the ring wait assumes a look-ahead of at least two planes");
constexpr int kRingT = 5 + kDmaDepth;
constexpr int kRingH = kDmaDepth + 1;
constexpr int kTile = 256;  // tile slot size (elements), = 4 waves x 64 lanes

typedef __attribute__((address_space(3))) void lds_void;

__device__ __forceinline__ unsigned lds_addr(const void *p) {
  return (unsigned)(uintptr_t)((lds_void *)p);
}
// lane i of the wave writes its element to LDS byte address m0 + i * size
// (M0 is not used by compiler-generated gfx950 code in these kernels: LDS
// instructions do not read it)
__device__ __forceinline__ void dma16(const void *g, unsigned m0) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(m0), "v"(g) : "memory");
}
__device__ __forceinline__ void dma4(const void *g, unsigned m0) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dword %1, off" ::"s"(m0), "v"(g) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}


// One element chunk of 64 points (this wave's) into LDS at byte address m0:
// W = 1: off[0] = the lane's point; W = 2: off[k] = point 32k + lane/2.
template <typename E>
__device__ __forceinline__ void dma_chunk(const E *base, const size_t *off, unsigned m0, int lane) {
  if constexpr (DmaW<E>::W == 1) {
    dma16(base + off[0], m0);
  } else {
    dma4((const float *)(base + off[0]) + (lane & 1), m0);
    dma4((const float *)(base + off[1]) + (lane & 1), m0 + 256u);
  }
}

struct StencilArgs {
  const void *in;
  void *hout;
  double2 *sink;          // one element per thread absorbing the stores of lanes without a point
  const void *comb[kMaxComb];  // comb[0] double2 (psi); comb[n >= 1] the chain type
  double2 zc[kMaxComb + 1];
  const double *V;        // (nx, ny, nz, nspin)
  const double *kpar;     // (16, nk)
  double lap[12];         // coef_lap(4,3)
  size_t osz;
  int nx, ny, nz, ly, nspin, nb, nk;
  int TY, TZ, nyt, nzt, nblk;
  int TX, nxt;            // x tiles (stencil_tilez with XT; else one tile of nx)
  const int *skip;        // device flag: the launch does nothing when it is set (null: never)
};

// TI: element type of `in`; R: arithmetic of the stencil and local-potential
// products; TO: element type of `hout`.  Plain FP64: (double2, double, double2).
// Mixed form: (double2, float, float2) for the first term, (float2, float, float2)
// for the middle ones and (float2, float, double2) for the last, whose Taylor sum
// is formed in FP64 from psi (FP64) and h_1 .. h_N (FP32).  (FP64 arithmetic in the
// first term, rounded once at the store, measured 10% slower at 32^3.)
// One tile (orbital block, y-tile, z-chunk) = `bid` of the system described by `a`.
template <typename TI, typename R, typename TO, int HC, int NC, int BS>
__device__ __forceinline__ void stencil_tile(const StencilArgs &a, int bid, double2 *lds) {
  static_assert(HC == 0 || BS == kTile, "y-halo tiles are 4 waves wide");
  using CH = typename Cx<R>::T;
  constexpr bool FINAL = NC >= 0;
  constexpr int D = kDmaDepth;
  constexpr int WI = DmaW<TI>::W;
  constexpr int WC = DmaW<CH>::W;
  constexpr unsigned EB = sizeof(TI);
  // DMA instructions per wave per plane, in issue order: comb, tile (WI), halo (HC*WI), V (2 x dword);
  // then 1 store
  constexpr int kOpsAfterComb = WI + HC * WI + 2 + 1;
  TI *tileR = (TI *)lds;                                  // kRingT x BS
  TI *haloR = tileR + kRingT * BS;                     // kRingH x HC*BS
  double *vR = (double *)(haloR + kRingH * HC * BS);   // kRingH x BS doubles
  char *combR = (char *)(vR + kRingH * BS);            // 2 x NC x BS x 16 bytes

  const int ytile = bid % a.nyt;
  const int zt = (bid / a.nyt) % a.nzt;
  const int b = bid / (a.nyt * a.nzt);
  const int ik = b / a.nb;
  const int ispin = b % a.nspin;

  const int nx = a.nx, ny = a.ny, nz = a.nz, ly = a.ly;
  const int TY = a.TY;
  const int y0 = ytile * TY;
  // With one z chunk the column is a full period and may start anywhere: y-tile t starts 4t planes
  // earlier, so that its upper y-halo rows of plane p are fetched in the same iteration as the
  // next tile's own rows of p (4 planes ahead of their use) and come from the L2.  Planes are
  // counted unwrapped in [z0, z1) and wrapped on every access.
  const int zph = (HC > 0 && a.nzt == 1) ? (nz - (4 * ytile) % nz) % nz : 0;
  const int z0 = zt * a.TZ + zph;
  const int z1 = min(zt * a.TZ + a.TZ, nz) + zph;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int ntile = TY * nx;
  const bool active = tid < ntile;
  const int te = active ? tid : 0;          // element this lane computes (dummy lanes repeat element 0)
  const int tx = te % nx;
  const int ty = te / nx;
  const int y = y0 + ty;
  const bool outY = active && y < ny;
  const int yw = wrapi(y, ny);

  const size_t zs = (size_t)nx * ly;
  const size_t orbOff = (size_t)b * a.osz;
  const TI *in = (const TI *)a.in + orbOff;
  const size_t colOff = (size_t)tx + (size_t)nx * yw;
  const size_t gplane = (size_t)nx * ny;
  // tile points this lane moves (W = 1: its own; W = 2: points 32k + lane/2 of the wave's chunk)
  auto tile_off = [&](int W, size_t *off) {
    if (W == 1) {
      off[0] = colOff;
      return;
    }
    for (int k = 0; k < 2; ++k) {
      const int e = 64 * wave + 32 * k + (lane >> 1);
      const int ec = e < ntile ? e : 0;
      off[k] = (size_t)(ec % nx) + (size_t)nx * wrapi(y0 + ec / nx, ny);
    }
  };
  size_t toffI[2], toffC[2];
  tile_off(WI, toffI);
  tile_off(WC, toffC);
  // V: two dword DMAs per wave, each covering 32 points of the wave's 64 (lane i -> point i/2, half i%2)
  const double *Vb = a.V + (size_t)ispin * gplane * nz;
  size_t voff[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int e = 64 * wave + 32 * k + (lane >> 1);
    const int ec = e < ntile ? e : 0;
    voff[k] = 2 * ((size_t)(ec % nx) + (size_t)nx * wrapi(y0 + ec / nx, ny)) + (lane & 1);
  }

  // halo points of this lane: chunk c = wave + 4k, points 64c + (lane | 32kk + lane/2)
  size_t hoff[HC > 0 ? HC : 1][2];
#pragma unroll
  for (int k = 0; k < HC; ++k)
#pragma unroll
    for (int kk = 0; kk < WI; ++kk) {
      const int e = 64 * (wave + 4 * k) + (WI == 1 ? lane : 32 * kk + (lane >> 1));
      const int ec = e < 8 * nx ? e : 0;
      const int hr = ec / nx, hx = ec % nx;
      const int gy = hr < 4 ? y0 - 4 + hr : y0 + TY + (hr - 4);
      hoff[k][kk] = (size_t)hx + (size_t)nx * wrapi(gy, ny);
    }
  // LDS byte addresses of this wave's chunk in each ring (uniform per wave)
  const unsigned tileA = __builtin_amdgcn_readfirstlane(lds_addr(tileR) + EB * 64u * wave);
  const unsigned haloA = __builtin_amdgcn_readfirstlane(lds_addr(haloR) + EB * 64u * wave);
  const unsigned vA = __builtin_amdgcn_readfirstlane(lds_addr(vR) + 8u * 64u * wave);
  const unsigned combA = __builtin_amdgcn_readfirstlane(lds_addr(combR) + 16u * 64u * wave);
  const unsigned combAC = __builtin_amdgcn_readfirstlane(lds_addr(combR) + (unsigned)sizeof(CH) * 64u * wave);

  auto dma_tile = [&](int plane, int slot) {
    dma_chunk<TI>(in + zs * wrapi(plane, nz), toffI, tileA + EB * BS * slot, lane);
  };
  auto dma_halo = [&](int plane, int slot) {
#pragma unroll
    for (int k = 0; k < HC; ++k)
      dma_chunk<TI>(in + zs * wrapi(plane, nz), hoff[k], haloA + EB * (HC * BS * slot + 4 * 64 * k), lane);
  };
  auto dma_v = [&](int plane, int slot) {
    const float *vb = (const float *)Vb + 2 * gplane * wrapi(plane, nz);
    dma4(vb + voff[0], vA + 8u * BS * slot);
    dma4(vb + voff[1], vA + 8u * BS * slot + 256u);
  };
  auto dma_comb = [&](int plane, int slot) {
    const size_t pl = orbOff + zs * wrapi(plane, nz);
#pragma unroll
    for (int n = 0; n < (NC > 0 ? NC : 1); ++n) {
      if (n >= NC) break;
      // every comb array owns BS x 16 bytes per slot; psi is double2, the chain arrays CH
      if (n == 0) {
        size_t o0[1] = {colOff};
        dma_chunk<double2>((const double2 *)a.comb[0] + pl, o0, combA + 16u * BS * (NC * slot), lane);
      } else {
        dma_chunk<CH>((const CH *)a.comb[n] + pl, toffC, combAC + 16u * BS * (NC * slot + n), lane);
      }
    }
  };

  // y-neighbour LDS offsets: rows ty+n (n = 1..4, -1..-4) in the tile slot or the halo slot
  int yoff[8];
  bool yhal[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int n = i < 4 ? i + 1 : -(i - 3);
    const int r = ty + n;
    if (HC == 0) {  // the tile is the whole xy-plane (TY == ny): y wraps inside it
      yoff[i] = (r < 0 ? r + TY : (r >= TY ? r - TY : r)) * nx + tx;
      yhal[i] = false;
    } else if (r >= 0 && r < TY) {
      yoff[i] = r * nx + tx;
      yhal[i] = false;
    } else {
      yoff[i] = (r < 0 ? r + 4 : 4 + r - TY) * nx + tx;
      yhal[i] = true;
    }
  }
  int xo[8];
#pragma unroll
  for (int n = 1; n <= 4; ++n) {
    xo[n - 1] = ty * nx + wrapi(tx + n, nx);
    xo[3 + n] = ty * nx + wrapi(tx - n, nx);
  }
  const double *kp = a.kpar + 16 * ik;
  const R klap0 = (R)kp[0];
  R nab[12], lap[12];
#pragma unroll
  for (int i = 0; i < 12; ++i) {
    nab[i] = (R)kp[1 + i];
    lap[i] = (R)a.lap[i];
  }

  // prologue: queue planes z0-4 .. z0+3 (plain loads), rings for planes z0 .. z0+3+D
  CH q[9];
#pragma unroll
  for (int i = 0; i < 8; ++i) q[i] = cvt2<CH>(in[colOff + zs * wrapi(z0 - 4 + i, nz)]);
  __builtin_amdgcn_s_waitcnt(0);  // compiler-visible: the queue loads are complete
  if (FINAL) dma_comb(z0, z0 & 1);
  for (int p = 0; p < 4 + D; ++p) dma_tile(z0 + p, (z0 + p) % kRingT);
  for (int p = 0; p < D; ++p) {
    dma_halo(z0 + p, (z0 + p) % kRingH);
    dma_v(z0 + p, (z0 + p) % kRingH);
  }
  wait_vm<0>();

  int sT = z0 % kRingT, sH = z0 % kRingH;  // ring slots of plane z
  for (int z = z0; z < z1; ++z) {
    // planes z (halo, V, comb) and z+4 (tile) were issued >= one full plane ago
    wait_vm<kOpsAfterComb>();
    __syncthreads();
    const int sTn = (sT + 4 + D) % kRingT;  // slot of plane z+4+D (= slot of z-1)
    const int sHn = (sH + D) % kRingH;      // slot of plane z+D   (= slot of z-1)
    // past the chunk's last needed plane the look-ahead re-reads that plane (an L2 hit) into the
    // slot, which is never read: every wave still issues the same memory operations per plane
    if (FINAL) dma_comb(min(z + 1, z1 - 1), (z + 1) & 1);
    dma_tile(min(z + 4 + D, z1 + 3), sTn);
    dma_halo(min(z + D, z1 - 1), sHn);
    dma_v(min(z + D, z1 - 1), sHn);

    const TI *T = tileR + BS * sT;
    const TI *H = haloR + HC * BS * sH;
    q[8] = cvt2<CH>(tileR[BS * ((sT + 4) % kRingT) + te]);
    CH v, w;
    {
      const CH p1 = cvt2<CH>(T[xo[0]]), p2 = cvt2<CH>(T[xo[1]]), p3 = cvt2<CH>(T[xo[2]]), p4 = cvt2<CH>(T[xo[3]]);
      const CH m1 = cvt2<CH>(T[xo[4]]), m2 = cvt2<CH>(T[xo[5]]), m3 = cvt2<CH>(T[xo[6]]), m4 = cvt2<CH>(T[xo[7]]);
      v.x = lap[0] * (p1.x + m1.x) + lap[1] * (p2.x + m2.x) + lap[2] * (p3.x + m3.x) + lap[3] * (p4.x + m4.x);
      v.y = lap[0] * (p1.y + m1.y) + lap[1] * (p2.y + m2.y) + lap[2] * (p3.y + m3.y) + lap[3] * (p4.y + m4.y);
      w.x = nab[0] * (p1.x - m1.x) + nab[1] * (p2.x - m2.x) + nab[2] * (p3.x - m3.x) + nab[3] * (p4.x - m4.x);
      w.y = nab[0] * (p1.y - m1.y) + nab[1] * (p2.y - m2.y) + nab[2] * (p3.y - m3.y) + nab[3] * (p4.y - m4.y);
    }
    {
      const CH p1 = cvt2<CH>((yhal[0] ? H : T)[yoff[0]]), p2 = cvt2<CH>((yhal[1] ? H : T)[yoff[1]]);
      const CH p3 = cvt2<CH>((yhal[2] ? H : T)[yoff[2]]), p4 = cvt2<CH>((yhal[3] ? H : T)[yoff[3]]);
      const CH m1 = cvt2<CH>((yhal[4] ? H : T)[yoff[4]]), m2 = cvt2<CH>((yhal[5] ? H : T)[yoff[5]]);
      const CH m3 = cvt2<CH>((yhal[6] ? H : T)[yoff[6]]), m4 = cvt2<CH>((yhal[7] ? H : T)[yoff[7]]);
      v.x += lap[4] * (p1.x + m1.x) + lap[5] * (p2.x + m2.x) + lap[6] * (p3.x + m3.x) + lap[7] * (p4.x + m4.x);
      v.y += lap[4] * (p1.y + m1.y) + lap[5] * (p2.y + m2.y) + lap[6] * (p3.y + m3.y) + lap[7] * (p4.y + m4.y);
      w.x += nab[4] * (p1.x - m1.x) + nab[5] * (p2.x - m2.x) + nab[6] * (p3.x - m3.x) + nab[7] * (p4.x - m4.x);
      w.y += nab[4] * (p1.y - m1.y) + nab[5] * (p2.y - m2.y) + nab[6] * (p3.y - m3.y) + nab[7] * (p4.y - m4.y);
    }
    v.x += lap[8] * (q[5].x + q[3].x) + lap[9] * (q[6].x + q[2].x) + lap[10] * (q[7].x + q[1].x) + lap[11] * (q[8].x + q[0].x);
    v.y += lap[8] * (q[5].y + q[3].y) + lap[9] * (q[6].y + q[2].y) + lap[10] * (q[7].y + q[1].y) + lap[11] * (q[8].y + q[0].y);
    w.x += nab[8] * (q[5].x - q[3].x) + nab[9] * (q[6].x - q[2].x) + nab[10] * (q[7].x - q[1].x) + nab[11] * (q[8].x - q[0].x);
    w.y += nab[8] * (q[5].y - q[3].y) + nab[9] * (q[6].y - q[2].y) + nab[10] * (q[7].y - q[1].y) + nab[11] * (q[8].y - q[0].y);

    const CH t = q[4];
    const R vcur = (R)vR[BS * sH + te];
    CH hh;
    hh.x = (vcur * t.x + klap0 * t.x) - (R)0.5 * v.x + w.y;
    hh.y = (vcur * t.y + klap0 * t.y) - (R)0.5 * v.y - w.x;
    TO o;
    if constexpr (FINAL) {
      constexpr int N = NC + 1;
      const double2 td = cvt2<double2>(t), h = cvt2<double2>(hh);
      const char *Cb = combR + 16u * BS * (NC * (z & 1));
      double2 od;
      if (N == 1) {
        od = td;
      } else {
        od = ((const double2 *)Cb)[te];
#pragma unroll
        for (int n = 1; n < N - 1; ++n) {
          const double2 cc = cvt2<double2>(((const CH *)(Cb + 16u * BS * n))[te]);
          const double2 zc = a.zc[n - 1];
          od.x = od.x + (zc.x * cc.x - zc.y * cc.y);
          od.y = od.y + (zc.x * cc.y + zc.y * cc.x);
        }
        const double2 zc = a.zc[N > 1 ? N - 2 : 0];
        od.x = od.x + (zc.x * td.x - zc.y * td.y);
        od.y = od.y + (zc.x * td.y + zc.y * td.x);
      }
      const double2 zc = a.zc[N - 1];
      od.x = od.x + (zc.x * h.x - zc.y * h.y);
      od.y = od.y + (zc.x * h.y + zc.y * h.x);
      o = cvt2<TO>(od);
    } else {
      o = cvt2<TO>(hh);
    }
    // the store is the one compiler-visible vm op per plane (counted in kOpsAfterComb):
    // every lane stores, lanes without a point into the sink, so each wave issues it
    TO *dst = outY ? (TO *)a.hout + orbOff + colOff + zs * wrapi(z, nz) : (TO *)a.sink + tid;
    *dst = o;
#pragma unroll
    for (int i = 0; i < 8; ++i) q[i] = q[i + 1];
    sT = (sT + 1 == kRingT) ? 0 : sT + 1;
    sH = (sH + 1 == kRingH) ? 0 : sH + 1;
  }
  wait_vm<0>();  // drain the look-ahead DMAs before the LDS is released
}

// ---------------------------------------------------------------------------
// Whole-plane form of the terms without the Taylor sum, for planes of up to PY * BS
// points: lane `tid` computes the plane elements tid + k * BS (k < PY), so a 32 x 32
// plane takes 512 threads with two points each.  There is no y halo (y wraps inside
// the plane held in LDS), so every orbital plane is read once, plus the 4 + 4 wrap
// planes of the z period.  LDS: tile ring (5 + D) x PY*BS elements, V ring (D + 1) x
// PY*BS doubles, D = look-ahead in planes (D = 2: 136 KB for 32 x 32 in FP64, one block of
// 8 waves per CU, two waves per SIMD, which leaves 256 registers per lane for the two z
// queues).  The wait at the top of a plane lets the DMAs of the last D - 1 planes stay in
// flight.  The DMA issue discipline is the one of stencil_tile; lanes without a point
// store into the sink.
// ---------------------------------------------------------------------------
template <typename TI, typename R, typename TO, int PY, int BS, int D>
__device__ __forceinline__ void stencil_plane(const StencilArgs &a, int bid, double2 *lds) {
  static_assert(PY * BS <= 1024, "the sink holds 1024 elements");
  static_assert(D >= 2, "the ring wait assumes a look-ahead of at least two planes");
  using CH = typename Cx<R>::T;
  constexpr int kRingT = 5 + D, kRingH = D + 1;
  constexpr int WI = DmaW<TI>::W;
  constexpr unsigned EB = sizeof(TI);
  constexpr int SL = PY * BS;  // elements per ring slot
  // memory instructions per wave per plane, in issue order: tile DMAs (PY x WI), V DMAs (PY x 2), PY stores
  constexpr int kOps = PY * WI + 2 * PY + PY;
  TI *tileR = (TI *)lds;                       // kRingT x SL
  double *vR = (double *)(tileR + kRingT * SL);  // kRingH x SL

  const int zt = bid % a.nzt;
  const int b = bid / a.nzt;
  const int ik = b / a.nb;
  const int ispin = b % a.nspin;
  const int nx = a.nx, ny = a.ny, nz = a.nz, ly = a.ly;
  const int z0 = zt * a.TZ;
  const int z1 = min(z0 + a.TZ, nz);
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int ntile = nx * ny;
  const size_t zs = (size_t)nx * ly;
  const size_t orbOff = (size_t)b * a.osz;
  const TI *in = (const TI *)a.in + orbOff;
  const size_t gplane = (size_t)nx * ny;
  // in-plane offset x + nx y of element e (elements past the plane repeat element 0)
  auto pofs = [&](int e) {
    const int ec = e < ntile ? e : 0;
    return (size_t)(ec % nx) + (size_t)nx * (ec / nx);
  };

  int te[PY], xo[PY][8], yo[PY][8];
  bool act[PY];
  size_t col[PY], toff[PY][2], voff[PY][2];
#pragma unroll
  for (int k = 0; k < PY; ++k) {
    const int e = tid + k * BS;
    act[k] = e < ntile;
    te[k] = act[k] ? e : 0;
    const int tx = te[k] % nx, ty = te[k] / nx;
    col[k] = (size_t)tx + (size_t)nx * ty;
#pragma unroll
    for (int n = 1; n <= 4; ++n) {
      xo[k][n - 1] = ty * nx + wrapi(tx + n, nx);
      xo[k][3 + n] = ty * nx + wrapi(tx - n, nx);
      yo[k][n - 1] = wrapi(ty + n, ny) * nx + tx;
      yo[k][3 + n] = wrapi(ty - n, ny) * nx + tx;
    }
    // DMA sources: W = 1 the lane's own point; W = 2 (and V) points 32 kk + lane/2 of the wave's chunk
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const size_t p = pofs(64 * wave + k * BS + 32 * kk + (lane >> 1));
      toff[k][kk] = WI == 1 ? col[k] : p;
      voff[k][kk] = 2 * p + (lane & 1);
    }
  }
  const double *Vb = a.V + (size_t)ispin * gplane * nz;
  const unsigned tileA = __builtin_amdgcn_readfirstlane(lds_addr(tileR) + EB * 64u * wave);
  const unsigned vA = __builtin_amdgcn_readfirstlane(lds_addr(vR) + 8u * 64u * wave);
  auto dma_tile = [&](int plane, int slot) {
    const TI *src = in + zs * wrapi(plane, nz);
#pragma unroll
    for (int k = 0; k < PY; ++k) dma_chunk<TI>(src, toff[k], tileA + EB * (unsigned)(SL * slot + k * BS), lane);
  };
  auto dma_v = [&](int plane, int slot) {
    const float *vb = (const float *)Vb + 2 * gplane * wrapi(plane, nz);
#pragma unroll
    for (int k = 0; k < PY; ++k) {
      const unsigned m0 = vA + 8u * (unsigned)(SL * slot + k * BS);
      dma4(vb + voff[k][0], m0);
      dma4(vb + voff[k][1], m0 + 256u);
    }
  };
  const double *kp = a.kpar + 16 * ik;
  const R klap0 = (R)kp[0];
  R nab[12], lap[12];
#pragma unroll
  for (int i = 0; i < 12; ++i) {
    nab[i] = (R)kp[1 + i];
    lap[i] = (R)a.lap[i];
  }

  // prologue: queues of planes z0-4 .. z0+3 (plain loads), rings for planes z0 .. z0+3+D
  CH q[PY][9];
#pragma unroll
  for (int k = 0; k < PY; ++k)
#pragma unroll
    for (int i = 0; i < 8; ++i) q[k][i] = cvt2<CH>(in[col[k] + zs * wrapi(z0 - 4 + i, nz)]);
  __builtin_amdgcn_s_waitcnt(0);
  for (int p = 0; p < 4 + D; ++p) dma_tile(z0 + p, (z0 + p) % kRingT);
  for (int p = 0; p < D; ++p) dma_v(z0 + p, (z0 + p) % kRingH);
  wait_vm<0>();

  int sT = z0 % kRingT, sH = z0 % kRingH;
  for (int z = z0; z < z1; ++z) {
    wait_vm<(D - 1) * kOps>();
    __syncthreads();
    // past the chunk's last needed plane the look-ahead re-reads that plane into a slot never read
    dma_tile(min(z + 4 + D, z1 + 3), (sT + 4 + D) % kRingT);
    dma_v(min(z + D, z1 - 1), (sH + D) % kRingH);
    const TI *T = tileR + SL * sT;
    const TI *T4 = tileR + SL * ((sT + 4) % kRingT);
    const double *Vs = vR + SL * sH;
#pragma unroll
    for (int k = 0; k < PY; ++k) {
      q[k][8] = cvt2<CH>(T4[te[k]]);
      CH v, w;
      {
        const CH p1 = cvt2<CH>(T[xo[k][0]]), p2 = cvt2<CH>(T[xo[k][1]]), p3 = cvt2<CH>(T[xo[k][2]]),
                 p4 = cvt2<CH>(T[xo[k][3]]);
        const CH m1 = cvt2<CH>(T[xo[k][4]]), m2 = cvt2<CH>(T[xo[k][5]]), m3 = cvt2<CH>(T[xo[k][6]]),
                 m4 = cvt2<CH>(T[xo[k][7]]);
        v.x = lap[0] * (p1.x + m1.x) + lap[1] * (p2.x + m2.x) + lap[2] * (p3.x + m3.x) + lap[3] * (p4.x + m4.x);
        v.y = lap[0] * (p1.y + m1.y) + lap[1] * (p2.y + m2.y) + lap[2] * (p3.y + m3.y) + lap[3] * (p4.y + m4.y);
        w.x = nab[0] * (p1.x - m1.x) + nab[1] * (p2.x - m2.x) + nab[2] * (p3.x - m3.x) + nab[3] * (p4.x - m4.x);
        w.y = nab[0] * (p1.y - m1.y) + nab[1] * (p2.y - m2.y) + nab[2] * (p3.y - m3.y) + nab[3] * (p4.y - m4.y);
      }
      {
        const CH p1 = cvt2<CH>(T[yo[k][0]]), p2 = cvt2<CH>(T[yo[k][1]]), p3 = cvt2<CH>(T[yo[k][2]]),
                 p4 = cvt2<CH>(T[yo[k][3]]);
        const CH m1 = cvt2<CH>(T[yo[k][4]]), m2 = cvt2<CH>(T[yo[k][5]]), m3 = cvt2<CH>(T[yo[k][6]]),
                 m4 = cvt2<CH>(T[yo[k][7]]);
        v.x += lap[4] * (p1.x + m1.x) + lap[5] * (p2.x + m2.x) + lap[6] * (p3.x + m3.x) + lap[7] * (p4.x + m4.x);
        v.y += lap[4] * (p1.y + m1.y) + lap[5] * (p2.y + m2.y) + lap[6] * (p3.y + m3.y) + lap[7] * (p4.y + m4.y);
        w.x += nab[4] * (p1.x - m1.x) + nab[5] * (p2.x - m2.x) + nab[6] * (p3.x - m3.x) + nab[7] * (p4.x - m4.x);
        w.y += nab[4] * (p1.y - m1.y) + nab[5] * (p2.y - m2.y) + nab[6] * (p3.y - m3.y) + nab[7] * (p4.y - m4.y);
      }
      const CH *qq = q[k];
      v.x += lap[8] * (qq[5].x + qq[3].x) + lap[9] * (qq[6].x + qq[2].x) + lap[10] * (qq[7].x + qq[1].x) +
             lap[11] * (qq[8].x + qq[0].x);
      v.y += lap[8] * (qq[5].y + qq[3].y) + lap[9] * (qq[6].y + qq[2].y) + lap[10] * (qq[7].y + qq[1].y) +
             lap[11] * (qq[8].y + qq[0].y);
      w.x += nab[8] * (qq[5].x - qq[3].x) + nab[9] * (qq[6].x - qq[2].x) + nab[10] * (qq[7].x - qq[1].x) +
             nab[11] * (qq[8].x - qq[0].x);
      w.y += nab[8] * (qq[5].y - qq[3].y) + nab[9] * (qq[6].y - qq[2].y) + nab[10] * (qq[7].y - qq[1].y) +
             nab[11] * (qq[8].y - qq[0].y);
      const CH t = qq[4];
      const R vcur = (R)Vs[te[k]];
      CH hh;
      hh.x = (vcur * t.x + klap0 * t.x) - (R)0.5 * v.x + w.y;
      hh.y = (vcur * t.y + klap0 * t.y) - (R)0.5 * v.y - w.x;
      TO *dst = act[k] ? (TO *)a.hout + orbOff + col[k] + zs * z : (TO *)a.sink + tid + k * BS;
      *dst = cvt2<TO>(hh);
#pragma unroll
      for (int i = 0; i < 8; ++i) q[k][i] = q[k][i + 1];
    }
    sT = (sT + 1 == kRingT) ? 0 : sT + 1;
    sH = (sH + 1 == kRingH) ? 0 : sH + 1;
  }
  wait_vm<0>();
}

// ---------------------------------------------------------------------------
// Terms without the Taylor sum on 256-point y-tiles (TY rows, 4 + 4 halo rows, nx <= 32),
// with every LDS address fixed at compile time: one ring slot holds a plane's TY + 8 rows
// (tile and halo together, so y neighbours are row offsets in one slot), the ring has 8
// slots and the z loop is unrolled by 8, so slot offsets become immediate offsets of the
// LDS reads; z neighbours above come from the ring, those below from a 4-deep register
// queue whose rotation is resolved by the unrolling (no moves).  Issue order per plane and
// wave: the tile DMAs of plane z+7 (NCH x W, or with PR ceil(NCH/2) paired dwordx4 ones), the V
// DMAs of plane z+3 (2 dword, or with PR 1 dwordx4), 1 store; the wait at the top of a plane
// leaves the last two planes' operations in flight.  Needs TZ % 8 == 0.
// Used for the middle terms of the mixed chain (instruction-issue bound): the pair sums of
// the x, y and z neighbours go into one fused multiply-add chain per component, a regrouping
// of stencil_tile's sum that saves two instructions per component.
// ---------------------------------------------------------------------------
template <int P> struct Ph { static constexpr int v = P; };

template <typename TI, typename R, typename TO, int NCH, bool PR>
__device__ __forceinline__ void stencil_tile8(const StencilArgs &a, int bid, double2 *lds) {
  using CH = typename Cx<R>::T;
  constexpr int BS = kTile;
  constexpr int WI = DmaW<TI>::W;
  constexpr unsigned EB = sizeof(TI);
  constexpr int SLOT = NCH * BS;              // elements per slot: (TY + 8) * nx <= NCH * 256
  // PR (FP32 elements, rows of even length): the wave's 64 NCH slot elements move by paired dwordx4
  // DMAs (lane l: elements 2l and 2l + 1 of a 128-element piece, one row, 16-byte aligned), one
  // instruction for NCH = 2 and two for NCH = 3 (the second on lanes < 32), and the V of its 64
  // points by one more (lanes < 32: points 64 w + 2l, 2l + 1)
  constexpr bool X4 = PR;
  static_assert(!PR || WI == 2, "paired DMAs move FP32 elements");
  constexpr int NT4 = (NCH + 1) / 2;
  constexpr int kOps = X4 ? NT4 + 1 + 1 : NCH * WI + 2 + 1;
  TI *tileR = (TI *)lds;                      // 8 x SLOT
  double *vR = (double *)(tileR + 8 * SLOT);  // 4 x BS

  const int ytile = bid % a.nyt;
  const int zt = (bid / a.nyt) % a.nzt;
  const int b = bid / (a.nyt * a.nzt);
  const int ik = b / a.nb;
  const int ispin = b % a.nspin;
  const int nx = a.nx, ny = a.ny, nz = a.nz, ly = a.ly;
  const int TY = a.TY;
  const int y0 = ytile * TY;
  const int z0 = zt * a.TZ;
  const int z1 = min(z0 + a.TZ, nz);
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int ntile = TY * nx;
  const bool active = tid < ntile;
  const int te = active ? tid : 0;
  const int tx = te % nx, ty = te / nx;
  const int y = y0 + ty;
  const bool outY = active && y < ny;
  const size_t zs = (size_t)nx * ly;
  const size_t orbOff = (size_t)b * a.osz;
  const TI *in = (const TI *)a.in + orbOff;
  const size_t colOff = (size_t)tx + (size_t)nx * wrapi(y, ny);
  const size_t gplane = (size_t)nx * ny;
  const int nslot = (TY + 8) * nx;
  // slot element e -> in-plane source offset (row r = global row y0 - 4 + r)
  auto sofs = [&](int e) {
    const int ec = e < nslot ? e : 0;
    return (size_t)(ec % nx) + (size_t)nx * wrapi(y0 - 4 + ec / nx, ny);
  };
  size_t toff[NCH][2];
#pragma unroll
  for (int k = 0; k < NCH; ++k)
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
      toff[k][kk] = sofs(64 * (wave + 4 * k) + (WI == 1 ? lane : 32 * kk + (lane >> 1)));
  size_t voff[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    const int e = 64 * wave + 32 * kk + (lane >> 1);
    const int ec = e < ntile ? e : 0;
    voff[kk] = 2 * ((size_t)(ec % nx) + (size_t)nx * wrapi(y0 + ec / nx, ny)) + (lane & 1);
  }
  size_t toff4[2] = {0, 0}, voff4 = 0;
  if (X4) {
#pragma unroll
    for (int i = 0; i < NT4; ++i) toff4[i] = sofs(64 * NCH * wave + 128 * i + 2 * lane);
    const int e = 64 * wave + 2 * (lane & 31);
    const int ec = e < ntile ? e : 0;
    voff4 = (size_t)(ec % nx) + (size_t)nx * wrapi(y0 + ec / nx, ny);
  }
  const double *Vb = a.V + (size_t)ispin * gplane * nz;
  const unsigned tileA = __builtin_amdgcn_readfirstlane(lds_addr(tileR) + EB * (X4 ? 64u * NCH : 64u) * wave);
  const unsigned vA = __builtin_amdgcn_readfirstlane(lds_addr(vR) + 8u * 64u * wave);
  auto dma_tile = [&](int plane, int slot) {
    const TI *src = in + zs * wrapi(plane, nz);
    if constexpr (X4) {
      dma16(src + toff4[0], tileA + EB * (unsigned)(SLOT * slot));
      if constexpr (NT4 > 1) {
        if (lane < 32) dma16(src + toff4[1], tileA + EB * (unsigned)(SLOT * slot + 128));
      }
    } else {
#pragma unroll
      for (int k = 0; k < NCH; ++k) dma_chunk<TI>(src, toff[k], tileA + EB * (unsigned)(SLOT * slot + 4 * 64 * k), lane);
    }
  };
  auto dma_v = [&](int plane, int slot) {
    if constexpr (X4) {
      if (lane < 32) dma16(Vb + gplane * wrapi(plane, nz) + voff4, vA + 8u * BS * slot);
    } else {
      const float *vb = (const float *)Vb + 2 * gplane * wrapi(plane, nz);
      dma4(vb + voff[0], vA + 8u * BS * slot);
      dma4(vb + voff[1], vA + 8u * BS * slot + 256u);
    }
  };
  // element indices in a slot: own point, x and y neighbours
  const int own = (ty + 4) * nx + tx;
  int xo[8], yo[8];
#pragma unroll
  for (int n = 1; n <= 4; ++n) {
    xo[n - 1] = (ty + 4) * nx + wrapi(tx + n, nx);
    xo[3 + n] = (ty + 4) * nx + wrapi(tx - n, nx);
    yo[n - 1] = (ty + 4 + n) * nx + tx;
    yo[3 + n] = (ty + 4 - n) * nx + tx;
  }
  const double *kp = a.kpar + 16 * ik;
  const R klap0 = (R)kp[0];
  R nab[12], lap[12];
#pragma unroll
  for (int i = 0; i < 12; ++i) {
    nab[i] = (R)kp[1 + i];
    lap[i] = (R)a.lap[i];
  }
  CH q[4];  // planes z-4 .. z-1 at the own point; plane z-4+k sits in q[(phase + k) & 3]
#pragma unroll
  for (int i = 0; i < 4; ++i) q[i] = cvt2<CH>(in[colOff + zs * wrapi(z0 - 4 + i, nz)]);
  __builtin_amdgcn_s_waitcnt(0);
  for (int p = 0; p < 7; ++p) dma_tile(z0 + p, p);
  for (int p = 0; p < 3; ++p) dma_v(z0 + p, p);
  wait_vm<0>();

  auto body = [&](int z, auto ph) {
    constexpr int P = decltype(ph)::v;
    wait_vm<2 * kOps>();
    __syncthreads();
    dma_tile(min(z + 7, z1 + 3), (P + 7) & 7);
    dma_v(min(z + 3, z1 - 1), (P + 3) & 3);
    const TI *T = tileR + SLOT * P;
    // one accumulation chain per component (x, then y, then z pairs: 12 fused multiply-adds), then
    // hh = (V t + klap0 t) - v/2 + i w
    R vx, vy, wx, wy;
    {
      const CH p1 = cvt2<CH>(T[xo[0]]), p2 = cvt2<CH>(T[xo[1]]), p3 = cvt2<CH>(T[xo[2]]), p4 = cvt2<CH>(T[xo[3]]);
      const CH m1 = cvt2<CH>(T[xo[4]]), m2 = cvt2<CH>(T[xo[5]]), m3 = cvt2<CH>(T[xo[6]]), m4 = cvt2<CH>(T[xo[7]]);
      vx = lap[0] * (p1.x + m1.x);
      vy = lap[0] * (p1.y + m1.y);
      wx = nab[0] * (p1.x - m1.x);
      wy = nab[0] * (p1.y - m1.y);
      vx += lap[1] * (p2.x + m2.x); vy += lap[1] * (p2.y + m2.y); wx += nab[1] * (p2.x - m2.x); wy += nab[1] * (p2.y - m2.y);
      vx += lap[2] * (p3.x + m3.x); vy += lap[2] * (p3.y + m3.y); wx += nab[2] * (p3.x - m3.x); wy += nab[2] * (p3.y - m3.y);
      vx += lap[3] * (p4.x + m4.x); vy += lap[3] * (p4.y + m4.y); wx += nab[3] * (p4.x - m4.x); wy += nab[3] * (p4.y - m4.y);
    }
    {
      const CH p1 = cvt2<CH>(T[yo[0]]), p2 = cvt2<CH>(T[yo[1]]), p3 = cvt2<CH>(T[yo[2]]), p4 = cvt2<CH>(T[yo[3]]);
      const CH m1 = cvt2<CH>(T[yo[4]]), m2 = cvt2<CH>(T[yo[5]]), m3 = cvt2<CH>(T[yo[6]]), m4 = cvt2<CH>(T[yo[7]]);
      vx += lap[4] * (p1.x + m1.x); vy += lap[4] * (p1.y + m1.y); wx += nab[4] * (p1.x - m1.x); wy += nab[4] * (p1.y - m1.y);
      vx += lap[5] * (p2.x + m2.x); vy += lap[5] * (p2.y + m2.y); wx += nab[5] * (p2.x - m2.x); wy += nab[5] * (p2.y - m2.y);
      vx += lap[6] * (p3.x + m3.x); vy += lap[6] * (p3.y + m3.y); wx += nab[6] * (p3.x - m3.x); wy += nab[6] * (p3.y - m3.y);
      vx += lap[7] * (p4.x + m4.x); vy += lap[7] * (p4.y + m4.y); wx += nab[7] * (p4.x - m4.x); wy += nab[7] * (p4.y - m4.y);
    }
    const CH t = cvt2<CH>(T[own]);
    const CH u1 = cvt2<CH>(tileR[SLOT * ((P + 1) & 7) + own]), u2 = cvt2<CH>(tileR[SLOT * ((P + 2) & 7) + own]);
    const CH u3 = cvt2<CH>(tileR[SLOT * ((P + 3) & 7) + own]), u4 = cvt2<CH>(tileR[SLOT * ((P + 4) & 7) + own]);
    const CH d1 = q[(P + 3) & 3], d2 = q[(P + 2) & 3], d3 = q[(P + 1) & 3], d4 = q[P & 3];
    vx += lap[8] * (u1.x + d1.x); vy += lap[8] * (u1.y + d1.y); wx += nab[8] * (u1.x - d1.x); wy += nab[8] * (u1.y - d1.y);
    vx += lap[9] * (u2.x + d2.x); vy += lap[9] * (u2.y + d2.y); wx += nab[9] * (u2.x - d2.x); wy += nab[9] * (u2.y - d2.y);
    vx += lap[10] * (u3.x + d3.x); vy += lap[10] * (u3.y + d3.y); wx += nab[10] * (u3.x - d3.x); wy += nab[10] * (u3.y - d3.y);
    vx += lap[11] * (u4.x + d4.x); vy += lap[11] * (u4.y + d4.y); wx += nab[11] * (u4.x - d4.x); wy += nab[11] * (u4.y - d4.y);
    const R vcur = (R)vR[BS * (P & 3) + te];
    CH hh;
    hh.x = (vcur * t.x + klap0 * t.x) - (R)0.5 * vx + wy;
    hh.y = (vcur * t.y + klap0 * t.y) - (R)0.5 * vy - wx;
    TO *dst = outY ? (TO *)a.hout + orbOff + colOff + zs * z : (TO *)a.sink + tid;
    *dst = cvt2<TO>(hh);
    q[P & 3] = t;
  };
  for (int z = z0; z < z1; z += 8) {
    body(z, Ph<0>());
    body(z + 1, Ph<1>());
    body(z + 2, Ph<2>());
    body(z + 3, Ph<3>());
    body(z + 4, Ph<4>());
    body(z + 5, Ph<5>());
    body(z + 6, Ph<6>());
    body(z + 7, Ph<7>());
  }
  wait_vm<0>();
}

// ---------------------------------------------------------------------------
// The same terms with the z part of each output plane formed 4 planes late, so that a plane's
// LDS slot (tile and halo rows) is needed only while that plane is the current one: the ring
// has 4 slots (plane p read, p+1 and p+2 in flight, p+3 being written) and the block takes
// 40 KB of LDS in FP64 instead of 72 KB (four blocks per CU instead of two, twice the bytes in
// flight).  At plane p the kernel forms the x and y part and the centre term of plane p from
// the slot (kept in a 4-deep register queue), pushes p's own value into a 9-deep queue of own
// values (planes p-8 .. p) and completes plane p-4 with its z part.  The centre, x/y and z
// partial sums are added in that order (hh = ((V t + klap0 t) - v_xy/2 + i w_xy) - v_z/2 + i w_z),
// a regrouping of stencil_tile's sum.  Any number of planes: the z loop runs TZ + 4 planes
// (rounded up to 4), unrolled by 4 so that slot and queue indices are compile-time (a break per
// plane instead of the rounding cost 1% at 32^3).  A slot holds NCK chunks of 64 elements (8: rows of up to 32 points; 10: 13 rows of 48 points, so that the 48-point rows keep
// three blocks per CU; 12: up to 64 points); chunk c is moved by wave c % 4, and a wave with no
// chunk left for its last DMA of a plane moves its previous chunk again (the same data to the
// same place), so that every wave issues the same number of operations per plane.
// ---------------------------------------------------------------------------
// XT: tiles of TX x TY points with a halo on x too, for rows above 64 points (full rows would leave two
// or three of them per tile beside 8 halo rows).  HBM-bound; 96 x 14 x 12, 512 orbitals: 188 us with full
// rows (stencil_tile), 100 us so; the last term 244 and 174 us.
// NC >= 0 (FP64): the last term with the Taylor sum over NC earlier terms.  Their values at plane p - 4
// come two planes ahead through per-lane LDS slots (a wave reads only what it moved itself: no barrier).
// 32^3, 1024 orbitals: 593 us, 80 bytes a point at 4.5 TB/s (620 us in stencil_tile, one plane ahead).
template <typename TI, typename R, typename TO, int NCK, bool XT = false, int NC = -1>
__device__ __forceinline__ void stencil_tilez(const StencilArgs &a, int bid, double2 *lds) {
  using CH = typename Cx<R>::T;
  constexpr int BS = kTile;
  constexpr int WI = DmaW<TI>::W;
  constexpr unsigned EB = sizeof(TI);
  constexpr int SLOT = 64 * NCK;              // elements per slot: (TY + 8) * nx <= 64 NCK
  constexpr int NW = (NCK + 3) / 4;           // tile DMA chunks per wave and plane
  constexpr int NCB = NC > 0 ? NC : 0;
  static_assert(NC < 0 || std::is_same<TI, double2>::value, "the Taylor sum here is FP64");
  constexpr int kOps = NCB + NW * WI + 2 + 1;
  TI *tileR = (TI *)lds;                      // 4 x SLOT
  double *vR = (double *)(tileR + 4 * SLOT);  // 4 x BS
  double2 *combR = (double2 *)(vR + 4 * BS);  // 2 x NC x BS

  const int xtile = XT ? bid % a.nxt : 0;
  if (XT) bid /= a.nxt;
  const int ytile = bid % a.nyt;
  const int zt = (bid / a.nyt) % a.nzt;
  const int b = bid / (a.nyt * a.nzt);
  const int ik = b / a.nb;
  const int ispin = b % a.nspin;
  const int nx = a.nx, ny = a.ny, nz = a.nz, ly = a.ly;
  const int TY = a.TY;
  const int y0 = ytile * TY;
  const int z0 = zt * a.TZ;
  const int z1 = min(z0 + a.TZ, nz);
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int TX = XT ? a.TX : nx;           // points of a tile row
  const int SW = XT ? TX + 8 : nx;         // elements of a slot row
  const int x0 = xtile * TX;
  const int ntile = TY * TX;
  const bool active = tid < ntile;
  const int te = active ? tid : 0;
  const int tx = te % TX, ty = te / TX;
  const int y = y0 + ty;
  const bool outY = active && y < ny && (!XT || x0 + tx < nx);
  const size_t zs = (size_t)nx * ly;
  const size_t orbOff = (size_t)b * a.osz;
  const TI *in = (const TI *)a.in + orbOff;
  const size_t colOff = (size_t)(XT ? wrapi(x0 + tx, nx) : tx) + (size_t)nx * wrapi(y, ny);
  const size_t gplane = (size_t)nx * ny;
  const int nslot = (TY + 8) * SW;
  auto sofs = [&](int e) {
    const int ec = e < nslot ? e : 0;
    const int ex = XT ? wrapi(x0 - 4 + ec % SW, nx) : ec % SW;
    return (size_t)ex + (size_t)nx * wrapi(y0 - 4 + ec / SW, ny);
  };
  size_t toff[NW][2];
  unsigned kofs[NW];  // slot offset (elements) of the chunk of this wave's k-th DMA, wave-uniform
#pragma unroll
  for (int k = 0; k < NW; ++k) {
    const int kc = wave + 4 * k < NCK ? k : k - 1;
    kofs[k] = __builtin_amdgcn_readfirstlane(256u * (unsigned)kc);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
      toff[k][kk] = sofs(64 * (wave + 4 * kc) + (WI == 1 ? lane : 32 * kk + (lane >> 1)));
  }
  size_t voff[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    const int e = 64 * wave + 32 * kk + (lane >> 1);
    const int ec = e < ntile ? e : 0;
    const int ex = XT ? wrapi(x0 + ec % TX, nx) : ec % TX;
    voff[kk] = 2 * ((size_t)ex + (size_t)nx * wrapi(y0 + ec / TX, ny)) + (lane & 1);
  }
  const double *Vb = a.V + (size_t)ispin * gplane * nz;
  const unsigned tileA = __builtin_amdgcn_readfirstlane(lds_addr(tileR) + EB * 64u * wave);
  const unsigned vA = __builtin_amdgcn_readfirstlane(lds_addr(vR) + 8u * 64u * wave);
  auto dma_tile = [&](int plane, int slot) {
    const TI *src = in + zs * wrapi(plane, nz);
#pragma unroll
    for (int k = 0; k < NW; ++k) dma_chunk<TI>(src, toff[k], tileA + EB * (unsigned)(SLOT * slot) + EB * kofs[k], lane);
  };
  auto dma_v = [&](int plane, int slot) {
    const float *vb = (const float *)Vb + 2 * gplane * wrapi(plane, nz);
    dma4(vb + voff[0], vA + 8u * BS * slot);
    dma4(vb + voff[1], vA + 8u * BS * slot + 256u);
  };
  const unsigned combA = __builtin_amdgcn_readfirstlane(lds_addr(combR) + 16u * 64u * wave);
  auto dma_comb = [&](int plane, int slot) {
    const size_t at = orbOff + colOff + zs * plane;
#pragma unroll
    for (int n = 0; n < NCB; ++n) dma16((const double2 *)a.comb[n] + at, combA + 16u * BS * (NCB * slot + n));
  };
  const int own = (ty + 4) * SW + tx + (XT ? 4 : 0);
  int xo[8], yo[8];
#pragma unroll
  for (int n = 1; n <= 4; ++n) {
    xo[n - 1] = XT ? own + n : (ty + 4) * nx + wrapi(tx + n, nx);
    xo[3 + n] = XT ? own - n : (ty + 4) * nx + wrapi(tx - n, nx);
    yo[n - 1] = own + n * SW;
    yo[3 + n] = own - n * SW;
  }
  const double *kp = a.kpar + 16 * ik;
  const R klap0 = (R)kp[0];
  R nab[12], lap[12];
#pragma unroll
  for (int i = 0; i < 12; ++i) {
    nab[i] = (R)kp[1 + i];
    lap[i] = (R)a.lap[i];
  }
  CH q[9];   // own values of planes p-8 .. p (q[8] = p) after the push at plane p
  CH hq[4];  // centre + x/y part of planes p-3 .. p; plane p's sits in hq[(p - z0) & 3]
  // With the whole column in one chunk the planes past its end are its own first four planes
  // (periodic z), whose own values are kept from the first pass: the tail needs only those
  // (no x/y part is formed there), so it fetches nothing from HBM (its slot DMAs re-read the
  // last plane, an L2 hit, to keep the per-plane memory-op count fixed).
  const bool wrapkeep = a.nzt == 1 && nz % 4 == 0;  // the slot of a tail plane is then its own index
  CH keep[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    q[i] = cvt2<CH>(make_double2(0.0, 0.0));
    hq[i] = q[i];
    keep[i] = q[i];
    q[5 + i] = cvt2<CH>(in[colOff + zs * wrapi(z0 - 4 + i, nz)]);
  }
  q[4] = q[0];
  __builtin_amdgcn_s_waitcnt(0);
  for (int p = 0; p < 3; ++p) {
    dma_tile(z0 + p, p);
    dma_v(z0 + p, p);
  }
  wait_vm<0>();

  auto body = [&](int p, auto ph) {
    constexpr int P = decltype(ph)::v;
    wait_vm<2 * kOps - NCB>();
    __syncthreads();
    // the sum's values of plane p - 4, then its slot's next ones (plane p - 2)
    double2 cc[NCB > 0 ? NCB : 1];
    if constexpr (NCB > 0) {
#pragma unroll
      for (int n = 0; n < NCB; ++n) cc[n] = combR[BS * (NCB * (P & 1) + n) + tid];
#pragma unroll
      for (int n = 0; n < NCB; ++n) asm volatile("" : "+v"(cc[n].x), "+v"(cc[n].y)::"memory");
      dma_comb(min(max(p - 2, z0), z1 - 1), P & 1);
    }
    dma_tile(p + 3 < z1 ? p + 3 : (wrapkeep ? z1 - 1 : min(p + 3, z1 + 3)), (P + 3) & 3);
    dma_v(min(p + 3, z1 - 1), (P + 3) & 3);
    const TI *T = tileR + SLOT * P;
#pragma unroll
    for (int i = 0; i < 8; ++i) q[i] = q[i + 1];
    // in the tail of a whole-column chunk p = z1 + P wraps to plane P (z0 = 0, nz % 4 == 0)
    q[8] = (wrapkeep && p >= z1) ? keep[P] : cvt2<CH>(T[own]);
    if (p < z0 + 4) keep[P] = q[8];
    const CH hp = hq[P];  // plane p - 4
    if (p < z1) {
      CH v, w;
      {
        const CH p1 = cvt2<CH>(T[xo[0]]), p2 = cvt2<CH>(T[xo[1]]), p3 = cvt2<CH>(T[xo[2]]), p4 = cvt2<CH>(T[xo[3]]);
        const CH m1 = cvt2<CH>(T[xo[4]]), m2 = cvt2<CH>(T[xo[5]]), m3 = cvt2<CH>(T[xo[6]]), m4 = cvt2<CH>(T[xo[7]]);
        v.x = lap[0] * (p1.x + m1.x) + lap[1] * (p2.x + m2.x) + lap[2] * (p3.x + m3.x) + lap[3] * (p4.x + m4.x);
        v.y = lap[0] * (p1.y + m1.y) + lap[1] * (p2.y + m2.y) + lap[2] * (p3.y + m3.y) + lap[3] * (p4.y + m4.y);
        w.x = nab[0] * (p1.x - m1.x) + nab[1] * (p2.x - m2.x) + nab[2] * (p3.x - m3.x) + nab[3] * (p4.x - m4.x);
        w.y = nab[0] * (p1.y - m1.y) + nab[1] * (p2.y - m2.y) + nab[2] * (p3.y - m3.y) + nab[3] * (p4.y - m4.y);
      }
      {
        const CH p1 = cvt2<CH>(T[yo[0]]), p2 = cvt2<CH>(T[yo[1]]), p3 = cvt2<CH>(T[yo[2]]), p4 = cvt2<CH>(T[yo[3]]);
        const CH m1 = cvt2<CH>(T[yo[4]]), m2 = cvt2<CH>(T[yo[5]]), m3 = cvt2<CH>(T[yo[6]]), m4 = cvt2<CH>(T[yo[7]]);
        v.x += lap[4] * (p1.x + m1.x) + lap[5] * (p2.x + m2.x) + lap[6] * (p3.x + m3.x) + lap[7] * (p4.x + m4.x);
        v.y += lap[4] * (p1.y + m1.y) + lap[5] * (p2.y + m2.y) + lap[6] * (p3.y + m3.y) + lap[7] * (p4.y + m4.y);
        w.x += nab[4] * (p1.x - m1.x) + nab[5] * (p2.x - m2.x) + nab[6] * (p3.x - m3.x) + nab[7] * (p4.x - m4.x);
        w.y += nab[4] * (p1.y - m1.y) + nab[5] * (p2.y - m2.y) + nab[6] * (p3.y - m3.y) + nab[7] * (p4.y - m4.y);
      }
      const CH t = q[8];
      const R vcur = (R)vR[BS * P + te];
      CH hc;
      hc.x = (vcur * t.x + klap0 * t.x) - (R)0.5 * v.x + w.y;
      hc.y = (vcur * t.y + klap0 * t.y) - (R)0.5 * v.y - w.x;
      hq[P] = hc;
    }
    CH v, w;
    v.x = lap[8] * (q[5].x + q[3].x) + lap[9] * (q[6].x + q[2].x) + lap[10] * (q[7].x + q[1].x) + lap[11] * (q[8].x + q[0].x);
    v.y = lap[8] * (q[5].y + q[3].y) + lap[9] * (q[6].y + q[2].y) + lap[10] * (q[7].y + q[1].y) + lap[11] * (q[8].y + q[0].y);
    w.x = nab[8] * (q[5].x - q[3].x) + nab[9] * (q[6].x - q[2].x) + nab[10] * (q[7].x - q[1].x) + nab[11] * (q[8].x - q[0].x);
    w.y = nab[8] * (q[5].y - q[3].y) + nab[9] * (q[6].y - q[2].y) + nab[10] * (q[7].y - q[1].y) + nab[11] * (q[8].y - q[0].y);
    CH hh;
    hh.x = hp.x - (R)0.5 * v.x + w.y;
    hh.y = hp.y - (R)0.5 * v.y - w.x;
    // every lane stores every plane (the vm count per plane is fixed): the first four planes of
    // the chunk, what the loop runs past its last one and lanes without a point go to the sink
    const bool outP = outY && (unsigned)(p - z0 - 4) < (unsigned)(z1 - z0);
    TO *dst = outP ? (TO *)a.hout + orbOff + colOff + zs * (p - 4) : (TO *)a.sink + tid;
    if constexpr (NC >= 0) {
      auto add = [](double2 &o, double2 zc, double2 v) {
        o.x = o.x + (zc.x * v.x - zc.y * v.y);
        o.y = o.y + (zc.x * v.y + zc.y * v.x);
      };
      double2 od = NC > 0 ? cc[0] : q[4];
#pragma unroll
      for (int n = 1; n < NC; ++n) add(od, a.zc[n - 1], cc[n]);
      if (NC > 0) add(od, a.zc[NC > 0 ? NC - 1 : 0], q[4]);
      add(od, a.zc[NC >= 0 ? NC : 0], hh);
      hh = od;
    }
    *dst = cvt2<TO>(hh);
  };
  for (int p = z0; p < z1 + 4; p += 4) {
    body(p, Ph<0>());
    body(p + 1, Ph<1>());
    body(p + 2, Ph<2>());
    body(p + 3, Ph<3>());
  }
  wait_vm<0>();
}

template <typename TI, typename R, typename TO, int NCK, bool XT, int NC>
__global__ __launch_bounds__(kTile) void k_stencilz(StencilArgs a) {
  extern __shared__ double2 lds[];
  if (a.skip && *a.skip) return;  // a device-side gate switched this launch off
  int bid = blockIdx.x;
  const int nfull = (a.nblk / 8) * 8;
  if (bid < nfull) bid = (bid % 8) * (a.nblk / 8) + bid / 8;  // XCD-aware tile order
  stencil_tilez<TI, R, TO, NCK, XT, NC>(a, bid, lds);
}

// Over many systems (the batched step): block b takes tile `tiles[b]` = (system index, tile index).  One
// tile per block: a persistent loop over tiles keeps 10 more registers live and its blocks end
// unevenly (8 systems, 12 to 36 points an axis: 94 us a term and 119 us the last, 85 and 110 us so).
template <typename TI, typename R, typename TO, int NCK, int NC>
__global__ __launch_bounds__(kTile) void k_stencilz_packed(const StencilArgs *__restrict__ sys,
                                                           const int2 *__restrict__ tiles) {
  extern __shared__ double2 lds[];
  const int2 tr = tiles[blockIdx.x];
  const int si = __builtin_amdgcn_readfirstlane(tr.x);
  const int bid = __builtin_amdgcn_readfirstlane(tr.y);
  const StencilArgs a = sys[si];
  stencil_tilez<TI, R, TO, NCK, false, NC>(a, bid, lds);
}

template <typename TI, typename R, typename TO, int NCH, bool PR>
__global__ __launch_bounds__(kTile) void k_stencil8(StencilArgs a) {
  extern __shared__ double2 lds[];
  if (a.skip && *a.skip) return;  // a device-side gate switched this launch off
  int bid = blockIdx.x;
  const int nfull = (a.nblk / 8) * 8;
  if (bid < nfull) bid = (bid % 8) * (a.nblk / 8) + bid / 8;  // XCD-aware tile order
  stencil_tile8<TI, R, TO, NCH, PR>(a, bid, lds);
}

template <typename TI, typename R, typename TO, int HC, int NC, int BS>
__global__ __launch_bounds__(BS) void k_stencil(StencilArgs a) {
  extern __shared__ double2 lds[];
  if (a.skip && *a.skip) return;  // a device-side gate switched this launch off
  int bid = blockIdx.x;
  const int nfull = (a.nblk / 8) * 8;
  if (bid < nfull) bid = (bid % 8) * (a.nblk / 8) + bid / 8;  // XCD-aware tile order
  stencil_tile<TI, R, TO, HC, NC, BS>(a, bid, lds);
}

template <typename TI, typename R, typename TO, int PY, int BS, int D>
__global__ __launch_bounds__(BS) void k_stencil_plane(StencilArgs a) {
  extern __shared__ double2 lds[];
  if (a.skip && *a.skip) return;  // a device-side gate switched this launch off
  int bid = blockIdx.x;
  const int nfull = (a.nblk / 8) * 8;
  if (bid < nfull) bid = (bid % 8) * (a.nblk / 8) + bid / 8;  // XCD-aware tile order
  stencil_plane<TI, R, TO, PY, BS, D>(a, bid, lds);
}

// Persistent form over many systems (the batched step): block b takes tiles b, b + grid, ...
// of `tiles` = (system index, tile index); all systems share the template shape.
template <typename TI, typename R, typename TO, int HC, int NC, int BS>
__global__ __launch_bounds__(BS) void k_stencil_packed(const StencilArgs *__restrict__ sys,
                                                       const int2 *__restrict__ tiles, int ntiles) {
  extern __shared__ double2 lds[];
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const int2 tr = tiles[t];
    // the tile entry is the same for the whole block: uniform indices let the descriptor come in
    // through scalar loads, once per tile
    const int si = __builtin_amdgcn_readfirstlane(tr.x);
    const int bid = __builtin_amdgcn_readfirstlane(tr.y);
    const StencilArgs a = sys[si];
    stencil_tile<TI, R, TO, HC, NC, BS>(a, bid, lds);
    __syncthreads();  // every wave is done with the LDS rings before the next tile's DMAs
  }
}

// ---------------------------------------------------------------------------
// KB term of hpsi at the sphere points only (zpseudo's scatter,
// nonlocal_potential.f90:370-378), as a deterministic per-point gather over
// the point -> (atom, j) inverse map, entries in ascending ilma:
//   hout(p) += s * sum_e sum_l c(ilma0_e + l) zekr(j_e, ilma0_e + l)
// with s = 1 (plain / intermediate terms) or s = c_N (last Taylor term).
// One thread per touched point and G orbitals of one k-point.  The kernel is
// bound by the latency of its dependent loads, so the per-point record
// (orbital-block offset, first entry, entry count, first entry's ilma0 | cnt)
// comes in one 16-byte load, and with CM > 0 an entry's projectors are loaded CM at a
// time (clamped to the entry's own, which are skipped in the sum, so the order of the
// additions is the sequential one).
// ---------------------------------------------------------------------------
// Orbitals per thread and projectors of an entry loaded together, per element type of the chain:
// FP64 <8, 4>, FP32 <4, 0> (the fastest of G in {4, 8}, CM in {0, 4} measured at 32^3 with 64 s+p
// atoms; with 9 projectors each, 96 x 14 x 12 and 512 orbitals, CM = 4 takes 51 us and CM = 0 56 us).
// Up to four orbitals with more than four projectors per atom take CM = 0: the clamped loads of CM = 4
// are G per projector whatever the orbital count (256 x 8 x 8, 128 atoms of 16 projectors, one orbital:
// 32 us, 11 us with CM = 0; 24 x 22 x 16, 8 atoms, 16 orbitals: 18 us, 31 us with CM = 0).
constexpr int kScatG = 8, kScatCM = 4;
constexpr bool scat_plain(int cmax, int nb) { return cmax > kScatCM && 2 * nb <= kScatG; }
constexpr int kScatG32 = 4, kScatCM32 = 0;

struct ScatterArgs {
  void *hout;             // double2, or float2 in the mixed-precision chain
  const double2 *c;       // (nb, nlma, nk), orbital fastest
  const double2 *zent;    // (cmax, nent, nk)
  const int4 *tp_info;    // (ntp) orbital-block offset, first entry, entry count, pt_lma of the first entry
  const int *pt_lma;      // (nent) ilma0 | cnt << 24
  double2 s;
  size_t osz;
  int ntp, nb, nlma, nent, cmax, ngrp;
  const int *skip;        // device flag: the launch does nothing when it is set (null: never)
};

template <typename TH, int G, int CM>
__device__ __forceinline__ void nl_scatter_body(const ScatterArgs &a, int bx, int by) {
  const int i = bx * kBlock + threadIdx.x;
  const int ik = by / a.ngrp;
  const int b0 = (by % a.ngrp) * G;
  if (i >= a.ntp) return;
  const int4 inf = a.tp_info[i];
  const int nob = min(G, a.nb - b0);
  // the read half of the read-modify-write is issued first and overlaps the KB sum
  TH *p = (TH *)a.hout + ((size_t)ik * a.nb + b0) * a.osz + inf.x;
  double2 old[G];
#pragma unroll
  for (int o = 0; o < G; ++o)
    if (o < nob) old[o] = cvt2<double2>(p[(size_t)o * a.osz]);
  const double2 *zb = a.zent + (size_t)ik * a.nent * a.cmax;
  const double2 *cb = a.c + (size_t)ik * a.nlma * a.nb + b0;
  double2 acc[G];
#pragma unroll
  for (int o = 0; o < G; ++o) acc[o] = make_double2(0.0, 0.0);
  int lc = inf.w;
  for (int q = 0; q < inf.z; ++q) {
    const int e = inf.y + q;
    if (q > 0) lc = a.pt_lma[e];
    const int ilma0 = lc & 0xffffff;
    const int cnt = lc >> 24;
    const double2 *ze = zb + (size_t)e * a.cmax;
    if (CM > 0) {
      for (int l0 = 0; l0 < cnt; l0 += CM) {
        double2 zv[CM > 0 ? CM : 1], cv[CM > 0 ? CM : 1][G];
#pragma unroll
        for (int l = 0; l < CM; ++l) {
          const int lx = min(l0 + l, cnt - 1);
          zv[l] = ze[lx];
#pragma unroll
          for (int o = 0; o < G; ++o) cv[l][o] = cb[(size_t)(ilma0 + lx) * a.nb + min(o, nob - 1)];
        }
#pragma unroll
        for (int l = 0; l < CM; ++l) {
          if (l0 + l < cnt) {
#pragma unroll
            for (int o = 0; o < G; ++o) {
              acc[o].x += cv[l][o].x * zv[l].x - cv[l][o].y * zv[l].y;
              acc[o].y += cv[l][o].x * zv[l].y + cv[l][o].y * zv[l].x;
            }
          }
        }
      }
    } else {
      for (int l = 0; l < cnt; ++l) {
        const double2 zvl = ze[l];
        const double2 *cl = cb + (size_t)(ilma0 + l) * a.nb;
#pragma unroll
        for (int o = 0; o < G; ++o) {
          if (o < nob) {
            const double2 c = cl[o];
            acc[o].x += c.x * zvl.x - c.y * zvl.y;
            acc[o].y += c.x * zvl.y + c.y * zvl.x;
          }
        }
      }
    }
  }
#pragma unroll
  for (int o = 0; o < G; ++o) {
    if (o < nob) {
      double2 v = old[o];
      v.x += a.s.x * acc[o].x - a.s.y * acc[o].y;
      v.y += a.s.x * acc[o].y + a.s.y * acc[o].x;
      p[(size_t)o * a.osz] = cvt2<TH>(v);
    }
  }
}

template <typename TH, int G, int CM>
__global__ __launch_bounds__(kBlock) void k_nl_scatter(ScatterArgs a) {
  if (a.skip && *a.skip) return;  // a device-side gate switched this launch off
  nl_scatter_body<TH, G, CM>(a, blockIdx.x, blockIdx.y);
}

// ---------------------------------------------------------------------------
// h += dv * psi over the orbital blocks (dv per point and spin; padding rows untouched):
// turns H_old psi into H_new psi when only V_local changed (salmon_hip_taylor_reuse).
// ---------------------------------------------------------------------------
template <typename TH>
__global__ __launch_bounds__(kBlock) void k_vshift(TH *h, const double2 *psi, const double *dv, size_t osz, int nx,
                                                   int ny, int ly, int nz, int nspin, size_t ntot, const int *skip) {
  if (skip && *skip) return;  // a device-side gate switched this launch off
  const size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= ntot) return;
  const size_t b = i / osz;
  const size_t r = i % osz;
  const int x = (int)(r % nx);
  const int y = (int)((r / nx) % ly);
  const int z = (int)(r / ((size_t)nx * ly));
  if (y >= ny || z >= nz) return;
  const int ispin = (int)(b % nspin);
  const double d = dv[(size_t)ispin * nx * ny * nz + x + (size_t)nx * (y + (size_t)ny * z)];
  const double2 p = psi[i];
  double2 v = cvt2<double2>(h[i]);
  v.x += d * p.x;
  v.y += d * p.y;
  h[i] = cvt2<TH>(v);
}

// ---------------------------------------------------------------------------
// Density: rho(p) = sum_{ik, io} (|psi|^2 rocc) wtk, orbitals in (ik, io) order,
// in groups of gsz (kDensGroup by default) summed in order, groups combined in order.
// ---------------------------------------------------------------------------
struct DensArgs {
  const double2 *psi;
  const double *rocc;   // (no, nk, nspin)
  const double *wtk;
  double *part;         // (ngrid, nspin, ngrp)
  double *rho;          // (ngrid, nspin)
  size_t osz;
  int nx, ny, nz, ly, nspin, no, nk, ngrp, gsz;
  const int *skip;      // device flag: the launch does nothing when it is set (null: never)
};

__device__ __forceinline__ void density_part_body(const DensArgs &a, int bx, int grp, int ispin) {
  const size_t ngrid = (size_t)a.nx * a.ny * a.nz;
  const size_t g = (size_t)bx * kBlock + threadIdx.x;
  if (g >= ngrid) return;
  const int x = g % a.nx;
  const int yz = g / a.nx;
  const int y = yz % a.ny;
  const int z = yz / a.ny;
  const size_t off = (size_t)x + (size_t)a.nx * ((size_t)y + (size_t)a.ly * z);
  const int M = a.no * a.nk;
  const int m0 = grp * a.gsz, m1 = min(M, m0 + a.gsz);
  const double2 *pb = a.psi + off;
  const size_t bstride = (size_t)a.nspin * a.osz;  // one orbital to the next
  const double *occ = a.rocc + (size_t)a.no * a.nk * ispin;
  int io = m0 % a.no, ik = m0 / a.no;
  double acc = 0.0;
  int mm = m0;
  // U orbitals' loads in flight before the in-order sum consumes them
  constexpr int U = 8;
  for (; mm + U <= m1; mm += U) {
    double2 p[U];
#pragma unroll
    for (int u = 0; u < U; ++u) p[u] = pb[((size_t)ispin * a.osz) + (size_t)(mm + u) * bstride];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const double w2 = p[u].x * p[u].x + p[u].y * p[u].y;
      acc = acc + (w2 * occ[io + (size_t)a.no * ik]) * a.wtk[ik];
      if (++io == a.no) { io = 0; ++ik; }
    }
  }
  for (; mm < m1; ++mm) {
    const double2 p = pb[((size_t)ispin * a.osz) + (size_t)mm * bstride];
    const double w2 = p.x * p.x + p.y * p.y;
    acc = acc + (w2 * occ[io + (size_t)a.no * ik]) * a.wtk[ik];
    if (++io == a.no) { io = 0; ++ik; }
  }
  if (a.ngrp == 1)
    a.rho[g + ngrid * ispin] = acc;
  else
    a.part[g + ngrid * ((size_t)ispin + (size_t)a.nspin * grp)] = acc;
}

__global__ __launch_bounds__(kBlock) void k_density_part(DensArgs a) {
  if (a.skip && *a.skip) return;  // a device-side gate switched this launch off
  density_part_body(a, blockIdx.x, blockIdx.y, blockIdx.z);
}

// Partial sums of salmon_hip_density_noalloc: a file-scope device array (one copy per GPU,
// held until the process ends) in place of the handle's partial buffer.  Host code never
// passes its name to a kernel: the per-device address from hipGetSymbolAddress, resolved
// once per device when a handle is created there, is what the launches use.
constexpr size_t kNoAllocScratch = (size_t)8 << 20;  // doubles (64 MiB)
static __device__ __align__(256) double scratch[kNoAllocScratch];

__device__ __forceinline__ void density_sum_body(const DensArgs &a, int bx) {
  const size_t ngrid = (size_t)a.nx * a.ny * a.nz;
  const size_t i = (size_t)bx * kBlock + threadIdx.x;
  if (i >= ngrid * a.nspin) return;
  const size_t gs = ngrid * a.nspin;  // one group's partials to the next
  double acc = 0.0;
  int grp = 0;
  // 8 partials' loads in flight ahead of the in-order sum
  for (; grp + 8 <= a.ngrp; grp += 8) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = a.part[i + gs * (size_t)(grp + u)];
#pragma unroll
    for (int u = 0; u < 8; ++u) acc = acc + v[u];
  }
  for (; grp < a.ngrp; ++grp) acc = acc + a.part[i + gs * (size_t)grp];
  a.rho[i] = acc;
}

__global__ __launch_bounds__(kBlock) void k_density_sum(DensArgs a) {
  if (a.skip && *a.skip) return;  // a device-side gate switched this launch off
  density_sum_body(a, blockIdx.x);
}

// ---------------------------------------------------------------------------
// Current, local part (stencil_current, density_matrix.f90:465-530): per
// orbital sum |psi|^2 and Im sum_n (nab_n conj(psi)) psi(r + n e_d) over
// forward neighbours.  Block = full x rows x TY rows, streaming z over the
// whole column: z-forward neighbours from a 5-deep register queue, x and
// y-forward neighbours from an LDS plane carrying 4 extra rows below the tile.
// Each block writes its 4 partial sums (fixed-order tree) to part(4, tile, orbital).
// Bound by the rows read; in XCD order the tiles of one orbital share their halo rows' lines in one L2 (96 x 14
// x 12, 512 orbitals 76 us in launch order, 61 us so; 48^3, 1728 orbitals 868 and 831 us; full rows of 30 and 32
// points within 1 us, and no gain in the packed launch over many systems).
// ---------------------------------------------------------------------------
struct CurArgs {
  const double2 *psi;
  double *part;            // (4, nyt, norb)
  double coef_nab[12];
  size_t osz;
  int nx, ny, nz, ly, TY, nyt;
};

// f(integral_constant<int, I>) for I = 0, 1, ... in order while it returns true: a loop body
// whose iteration index is a compile-time constant (register-array slots stay registers).
template <int... I, typename F>
__device__ __forceinline__ void unroll_while(std::integer_sequence<int, I...>, F &&f) {
  (void)(f(std::integral_constant<int, I>{}) && ...);
}

__device__ __forceinline__ double block_sum(double v, double *sh) {
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int s = kBlock / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) sh[threadIdx.x] = sh[threadIdx.x] + sh[threadIdx.x + s];
    __syncthreads();
  }
  const double r = sh[0];
  __syncthreads();
  return r;
}

__device__ __forceinline__ void current_local_body(const CurArgs &a, int bid) {
  extern __shared__ double2 lds[];
  __shared__ double sh[kBlock];
  const int ytile = bid % a.nyt;
  const int b = bid / a.nyt;
  const int nx = a.nx, ny = a.ny, nz = a.nz, TY = a.TY;
  const int y0 = ytile * TY;
  const int tid = threadIdx.x;
  const bool active = tid < TY * nx;
  const int te = active ? tid : 0;
  const int tx = te % nx, ty = te / nx;
  const int y = y0 + ty;
  const bool own = active && y < ny;  // this lane's point belongs to the tile
  const int yw = wrapi(y, ny);
  const size_t zs = (size_t)nx * a.ly;
  const double2 *p = a.psi + (size_t)b * a.osz;
  const size_t col = (size_t)tx + (size_t)nx * yw;
  const int planeL = (TY + 4) * nx;
  // z neighbours: a register ring of R planes, plane z in slot z % R (the z loop is unrolled by R,
  // so every slot index is a constant and no register moves wait on a load); plane z + R - 1 is
  // loaded R - 5 iterations before its first use.  Halo: rows y0+TY .. y0+TY+3, 4*nx elements,
  // element e = tid + k * kBlock (k < nh <= 4, nx <= 256), loaded one plane ahead into a
  // two-deep register ring (R even: slot parity = plane parity).
  constexpr int R = 8;
  double2 q[R];
#pragma unroll
  for (int i = 0; i < R - 1; ++i) q[i] = p[col + zs * wrapi(i, nz)];
  const int nh = (4 * nx + kBlock - 1) / kBlock;
  int hoff[4];     // halo element k's offset within a plane (element 0's where the lane has none: loaded, unused)
  bool hown[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int e = tid + k * kBlock;
    hown[k] = k < nh && e < 4 * nx;
    const int ee = hown[k] ? e : 0;
    hoff[k] = ee % nx + nx * wrapi(y0 + TY + ee / nx, ny);
  }
  // halo rows of the even (hA*) and odd (hB*) planes; named registers, not arrays
  double2 hA0 = {}, hA1 = {}, hA2 = {}, hA3 = {}, hB0 = {}, hB1 = {}, hB2 = {}, hB3 = {};
  auto halo_get = [&](size_t zoff, double2 &v0, double2 &v1, double2 &v2, double2 &v3)
                      __attribute__((always_inline)) {
    v0 = p[(size_t)hoff[0] + zoff];
    if (nh > 1) v1 = p[(size_t)hoff[1] + zoff];
    if (nh > 2) v2 = p[(size_t)hoff[2] + zoff];
    if (nh > 3) v3 = p[(size_t)hoff[3] + zoff];
  };
  auto halo_put = [&](double2 *P, const double2 &v0, const double2 &v1, const double2 &v2, const double2 &v3)
                      __attribute__((always_inline)) {
    double2 *H = P + TY * nx + tid;
    if (hown[0]) H[0] = v0;
    if (hown[1]) H[kBlock] = v1;
    if (hown[2]) H[2 * kBlock] = v2;
    if (hown[3]) H[3 * kBlock] = v3;
  };
  halo_get(0, hA0, hA1, hA2, hA3);
  double r0 = 0.0, sx = 0.0, sy = 0.0, sz = 0.0;
  for (int z0 = 0; z0 < nz; z0 += R) {
    // plane z = z0 + u for the constants u = 0 .. R-1, while z < nz
    unroll_while(std::make_integer_sequence<int, R>{}, [&](auto uc) __attribute__((always_inline)) {
      constexpr int u = decltype(uc)::value;
      const int z = z0 + u;
      if (z >= nz) return false;
      double2 *P = lds + (u & 1) * planeL;
      if (active) P[ty * nx + tx] = q[u];
      const size_t zn = zs * wrapi(z + 1, nz);
      if constexpr ((u & 1) == 0) {
        halo_put(P, hA0, hA1, hA2, hA3);
        halo_get(zn, hB0, hB1, hB2, hB3);
      } else {
        halo_put(P, hB0, hB1, hB2, hB3);
        halo_get(zn, hA0, hA1, hA2, hA3);
      }
      q[(u + R - 1) % R] = p[col + zs * wrapi(z + R - 1, nz)];
      __syncthreads();
      if (own) {
        const double2 c = q[u];
        r0 += c.x * c.x + c.y * c.y;
        const double cr = c.x, ci = -c.y;
#pragma unroll
        for (int n = 1; n <= 4; ++n) {
          const double2 px = P[ty * nx + wrapi(tx + n, nx)];
          const double2 py = P[(ty + n) * nx + tx];
          const double2 pz = q[(u + n) % R];
          const double ax = a.coef_nab[n - 1] * cr, bx = a.coef_nab[n - 1] * ci;
          const double ay = a.coef_nab[3 + n] * cr, by = a.coef_nab[3 + n] * ci;
          const double az = a.coef_nab[7 + n] * cr, bz = a.coef_nab[7 + n] * ci;
          sx += ax * px.y + bx * px.x;
          sy += ay * py.y + by * py.x;
          sz += az * pz.y + bz * pz.x;
        }
      }
      return true;
    });
  }
  r0 = block_sum(r0, sh);
  sx = block_sum(sx, sh);
  sy = block_sum(sy, sh);
  sz = block_sum(sz, sh);
  if (tid == 0) {
    double *o = a.part + 4 * ((size_t)ytile + (size_t)a.nyt * b);
    o[0] = r0;
    o[1] = sx;
    o[2] = sy;
    o[3] = sz;
  }
}

__global__ __launch_bounds__(kBlock) void k_current_local(CurArgs a) {
  current_local_body(a, xcd_order(blockIdx.x, gridDim.x));
}

struct CurFinArgs {
  const double *part;      // (4, nslab, norb)
  const double2 *nl;       // (4, nlma, nb, nk) raw moments, or null
  const double *rinv;      // (nlma)
  const double *veck;      // (3, nk)
  const double *rocc;      // (no, nk, nspin)
  const double *wtk;       // (nk)
  double *contrib;         // (3, no*nk, nspin) scratch
  double *curr;            // (3, nspin)
  double ax, ay, az;
  const double *actab;     // with actab: vec_Ac = actab(:, *itt) (Ac_tot at the device step counter)
  const int *itt;
  int tmax;                // last row of actab (nt + 1); the step counter is clamped to 0..tmax
  double inv_ngrid;
  int nslab, nspin, no, nk, nlma;
};

// One wave per orbital (ik, io) of spin ispin: its weighted current
// ((j1 + j2) + jNL) rocc wtk (calc_current, density_matrix.f90:405-450), with
// jNL = 2 sum_lma Im(conj(uVpsi_r) uVpsi) (calc_current_nonlocal :532-591)
// reduced across the wave in a fixed tree.
__device__ __forceinline__ void current_orb_body(const CurFinArgs &a, int bx, int ispin) {
  const int M = a.no * a.nk;
  const int mm = bx * (kBlock / 64) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (mm >= M) return;
  const int io = mm % a.no, ik = mm / a.no;
  double jw[3] = {0.0, 0.0, 0.0};
  if (a.nl) {
    const int nb = a.no * a.nspin;
    const size_t ob = (size_t)ik * nb + (size_t)(ispin + a.nspin * io);
    for (int l = lane; l < a.nlma; l += 64) {
      const double2 *u4 = a.nl + (ob * a.nlma + l) * 4;
      const double rv = a.rinv[l];
      const double ur = u4[0].x * rv, ui = u4[0].y * rv;
      for (int d = 0; d < 3; ++d) jw[d] += u4[1 + d].x * ui - u4[1 + d].y * ur;
    }
    for (int d = 0; d < 3; ++d)
      for (int off = 32; off > 0; off >>= 1) jw[d] += __shfl_down(jw[d], off, 64);
  }
  if (lane == 0) {
    const size_t b = (size_t)ispin + (size_t)a.nspin * mm;
    double rt = 0.0, s[3] = {0.0, 0.0, 0.0};
    for (int sl = 0; sl < a.nslab; ++sl) {
      const double *o = a.part + 4 * ((size_t)sl + (size_t)a.nslab * b);
      rt = rt + o[0];
      s[0] = s[0] + o[1];
      s[1] = s[1] + o[2];
      s[2] = s[2] + o[3];
    }
    double A[3] = {a.ax, a.ay, a.az};
    if (a.actab) {
      const int t = min(max(*a.itt, 0), a.tmax);
      A[0] = a.actab[3 * t];
      A[1] = a.actab[3 * t + 1];
      A[2] = a.actab[3 * t + 2];
    }
    const double kA[3] = {a.veck[3 * ik] + A[0], a.veck[3 * ik + 1] + A[1], a.veck[3 * ik + 2] + A[2]};
    const double occ = a.rocc[io + (size_t)a.no * (ik + (size_t)a.nk * ispin)];
    for (int d = 0; d < 3; ++d) {
      const double j1 = kA[d] * rt;
      const double j2 = s[d] * 2.0;
      a.contrib[3 * ((size_t)mm + (size_t)M * ispin) + d] = (((j1 + j2) + jw[d] * 2.0) * occ) * a.wtk[ik];
    }
  }
}

__global__ __launch_bounds__(kBlock) void k_current_orb(CurFinArgs a, int ispin) { current_orb_body(a, blockIdx.x, ispin); }

// Sum of the orbital contributions divided by N_grid: one wave per component, lanes on every 64th
// orbital with 8 loads in flight, combined over the lanes in a fixed tree.
__device__ __forceinline__ void current_sum_body(const CurFinArgs &a, int ispin) {
  const int M = a.no * a.nk;
  const int d = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (d >= 3) return;
  const double *cs = a.contrib + 3 * (size_t)M * ispin + d;  // this spin's contributions
  double acc = 0.0;
  for (int m0 = lane; m0 < M; m0 += 64 * 8) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = m0 + 64 * u < M ? cs[3 * (size_t)(m0 + 64 * u)] : 0.0;
#pragma unroll
    for (int u = 0; u < 8; ++u) acc += v[u];
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if (lane == 0) a.curr[3 * ispin + d] = acc * a.inv_ngrid;
}

__global__ __launch_bounds__(kBlock) void k_current_sum(CurFinArgs a, int ispin) { current_sum_body(a, ispin); }

// ---------------------------------------------------------------------------
// Dipole: out[0:3] = -sum(pos_d rho) Hgs_d Hvol, out[3] = sum(rho) Hvol
// pos = i (odd n) or i - 1/2 (even n), i the 1-based grid index.
// ---------------------------------------------------------------------------
// Dipole moment and electron count (calc_dip / subdip, src/rt/dip.f90:114-225): per block a
// strided share of the points (32-bit indices), tree-reduced in LDS into part(4, block); the
// final kernel sums the block partials in block order.  Positions are the grid indices with
// the reference's half-cell shift on even extents.
constexpr int kDipBlocks = 128;

struct DipArgs {
  const double *rho;
  double *part, *out;    // part(4, kDipBlocks); out: dipole (3) and electron count
  int nx, ny, nz, nspin;
  double hx, hy, hz, hvol;
};

__device__ __forceinline__ void dipole_part_body(const DipArgs &a, int bx) {
  const double *rho = a.rho;
  double *part = a.part;
  const int nx = a.nx, ny = a.ny, nz = a.nz, nspin = a.nspin;
  __shared__ double sh[4][256];
  const int ngrid = nx * ny * nz;
  const double sx = (nx % 2 == 1) ? 1.0 : 0.5, sy = (ny % 2 == 1) ? 1.0 : 0.5, sz = (nz % 2 == 1) ? 1.0 : 0.5;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  for (int is = 0; is < nspin; ++is)
    for (int g = bx * 256 + threadIdx.x; g < ngrid; g += 256 * kDipBlocks) {
      const int x = g % nx;
      const int yz = g / nx;
      const int y = yz % ny;
      const int z = yz / ny;
      const double r = rho[(size_t)g + (size_t)ngrid * is];
      acc[0] += ((double)x + sx) * r;
      acc[1] += ((double)y + sy) * r;
      acc[2] += ((double)z + sz) * r;
      acc[3] += r;
    }
  for (int d = 0; d < 4; ++d) sh[d][threadIdx.x] = acc[d];
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s)
      for (int d = 0; d < 4; ++d) sh[d][threadIdx.x] = sh[d][threadIdx.x] + sh[d][threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x < 4) part[4 * bx + threadIdx.x] = sh[threadIdx.x][0];
}

__global__ __launch_bounds__(256) void k_dipole_part(DipArgs a) { dipole_part_body(a, blockIdx.x); }

// the final sum, on the first kDipBlocks threads of the block
__device__ __forceinline__ void dipole_sum_body(const DipArgs &a) {
  __shared__ double sh[4][kDipBlocks];
  const bool on = threadIdx.x < kDipBlocks;
  for (int d = 0; d < 4; ++d)
    if (on) sh[d][threadIdx.x] = a.part[4 * threadIdx.x + d];
  __syncthreads();
  for (int s = kDipBlocks / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s)
      for (int d = 0; d < 4; ++d) sh[d][threadIdx.x] = sh[d][threadIdx.x] + sh[d][threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    a.out[0] = -sh[0][0] * a.hx * a.hvol;
    a.out[1] = -sh[1][0] * a.hy * a.hvol;
    a.out[2] = -sh[2][0] * a.hz * a.hvol;
    a.out[3] = sh[3][0] * a.hvol;
  }
}

__global__ __launch_bounds__(256) void k_dipole_sum(DipArgs a) { dipole_sum_body(a); }

#include "small_grid.h"

// PZ81 LDA, unpolarised (exc_cor_pz / PZxc, src/xc/builtin_pz.f90:23-83), trho = rho.
__device__ __forceinline__ void pz_point(double rho, double &vxc, double &exc) {
  const double Pi = 3.141592653589793;
  const double gammaU = -0.1423, beta1U = 1.0529, beta2U = 0.3334, AU = 0.0311, BU = -0.048;
  const double CU = 0.002, DU = -0.0116;
  const double cst = 0.75 * pow(3.0 / (2.0 * Pi), 2.0 / 3.0);
  const double trho = 2.0 * (rho * 0.5);
  const double ttrho = trho + 1e-10;
  const double rs = pow(3.0 / (4 * Pi * ttrho), 1.0 / 3.0);
  double e = -cst / rs;
  double de = e / (3 * ttrho);
  if (rs > 1.0) {
    const double rssq = sqrt(rs);
    const double den = 1.0 + beta1U * rssq + beta2U * rs;
    e = e + gammaU / den;
    de = de + gammaU * (0.5 * beta1U * rssq + beta2U * rs) / (3 * ttrho) / (den * den);
  } else {
    const double rsln = log(rs);
    e = e + AU * rsln + BU + CU * rs * rsln + DU * rs;
    de = de - rs / (3 * ttrho) * (AU / rs + CU * (rsln + 1) + DU);
  }
  vxc = e + trho * de;
  exc = e;
}

// PZ81 LDA, spin-polarised (exc_cor_pz_sp / PZxc_sp, src/xc/builtin_pz_sp.f90:23-98) at one
// point from the two channel densities; terms in the order of the source's expressions.
__device__ __forceinline__ void pz_sp_point(double ru, double rd, double &vu, double &vd, double &exc) {
  const double Pi = 3.141592653589793;
  const double gammaU = -0.1423, gammaP = -0.0843;
  const double beta1U = 1.0529, beta2U = 0.3334, beta1P = 1.3981, beta2P = 0.2611;
  const double AU = 0.0311, BU = -0.048, CU = 0.002, DU = -0.0116;
  const double AP = 0.01555, BP = -0.0269, CP = 0.0007, DP = -0.0048;
  const double cx = 3.0 / 4.0 * pow(3.0 / (2 * Pi), 2.0 / 3.0);
  const double c13 = -pow(2.0, 1.0 / 3.0) + 1.0;
  const double fden = pow(2.0, 4.0 / 3.0) - 2.0;
  const double trho = ru + rd + 1e-20;
  const double tu = ru + 5e-21, td = rd + 5e-21;
  const double rs = pow(3.0 / (4.0 * Pi * trho), 1.0 / 3.0);
  const double zeta = (tu - td) / trho;
  const double sf = (pow(1.0 + zeta, 4.0 / 3.0) + pow(1.0 - zeta, 4.0 / 3.0) - 2.0) / fden;
  const double dsf = 4.0 / 3.0 * (pow(1.0 + zeta, 1.0 / 3.0) - pow(1.0 - zeta, 1.0 / 3.0)) / fden;
  double e = -cx / rs + c13 * cx / rs * sf;
  const double vs = e - 1.0 / 3.0 * cx / rs + 1.0 / 3.0 * c13 * cx / rs * sf;  // common to both channels
  double v0 = vs + c13 * cx / rs * (1.0 - zeta) * dsf;
  double v1 = vs + c13 * cx / rs * (-1.0 - zeta) * dsf;
  double ecu, ecp, vcu, vcp;
  if (rs > 1.0) {
    const double sq = sqrt(rs);
    const double du = 1.0 + beta1U * sq + beta2U * rs, dp = 1.0 + beta1P * sq + beta2P * rs;
    ecu = gammaU / du;
    ecp = gammaP / dp;
    vcu = gammaU * (1.0 + 7.0 / 6.0 * beta1U * sq + 4.0 / 3.0 * beta2U * rs) / (du * du);
    vcp = gammaP * (1.0 + 7.0 / 6.0 * beta1P * sq + 4.0 / 3.0 * beta2P * rs) / (dp * dp);
  } else {
    const double L = log(rs);
    ecu = AU * L + BU + CU * rs * L + DU * rs;
    ecp = AP * L + BP + CP * rs * L + DP * rs;
    vcu = AU * L + (BU - AU / 3.0) + 2.0 / 3.0 * CU * rs * L + (2.0 * DU - CU) / 3.0 * rs;
    vcp = AP * L + (BP - AP / 3.0) + 2.0 / 3.0 * CP * rs * L + (2.0 * DP - CP) / 3.0 * rs;
  }
  e = e + ecu + sf * (ecp - ecu);
  vu = v0 + vcu + sf * (vcp - vcu) + (ecp - ecu) * (1.0 - zeta) * dsf;
  vd = v1 + vcu + sf * (vcp - vcu) + (ecp - ecu) * (-1.0 - zeta) * dsf;
  exc = e;
}

// nspin = 1: rho, vxc (n); nspin = 2: rho_s, vxc_s (n, 2) channel-major; exc (n) or null
__global__ __launch_bounds__(256) void k_xc_pz(const double *rho, double *vxc, double *exc, size_t n, int nspin) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double e;
  if (nspin == 2) {
    double vu, vd;
    pz_sp_point(rho[i], rho[n + i], vu, vd, e);
    vxc[i] = vu;
    vxc[n + i] = vd;
  } else {
    double v;
    pz_point(rho[i], v, e);
    vxc[i] = v;
  }
  if (exc) exc[i] = e;
}

// update_vlocal (src/common/hamiltonian.f90:813-843): V(is) = Vpsl + Vh + Vxc(is), with Vxc
// either given or formed from rho on the fly (PZ, or spin-polarised PZ from the two channel
// densities); optionally the predictor-corrector average V(is) = (Vmix(is) + V(is))/2
// (src/rt/time_evolution_step.f90:404-409).  vpsl, vh: one channel; vxc, rho, vmix, V, vout:
// nspin channels of n points.
struct VlocArgs {
  const double *vpsl, *vh, *vxc, *rho, *vmix;
  double *V, *vout;
  size_t n;
  int nspin;
  const int *skip;    // device flag: the launch does nothing when it is set (null: never)
};

// V_local of point i from its Hartree potential
__device__ __forceinline__ void vlocal_point(const VlocArgs &a, size_t i, double vh) {
  double vx[2];
  if (a.rho) {
    double e;
    if (a.nspin == 2) pz_sp_point(a.rho[i], a.rho[a.n + i], vx[0], vx[1], e);
    else pz_point(a.rho[i], vx[0], e);
  } else {
    vx[0] = a.vxc[i];
    if (a.nspin == 2) vx[1] = a.vxc[a.n + i];
  }
  const double base = a.vpsl[i] + vh;
  for (int is = 0; is < a.nspin; ++is) {
    const size_t j = (size_t)is * a.n + i;
    double v = base + vx[is];
    if (a.vmix) v = 0.5 * (a.vmix[j] + v);
    a.V[j] = v;
    if (a.vout) a.vout[j] = v;
  }
}

__global__ __launch_bounds__(256) void k_update_vlocal(VlocArgs a) {
  if (a.skip && *a.skip) return;  // a device-side gate switched this launch off
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < a.n) vlocal_point(a, i, a.vh[i]);
}

// ---------------------------------------------------------------------------
// Hartree potential: poisson_ft (src/poisson/poisson_periodic.f90:23-242) as separable DFT passes in
// five launches: forward z, forward y, along x forward, times 4 pi/|G|^2/N and back in one, inverse y,
// inverse z.  The density is real, so only kz = 0 .. nz/2 is kept (the others are the conjugates), and
// the last pass can finish with V_local of its points instead of storing Vh.  A pass views the grid as
// columns of the transformed axis; a block stages COLS of them in LDS and folds them, u_j = x_j +
// x_{n-j} and v_j = x_j - x_{n-j}: with A = sum_j u_j cos(2 pi jk/n) and B = sum_j v_j sin(2 pi jk/n)
// over half the points, one thread has both X_k = A + i sg B and X_{n-k} = A - i sg B, a quarter of the
// plain sum's operations.  The n values exp(2 pi i m/n) are in LDS too, read at m = jk mod n.
//
// Bound by launch and LDS latency (a few thousand operations per thread's pair at most).  Measured, per
// potential update: seven launches with n x n twiddle tables gathered from memory took 75 us at
// 56x50x42 and 31 us at 12^3, these 29 us and 20 us.  256 threads (32 output pairs of 8 columns) beat
// 128 by a quarter at 56x50x42 (29 against 38 us): one round of pairs instead of two.
// ---------------------------------------------------------------------------
constexpr int kDftMaxN = 256;

struct DftArgs {
  const double *rho, *rho2;  // density, and the other spin channel's to be added (or null)
  const double2 *in;
  double2 *out;
  const double2 *tw;  // exp(2 pi i m / n), m = 0 .. n-1
  const double *coef;  // 4 pi/|G|^2 (nx, ny, nz)
  double *vh;          // Hartree potential, or null: finish with V_local (v)
  VlocArgs v;
  double rn;           // 1 / N_grid
  double sg;           // -1 forward, +1 inverse
  int n, inner, ncols; // transformed extent, its stride, columns
  const int *skip;     // device flag: the launch does nothing when it is set (null: never)
};

__device__ __forceinline__ double2 operator+(const double2 &a, const double2 &b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 operator-(const double2 &a, const double2 &b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 operator*(double a, const double2 &b) { return make_double2(a * b.x, a * b.y); }

// Columns of [n][COLS] in place: u_j at j, v_j at n - j (j = 1 .. (n-1)/2); ends with a barrier.
template <int COLS, int BS, typename T>
__device__ __forceinline__ void dft_fold(T *x, int n) {
  const int h = (n - 1) / 2;
  for (int t = threadIdx.x; t < h * COLS; t += BS) {
    const int j = 1 + t / COLS, cl = t % COLS;
    const T a = x[j * COLS + cl], b = x[(n - j) * COLS + cl];
    x[j * COLS + cl] = a + b;
    x[(n - j) * COLS + cl] = a - b;
  }
  __syncthreads();
}

// A and B of output pair k of folded column cl
template <int COLS, typename T>
__device__ __forceinline__ void dft_pair(const T *x, const double2 *tw, int n, int k, int cl, T &A, T &B) {
  const int h = (n - 1) / 2;
  A = x[cl];
  if (n % 2 == 0) A = k % 2 ? A - x[(n / 2) * COLS + cl] : A + x[(n / 2) * COLS + cl];
  B = 0.0 * x[cl];
  int m = 0;
#pragma unroll 4
  for (int j = 1; j <= h; ++j) {
    m += k;
    m -= m >= n ? n : 0;
    const double2 w = tw[m];
    A = A + w.x * x[j * COLS + cl];
    B = B + w.y * x[(n - j) * COLS + cl];
  }
}

__device__ __forceinline__ double2 times_i(double s, const double2 &b) { return make_double2(-s * b.y, s * b.x); }

// forward z of the real density: out[kz][column], kz = 0 .. n/2
template <int COLS>
__global__ __launch_bounds__(256) void k_dft_zr(DftArgs a) {
  constexpr int BS = 256;
  extern __shared__ double2 lds[];
  if (a.skip && *a.skip) return;  // a device-side gate switched this launch off
  double2 *tw = lds;
  double *x = (double *)(lds + a.n);  // [n][COLS]
  const int c0 = blockIdx.x * COLS;
  for (int t = threadIdx.x; t < a.n; t += BS) tw[t] = a.tw[t];
  for (int t = threadIdx.x; t < a.n * COLS; t += BS) {
    const int j = t / COLS, c = c0 + t % COLS;
    const size_t g = (size_t)j * a.inner + c;
    x[t] = c >= a.ncols ? 0.0 : a.rho2 ? a.rho[g] + a.rho2[g] : a.rho[g];
  }
  __syncthreads();
  dft_fold<COLS, BS>(x, a.n);
  const int cl = threadIdx.x % COLS;
  if (c0 + cl >= a.ncols) return;
  for (int k = threadIdx.x / COLS; k <= a.n / 2; k += BS / COLS) {
    double A, B;
    dft_pair<COLS>(x, tw, a.n, k, cl, A, B);
    a.out[(size_t)k * a.inner + c0 + cl] = make_double2(A, a.sg * B);
  }
}

// y pass: columns (kz, x)
template <int COLS>
__global__ __launch_bounds__(256) void k_dft_y(DftArgs a) {
  constexpr int BS = 256;
  extern __shared__ double2 lds[];
  if (a.skip && *a.skip) return;  // a device-side gate switched this launch off
  const int n = a.n;
  double2 *tw = lds, *x = lds + n;  // [n][COLS]
  const int cl = threadIdx.x % COLS, c = blockIdx.x * COLS + cl;
  const bool on = c < a.ncols;
  const int o = on ? c / a.inner : 0;
  const size_t g0 = (size_t)o * n * a.inner + (on ? c - o * a.inner : 0);
  for (int t = threadIdx.x; t < n; t += BS) tw[t] = a.tw[t];
  for (int j = threadIdx.x / COLS; j < n; j += BS / COLS) x[j * COLS + cl] = a.in[g0 + (size_t)j * a.inner];
  __syncthreads();
  dft_fold<COLS, BS>(x, n);
  if (!on) return;
  for (int k = threadIdx.x / COLS; k <= n / 2; k += BS / COLS) {
    double2 A, B;
    dft_pair<COLS>(x, tw, n, k, cl, A, B);
    const double2 iB = times_i(a.sg, B);
    a.out[g0 + (size_t)k * a.inner] = A + iB;
    if (k > 0 && 2 * k < n) a.out[g0 + (size_t)(n - k) * a.inner] = A - iB;
  }
}

// along x: forward, times coef / N, inverse, in place; columns are rows (ky, kz) of n points
template <int COLS>
__global__ __launch_bounds__(256) void k_dft_x(DftArgs a) {
  constexpr int BS = 256;
  extern __shared__ double2 lds[];
  if (a.skip && *a.skip) return;  // a device-side gate switched this launch off
  const int n = a.n;
  double2 *tw = lds, *x = lds + n, *y = x + n * COLS;  // [n][COLS] each
  const int c0 = blockIdx.x * COLS, ncl = min(COLS, a.ncols - c0);
  for (int t = threadIdx.x; t < n; t += BS) tw[t] = a.tw[t];
  for (int t = threadIdx.x; t < n * COLS; t += BS) {
    const int r = t / n, j = t - r * n;
    x[j * COLS + r] = r < ncl ? a.in[(size_t)(c0 + r) * n + j] : make_double2(0.0, 0.0);
  }
  __syncthreads();
  dft_fold<COLS, BS>(x, n);
  const int cl = threadIdx.x % COLS;
  const bool on = cl < ncl;
  const double *cf = a.coef + (size_t)(c0 + (on ? cl : 0)) * n;
  for (int k = threadIdx.x / COLS; k <= n / 2; k += BS / COLS) {
    const int kk = k > 0 && 2 * k < n ? n - k : k;
    const double f0 = a.rn * cf[k], f1 = a.rn * cf[kk];
    double2 A, B;
    dft_pair<COLS>(x, tw, n, k, cl, A, B);
    const double2 iB = times_i(-1.0, B);
    y[k * COLS + cl] = f0 * (A + iB);
    if (kk != k) y[kk * COLS + cl] = f1 * (A - iB);
  }
  __syncthreads();
  dft_fold<COLS, BS>(y, n);
  for (int k = threadIdx.x / COLS; k <= n / 2; k += BS / COLS) {
    double2 A, B;
    dft_pair<COLS>(y, tw, n, k, cl, A, B);
    const double2 iB = times_i(1.0, B);
    x[k * COLS + cl] = A + iB;
    if (k > 0 && 2 * k < n) x[(n - k) * COLS + cl] = A - iB;
  }
  __syncthreads();
  for (int t = threadIdx.x; t < n * ncl; t += BS) {
    const int r = t / n, j = t - r * n;
    a.out[(size_t)(c0 + r) * n + j] = x[j * COLS + r];
  }
}

// inverse z from kz = 0 .. n/2 to real values at z and n - z, which are Vh or end in V_local
template <int COLS>
__global__ __launch_bounds__(256) void k_dft_zi(DftArgs a) {
  constexpr int BS = 256;
  extern __shared__ double2 lds[];
  if (a.skip && *a.skip) return;  // a device-side gate switched this launch off
  const int n = a.n, h = (n - 1) / 2;
  double2 *tw = lds, *x = lds + n;  // [n/2 + 1][COLS]
  const int cl = threadIdx.x % COLS, c = blockIdx.x * COLS + cl;
  const bool on = c < a.ncols;
  for (int t = threadIdx.x; t < n; t += BS) tw[t] = a.tw[t];
  for (int k = threadIdx.x / COLS; k <= n / 2; k += BS / COLS)
    x[k * COLS + cl] = on ? a.in[(size_t)k * a.inner + c] : make_double2(0.0, 0.0);
  __syncthreads();
  if (!on) return;
  for (int z = threadIdx.x / COLS; z <= n / 2; z += BS / COLS) {
    double A = 0.0, B = 0.0;
    int m = 0;
#pragma unroll 4
    for (int k = 1; k <= h; ++k) {
      m += z;
      m -= m >= n ? n : 0;
      const double2 w = tw[m], v = x[k * COLS + cl];
      A += w.x * v.x;
      B += w.y * v.y;
    }
    A = x[cl].x + 2.0 * A;
    B = 2.0 * B;
    if (n % 2 == 0) A += z % 2 ? -x[(n / 2) * COLS + cl].x : x[(n / 2) * COLS + cl].x;
    const size_t g = (size_t)z * a.inner + c, gm = (size_t)(n - z) * a.inner + c;
    const bool two = z > 0 && 2 * z < n;
    if (a.vh) {
      a.vh[g] = A - B;
      if (two) a.vh[gm] = A + B;
    } else {
      vlocal_point(a.v, g, A - B);
      if (two) vlocal_point(a.v, gm, A + B);
    }
  }
}

// The aetrs propagator's potential extrapolation (src/rt/time_evolution_step.f90:432-445):
// V_new = 3 V - 3 V_old1 + V_old2, then V_old2 = V_old1, V_old1 = V, V = V_new, over all
// spin channels of the handle's potential.
__global__ __launch_bounds__(256) void k_vextrap(double *V, double *v1, double *v2, double *vout, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double v = V[i];
  const double vn = 3.0 * v - 3.0 * v1[i] + v2[i];
  v2[i] = v1[i];
  v1[i] = v;
  V[i] = vn;
  if (vout) vout[i] = vn;
}

// Streaming copy of n 16-byte elements (HBM ceiling of the box): dwordx4 loads and stores,
// non-temporal, four elements per thread in flight.
typedef unsigned int u4v __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(256) void k_stream_copy(u4v *__restrict__ dst, const u4v *__restrict__ src, size_t n) {
  const size_t stride = (size_t)gridDim.x * 256;
  size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  for (; i + 3 * stride < n; i += 4 * stride) {
    u4v v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = __builtin_nontemporal_load(src + i + k * stride);
#pragma unroll
    for (int k = 0; k < 4; ++k) __builtin_nontemporal_store(v[k], dst + i + k * stride);
  }
  for (; i < n; i += stride) __builtin_nontemporal_store(__builtin_nontemporal_load(src + i), dst + i);
}

// dst = src where the device flag is set (the accepted branch of a device-side gate)
__global__ __launch_bounds__(256) void k_copy_if(const int *flag, double *dst, const double *src, size_t n) {
  if (!*flag) return;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

template <typename T>
int dalloc(T **p, size_t n) {
  *p = nullptr;
  if (n == 0) return 0;
  hipError_t e = hipMalloc((void **)p, n * sizeof(T));
  if (e != hipSuccess) {
    *p = nullptr;
    return fail(SALMON_HIP_ENOMEM, "hipMalloc(%zu bytes): %s", n * sizeof(T), hipGetErrorString(e));
  }
  return 0;
}

template <typename T>
void dfree(T *&p) {
  if (p) (void)hipFree((void *)p);
  p = nullptr;
}

}  // namespace

struct salmon_hip_ctx {
  int nx = 0, ny = 0, nz = 0, ly = 0, nspin = 0, no = 0, nk = 0;
  int nb = 0, norb = 0;
  size_t osz = 0, ngrid = 0;
  double coef_lap[12] = {}, coef_nab[12] = {}, coef_lap0 = 0, hgs[3] = {}, hvol = 0;
  hipStream_t own = nullptr, stream = nullptr;
  // projections run on `side`, forked from and joined back into `stream` by events, so
  // that they overlap the stencil pass reading the same input
  hipStream_t side = nullptr;
  hipEvent_t ev_fork = nullptr, ev_join = nullptr;
  bool join_pending = false;
  bool overlap = false;  // salmon_hip_set_overlap
  bool have_V = false, have_k = false;
  double *d_veck = nullptr, *d_rocc = nullptr, *d_wtk = nullptr, *d_V = nullptr, *d_kpar = nullptr;
  // nonlocal
  int natom = 0, nps = 0, nlma = 0, nent = 0;
  int cmax = 0;
  double kbval = 0.0;  // projector values of an orbital: sum over atoms of sphere points x projectors
  int *d_mps = nullptr, *d_jidx = nullptr, *d_pt_off = nullptr;
  int *d_pt_lma = nullptr, *d_entof = nullptr;
  int4 *d_tp_info = nullptr;  // per touched point: orbital-block offset, first entry, entry count, its pt_lma
  int ntp = 0;
  // fused KB pass (k_proj_scatter): per sphere point its offset if one (atom, point) pair covers
  // it, else -1; the touched points with several pairs (completed by k_nl_scatter first)
  int *d_jexcl = nullptr;
  int4 *d_tp_shared = nullptr;
  int ntp_shared = 0;
  bool kb_fused = true;
  double2 *d_sink = nullptr;
  int2 *d_atom_lma = nullptr;
  double *d_rxyz = nullptr, *d_uv = nullptr, *d_rinv = nullptr;
  double2 *d_zekr = nullptr, *d_zent = nullptr, *d_c = nullptr, *d_curnl = nullptr;
  // salmon_hip_current_next: the next step's phase table built ahead into d_*_n (staged, for the
  // field staged_A) and the projection of that step's orbitals pre_psi under it left in d_c;
  // pre_state 1 = made, table not yet promoted; 2 = promoted by update_kvector(staged_A), d_c
  // holds c of pre_psi for its first Taylor term; 0 = none
  double2 *d_zekr_n = nullptr, *d_zent_n = nullptr;
  double *d_kpar_n = nullptr;
  bool staged = false;
  double staged_A[3] = {0.0, 0.0, 0.0};
  const void *pre_psi = nullptr;
  int pre_state = 0;
  bool in_batch = false;  // a batch's packed records hold this handle's table pointers
  double2 *d_c2 = nullptr;  // the fused pass writes the next term's c here; the two are then swapped
  // Taylor scratch: H^2 psi .. H^(N-2) psi (allocated on first use); FP32 chain h_1 .. h_{N-1}
  std::vector<double2 *> tscr;
  std::vector<float2 *> tscr32;
  int prec = SALMON_HIP_PREC_FP64;
  // observables scratch
  double *d_curpart = nullptr, *d_contrib = nullptr, *d_denspart = nullptr;
  double *d_scratch = nullptr;  // this device's copy of `scratch` (salmon_hip_density_noalloc)
  double *d_dippart = nullptr;  // dipole block partials (4 x kDipBlocks)
  int dens_ngrp = 1;
  // Hartree (salmon_hip_set_poisson): exp(2 pi i m/n) per axis, 4 pi/|G|^2 table, half-spectrum work grids
  bool have_cell = false;
  double2 *d_tw[3] = {nullptr, nullptr, nullptr};
  double *d_gcoef = nullptr;
  double2 *d_fft[2] = {nullptr, nullptr};
  // stencil launch shape
  int TY = 1, TZ = 1, nyt = 1, nzt = 1;
  // launch shape of the terms without the Taylor sum (salmon_hip_autotune): tile_plane -1 = rule
  // (whole plane when it fits 256 threads), 0 = y tiles, 1 = whole plane; mid_nzt 0 = rule
  int tile_plane = -1, mid_nzt = 0;
  bool tile8 = true;  // stencil_tile8 for the mixed middle terms where the shape allows it
  bool small_grid = true;  // k_taylor_small where the grid fits (salmon_hip_set_launch_shape turns it off)
  // salmon_hip_set_skip: device flag read by the launches of hpsi/taylor, density and the
  // potential update (they do nothing while it is set); null = none
  const int *d_skip = nullptr;
  // kernel timing (salmon_hip_prof_*): start/stop event pairs per launch
  bool prof = false;
  std::vector<hipEvent_t> ev;
  std::vector<int> ev_kind;
  size_t ev_used = 0;
};

// Events for one timed launch, or nullptr pair when timing is off / the pool is full.
static void prof_events(salmon_hip_ctx *c, int kind, hipEvent_t *s, hipEvent_t *e) {
  *s = nullptr;
  *e = nullptr;
  if (!c->prof || 2 * (c->ev_used + 1) > c->ev.size()) return;
  *s = c->ev[2 * c->ev_used];
  *e = c->ev[2 * c->ev_used + 1];
  c->ev_kind[c->ev_used] = kind;
  c->ev_used += 1;
}

static int check(salmon_hip_t h) {
  if (!h) return fail(SALMON_HIP_EINVAL, "null handle");
  return 0;
}

// Per-device address of `scratch`, resolved once per device with that device current.
constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static double *g_scratch_dev[kMaxDevices] = {};

static int resolve_scratch(double **out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return fail(SALMON_HIP_EHIP, "hipGetDevice failed or device %d beyond %d", dev, kMaxDevices);
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_dev[dev]) {
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
      return fail(SALMON_HIP_EHIP, "hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
    g_scratch_dev[dev] = (double *)ptr;
  }
  *out = g_scratch_dev[dev];
  return 0;
}

// Error text from the other translation units of the library (the predictor).
void salmon_hip_internal_error(const char *msg) { g_err = msg; }

extern "C" {

const char *salmon_hip_last_error(void) { return g_err.c_str(); }

int salmon_hip_create(int nx, int ny, int nz, int ly, int nspin, int no, int nk, const double *coef_lap,
                      const double *coef_nab, double coef_lap0, const double *vec_k, const double *rocc,
                      const double *wtk, const double *hgs, double hvol, salmon_hip_t *out) {
  if (!out) return fail(SALMON_HIP_EINVAL, "out is null");
  *out = nullptr;
  if (nx < 4 || ny < 4 || nz < 4) return fail(SALMON_HIP_EINVAL, "grid %dx%dx%d below Nd=4", nx, ny, nz);
  if (nx > kBlock) return fail(SALMON_HIP_EUNSUPPORTED, "nx=%d above %d", nx, kBlock);
  if (ly < ny) return fail(SALMON_HIP_EINVAL, "ly=%d < ny=%d", ly, ny);
  if ((size_t)nx * ly * nz > (size_t)INT_MAX) return fail(SALMON_HIP_EUNSUPPORTED, "grid of %dx%dx%d above 2^31 points", nx, ly, nz);
  if (nspin != 1 && nspin != 2) return fail(SALMON_HIP_EINVAL, "nspin=%d", nspin);
  if (no < 1 || nk < 1) return fail(SALMON_HIP_EINVAL, "no=%d nk=%d", no, nk);
  if (!coef_lap || !coef_nab || !vec_k || !rocc || !wtk || !hgs) return fail(SALMON_HIP_EINVAL, "null input");
  salmon_hip_ctx *c = new salmon_hip_ctx();
  c->nx = nx; c->ny = ny; c->nz = nz; c->ly = ly;
  c->nspin = nspin; c->no = no; c->nk = nk;
  c->nb = nspin * no;
  c->norb = c->nb * nk;
  c->osz = (size_t)nx * ly * nz;
  c->ngrid = (size_t)nx * ny * nz;
  memcpy(c->coef_lap, coef_lap, sizeof(c->coef_lap));
  memcpy(c->coef_nab, coef_nab, sizeof(c->coef_nab));
  c->coef_lap0 = coef_lap0;
  memcpy(c->hgs, hgs, sizeof(c->hgs));
  c->hvol = hvol;
  int rc = 0;
  auto bail = [&](int code) { salmon_hip_destroy(c); return code; };
  if (hipStreamCreateWithFlags(&c->own, hipStreamNonBlocking) != hipSuccess ||
      hipStreamCreateWithFlags(&c->side, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreateWithFlags(&c->ev_fork, hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&c->ev_join, hipEventDisableTiming) != hipSuccess)
    return bail(fail(SALMON_HIP_EHIP, "stream / event creation failed"));
  c->stream = c->own;
  if ((rc = dalloc(&c->d_veck, 3 * (size_t)nk))) return bail(rc);
  if ((rc = dalloc(&c->d_rocc, (size_t)no * nk * nspin))) return bail(rc);
  if ((rc = dalloc(&c->d_wtk, (size_t)nk))) return bail(rc);
  if ((rc = dalloc(&c->d_V, c->ngrid * nspin))) return bail(rc);
  if ((rc = dalloc(&c->d_kpar, 16 * (size_t)nk))) return bail(rc);
  if (hipMemcpy(c->d_veck, vec_k, sizeof(double) * 3 * nk, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(c->d_rocc, rocc, sizeof(double) * no * nk * nspin, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(c->d_wtk, wtk, sizeof(double) * nk, hipMemcpyHostToDevice) != hipSuccess)
    return bail(fail(SALMON_HIP_EHIP, "upload of k-point tables failed"));
  // stencil tile shape: full x rows, TY rows, z chunks so that the launch has
  // at least ~2048 blocks where the orbital count allows it
  c->TY = std::min(ny, std::max(1, kBlock / nx));
  c->nyt = (ny + c->TY - 1) / c->TY;
  int want = 2048;
  int nzt = (want + c->norb * c->nyt - 1) / (c->norb * c->nyt);
  nzt = std::max(1, std::min(nzt, std::max(1, nz / 8)));
  c->TZ = (nz + nzt - 1) / nzt;
  c->nzt = (nz + c->TZ - 1) / c->TZ;
  // observables scratch
  c->dens_ngrp = (no * nk + kDensGroup - 1) / kDensGroup;
  if (c->dens_ngrp > 1 && (rc = dalloc(&c->d_denspart, c->ngrid * nspin * c->dens_ngrp))) return bail(rc);
  if ((rc = dalloc(&c->d_curpart, 4 * (size_t)c->nyt * c->norb))) return bail(rc);
  // per spin: the batched step forms both spins' orbital contributions in one launch
  if ((rc = dalloc(&c->d_contrib, 3 * (size_t)no * nk * nspin))) return bail(rc);
  if ((rc = dalloc(&c->d_sink, 1024))) return bail(rc);  // one element per thread of the largest tile
  if ((rc = dalloc(&c->d_dippart, 4 * (size_t)kDipBlocks))) return bail(rc);
  if ((rc = resolve_scratch(&c->d_scratch))) return bail(rc);
  *out = c;
  return 0;
}

int salmon_hip_destroy(salmon_hip_t c) {
  if (!c) return 0;
  if (c->own) (void)hipStreamSynchronize(c->own);
  if (c->stream && c->stream != c->own) (void)hipStreamSynchronize(c->stream);
  dfree(c->d_veck); dfree(c->d_rocc); dfree(c->d_wtk); dfree(c->d_V); dfree(c->d_kpar); dfree(c->d_kpar_n);
  dfree(c->d_mps); dfree(c->d_jidx); dfree(c->d_pt_off);
  dfree(c->d_atom_lma); dfree(c->d_pt_lma); dfree(c->d_entof); dfree(c->d_rxyz); dfree(c->d_uv);
  dfree(c->d_rinv); dfree(c->d_zekr); dfree(c->d_zent); dfree(c->d_c); dfree(c->d_curnl);
  dfree(c->d_zekr_n); dfree(c->d_zent_n);
  c->staged = false;
  c->pre_state = 0;
  dfree(c->d_c2); dfree(c->d_jexcl); dfree(c->d_tp_shared);
  dfree(c->d_tp_info); dfree(c->d_sink);
  dfree(c->d_curpart); dfree(c->d_contrib); dfree(c->d_denspart); dfree(c->d_dippart);
  for (int d = 0; d < 3; ++d) dfree(c->d_tw[d]);
  dfree(c->d_gcoef); dfree(c->d_fft[0]); dfree(c->d_fft[1]);
  for (double2 *&p : c->tscr) dfree(p);
  for (float2 *&p : c->tscr32) dfree(p);
  for (hipEvent_t e : c->ev) (void)hipEventDestroy(e);
  if (c->side) (void)hipStreamSynchronize(c->side);
  if (c->ev_fork) (void)hipEventDestroy(c->ev_fork);
  if (c->ev_join) (void)hipEventDestroy(c->ev_join);
  if (c->side) (void)hipStreamDestroy(c->side);
  if (c->own) (void)hipStreamDestroy(c->own);
  delete c;
  return 0;
}

int salmon_hip_set_stream(salmon_hip_t c, void *stream) {
  if (int rc = check(c)) return rc;
  c->stream = (hipStream_t)stream;  // NULL: HIP's null stream (ordered with every blocking stream)
  return 0;
}

void *salmon_hip_get_stream(salmon_hip_t c) { return c ? (void *)c->stream : nullptr; }

int salmon_hip_set_nonlocal(salmon_hip_t c, int natom, int nps, const int *mps, const int *jxyz,
                            const double *rxyz, int nlma, const int *ia_tbl, const double *rinv_uvu,
                            const double *uv) {
  if (int rc = check(c)) return rc;
  HIPCHK(hipStreamSynchronize(c->stream));
  dfree(c->d_mps); dfree(c->d_jidx); dfree(c->d_pt_off);
  dfree(c->d_atom_lma); dfree(c->d_pt_lma); dfree(c->d_entof); dfree(c->d_rxyz); dfree(c->d_uv);
  dfree(c->d_rinv); dfree(c->d_zekr); dfree(c->d_zent); dfree(c->d_c); dfree(c->d_curnl);
  dfree(c->d_zekr_n); dfree(c->d_zent_n);
  c->staged = false;
  c->pre_state = 0;
  dfree(c->d_c2); dfree(c->d_jexcl); dfree(c->d_tp_shared);
  dfree(c->d_tp_info);
  c->kbval = 0.0;
  c->natom = c->nps = c->nlma = c->nent = c->cmax = c->ntp = c->ntp_shared = 0;
  c->have_k = false;
  if (natom == 0 || nlma == 0) return 0;
  if (natom < 0 || nps < 1 || nlma < 0 || !mps || !jxyz || !rxyz || !ia_tbl || !rinv_uvu || !uv)
    return fail(SALMON_HIP_EINVAL, "invalid projector tables");
  // validate: sphere sizes and grid indices, projectors contiguous per atom
  std::vector<int2> atom_lma(natom, make_int2(0, 0));
  for (int l = 0; l < nlma; ++l) {
    const int ia = ia_tbl[l] - 1;
    if (ia < 0 || ia >= natom) return fail(SALMON_HIP_EINVAL, "ia_tbl(%d)=%d out of range", l + 1, ia + 1);
    if (l > 0 && ia < ia_tbl[l - 1] - 1) return fail(SALMON_HIP_EUNSUPPORTED, "ia_tbl not atom-ordered");
    if (atom_lma[ia].y == 0) atom_lma[ia].x = l;
    else if (atom_lma[ia].x + atom_lma[ia].y != l)
      return fail(SALMON_HIP_EUNSUPPORTED, "projectors of atom %d not contiguous", ia + 1);
    atom_lma[ia].y += 1;
  }
  for (int ia = 0; ia < natom; ++ia)
    if (atom_lma[ia].y > kMaxLmaPerAtom)
      return fail(SALMON_HIP_EUNSUPPORTED, "atom %d has %d projectors (max %d)", ia + 1, atom_lma[ia].y,
                  kMaxLmaPerAtom);
  if (nlma >= (1 << 24)) return fail(SALMON_HIP_EUNSUPPORTED, "nlma too large");
  std::vector<int> jidx((size_t)natom * nps, 0);
  std::vector<int> cnt(c->ngrid + 1, 0);
  for (int ia = 0; ia < natom; ++ia) {
    if (mps[ia] < 0 || mps[ia] > nps) return fail(SALMON_HIP_EINVAL, "mps(%d)=%d", ia + 1, mps[ia]);
    for (int j = 0; j < mps[ia]; ++j) {
      const int *p = jxyz + 3 * ((size_t)j + (size_t)nps * ia);
      const int x = p[0] - 1, y = p[1] - 1, z = p[2] - 1;
      if (x < 0 || x >= c->nx || y < 0 || y >= c->ny || z < 0 || z >= c->nz)
        return fail(SALMON_HIP_EINVAL, "jxyz(:,%d,%d) outside the grid", j + 1, ia + 1);
      jidx[(size_t)nps * ia + j] = x + c->nx * (y + c->ly * z);
      const size_t g = (size_t)x + (size_t)c->nx * ((size_t)y + (size_t)c->ny * z);
      if (atom_lma[ia].y > 0) cnt[g + 1] += 1;
    }
  }
  for (size_t g = 0; g < c->ngrid; ++g) cnt[g + 1] += cnt[g];
  const int nent = cnt[c->ngrid];
  int cmax = 1;
  double kbval = 0.0;
  for (int ia = 0; ia < natom; ++ia) {
    cmax = std::max(cmax, atom_lma[ia].y);
    kbval += (double)mps[ia] * atom_lma[ia].y;
  }
  // CSR point -> (atom, j) entries; atom-major fill keeps each point's entries
  // in ascending ilma, the order zpseudo adds them in
  std::vector<int> pt_lma(std::max(nent, 1), 0);
  std::vector<int> entof((size_t)natom * nps, 0);
  std::vector<int> fillp(cnt.begin(), cnt.end() - 1);
  for (int ia = 0; ia < natom; ++ia) {
    if (atom_lma[ia].y == 0) continue;
    for (int j = 0; j < mps[ia]; ++j) {
      const int *p = jxyz + 3 * ((size_t)j + (size_t)nps * ia);
      const size_t g = (size_t)(p[0] - 1) + (size_t)c->nx * ((size_t)(p[1] - 1) + (size_t)c->ny * (p[2] - 1));
      const int e = fillp[g]++;
      pt_lma[e] = atom_lma[ia].x | (atom_lma[ia].y << 24);
      entof[(size_t)nps * ia + j] = e;
    }
  }
  std::vector<int4> tp_info;
  for (int z = 0; z < c->nz; ++z)
    for (int y = 0; y < c->ny; ++y)
      for (int x = 0; x < c->nx; ++x) {
        const size_t g = (size_t)x + (size_t)c->nx * ((size_t)y + (size_t)c->ny * z);
        if (cnt[g + 1] > cnt[g])
          tp_info.push_back(make_int4(x + c->nx * (y + c->ly * z), cnt[g], cnt[g + 1] - cnt[g], pt_lma[cnt[g]]));
      }
  // fused-pass tables: a sphere point's offset where its grid point has one entry, else -1;
  // the touched points with several entries
  std::vector<int> jexcl((size_t)natom * nps, -1);
  for (int ia = 0; ia < natom; ++ia) {
    if (atom_lma[ia].y == 0) continue;
    for (int j = 0; j < mps[ia]; ++j) {
      const int *p = jxyz + 3 * ((size_t)j + (size_t)nps * ia);
      const size_t g = (size_t)(p[0] - 1) + (size_t)c->nx * ((size_t)(p[1] - 1) + (size_t)c->ny * (p[2] - 1));
      if (cnt[g + 1] - cnt[g] == 1) jexcl[(size_t)nps * ia + j] = jidx[(size_t)nps * ia + j];
    }
  }
  std::vector<int4> tp_shared;
  for (const int4 &t : tp_info)
    if (t.z > 1) tp_shared.push_back(t);
  int rc = 0;
  if (!tp_info.empty()) {
    if ((rc = dalloc(&c->d_tp_info, tp_info.size()))) return rc;
    HIPCHK(hipMemcpy(c->d_tp_info, tp_info.data(), sizeof(int4) * tp_info.size(), hipMemcpyHostToDevice));
  }
  if (!tp_shared.empty()) {
    if ((rc = dalloc(&c->d_tp_shared, tp_shared.size()))) return rc;
    HIPCHK(hipMemcpy(c->d_tp_shared, tp_shared.data(), sizeof(int4) * tp_shared.size(), hipMemcpyHostToDevice));
  }
  if ((rc = dalloc(&c->d_jexcl, jexcl.size())) || (rc = dalloc(&c->d_c2, (size_t)nlma * c->norb))) return rc;
  HIPCHK(hipMemcpy(c->d_jexcl, jexcl.data(), sizeof(int) * jexcl.size(), hipMemcpyHostToDevice));
  if ((rc = dalloc(&c->d_mps, natom)) || (rc = dalloc(&c->d_jidx, (size_t)natom * nps)) ||
      (rc = dalloc(&c->d_pt_off, c->ngrid + 1)) ||
      (rc = dalloc(&c->d_atom_lma, natom)) || (rc = dalloc(&c->d_pt_lma, pt_lma.size())) ||
      (rc = dalloc(&c->d_entof, entof.size())) ||
      (rc = dalloc(&c->d_rxyz, 3 * (size_t)nps * natom)) || (rc = dalloc(&c->d_uv, (size_t)nps * nlma)) ||
      (rc = dalloc(&c->d_rinv, nlma)) || (rc = dalloc(&c->d_zekr, (size_t)nps * nlma * c->nk)) ||
      (rc = dalloc(&c->d_zent, (size_t)cmax * std::max(nent, 1) * c->nk)) ||
      (rc = dalloc(&c->d_c, (size_t)nlma * c->norb)) || (rc = dalloc(&c->d_curnl, 4 * (size_t)nlma * c->norb)))
    return rc;
  HIPCHK(hipMemcpy(c->d_mps, mps, sizeof(int) * natom, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(c->d_jidx, jidx.data(), sizeof(int) * jidx.size(), hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(c->d_pt_off, cnt.data(), sizeof(int) * cnt.size(), hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(c->d_atom_lma, atom_lma.data(), sizeof(int2) * natom, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(c->d_pt_lma, pt_lma.data(), sizeof(int) * pt_lma.size(), hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(c->d_entof, entof.data(), sizeof(int) * entof.size(), hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(c->d_rxyz, rxyz, sizeof(double) * 3 * nps * natom, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(c->d_uv, uv, sizeof(double) * (size_t)nps * nlma, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(c->d_rinv, rinv_uvu, sizeof(double) * nlma, hipMemcpyHostToDevice));
  c->natom = natom;
  c->nps = nps;
  c->nlma = nlma;
  c->nent = nent;
  c->cmax = cmax;
  c->kbval = kbval;
  c->ntp = (int)tp_info.size();
  c->ntp_shared = (int)tp_shared.size();
  return 0;
}

int salmon_hip_set_vlocal(salmon_hip_t c, const double *vlocal) {
  if (int rc = check(c)) return rc;
  if (!vlocal) return fail(SALMON_HIP_EINVAL, "vlocal is null");
  HIPCHK(hipMemcpyAsync(c->d_V, vlocal, sizeof(double) * c->ngrid * c->nspin, hipMemcpyHostToDevice, c->stream));
  HIPCHK(hipStreamSynchronize(c->stream));
  c->have_V = true;
  return 0;
}

int salmon_hip_set_vlocal_device(salmon_hip_t c, const double *vlocal_dev) {
  if (int rc = check(c)) return rc;
  if (!vlocal_dev) return fail(SALMON_HIP_EINVAL, "vlocal is null");
  HIPCHK(hipMemcpyAsync(c->d_V, vlocal_dev, sizeof(double) * c->ngrid * c->nspin, hipMemcpyDeviceToDevice,
                        c->stream));
  c->have_V = true;
  return 0;
}

int salmon_hip_stream_copy(salmon_hip_t c, void *dst_dev, const void *src_dev, size_t bytes, int reps,
                           double *avg_ms) {
  if (int rc = check(c)) return rc;
  if (!dst_dev || !src_dev || bytes % 16 != 0 || bytes == 0 || reps < 1)
    return fail(SALMON_HIP_EINVAL, "stream_copy: null buffer, %zu bytes (a positive multiple of 16) or reps %d",
                bytes, reps);
  const size_t n = bytes / 16;
  const unsigned grid = (unsigned)std::min<size_t>((n + 4 * 256 - 1) / (4 * 256), 1u << 20);
  hipEvent_t e0, e1;
  HIPCHK(hipEventCreate(&e0));
  HIPCHK(hipEventCreate(&e1));
  hipLaunchKernelGGL(k_stream_copy, dim3(grid), dim3(256), 0, c->stream, (u4v *)dst_dev, (const u4v *)src_dev, n);
  int rc = 0;
  if (hipEventRecord(e0, c->stream) != hipSuccess) rc = fail(SALMON_HIP_EHIP, "event");
  for (int r = 0; r < reps && !rc; ++r)
    hipLaunchKernelGGL(k_stream_copy, dim3(grid), dim3(256), 0, c->stream, (u4v *)dst_dev, (const u4v *)src_dev, n);
  float ms = 0.f;
  if (!rc && (hipGetLastError() != hipSuccess || hipEventRecord(e1, c->stream) != hipSuccess ||
              hipEventSynchronize(e1) != hipSuccess || hipEventElapsedTime(&ms, e0, e1) != hipSuccess))
    rc = fail(SALMON_HIP_EHIP, "stream_copy timing");
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (rc) return rc;
  if (avg_ms) *avg_ms = (double)ms / reps;
  return 0;
}

int salmon_hip_set_skip(salmon_hip_t c, const int *flag_dev) {
  if (int rc = check(c)) return rc;
  c->d_skip = flag_dev;
  return 0;
}

int salmon_hip_copy_if(salmon_hip_t c, const int *flag_dev, double *dst_dev, const double *src_dev, size_t n) {
  if (int rc = check(c)) return rc;
  if (!flag_dev || !dst_dev || !src_dev) return fail(SALMON_HIP_EINVAL, "null pointer");
  if (n == 0) return 0;
  hipLaunchKernelGGL(k_copy_if, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream, flag_dev, dst_dev,
                     src_dev, n);
  LAUNCHCHK("k_copy_if");
  return 0;
}

// Blocks per atom and k of the phase table for a launch over `atoms` (atom, k) pairs: one (one phase a point) from
// half a block per CU on; fewer leave the chip idle and take one per projector (32^3, one atom of 16 projectors, 4
// bohr: 21 us against 161; 64 atoms, radius 5: 16 projectors each 35 and 49 us, four 12.4 and 13.3; 128 pairs
// of them 68 and 49 us, 18.7 and 15.3; 512 pairs of 16 at radius 2.5 33 and 26 us).
static int kvec_split(long atoms, int cmax) { return atoms >= 128 ? 1 : std::max(1, cmax); }

static int kvec_blocks(const KvecArgs &a) { return std::max(1, a.natom * a.split); }

static KvecArgs kvec_args(salmon_hip_t c, const double *vec_Ac, const double *actab, const int *itt, int tmax) {
  KvecArgs a;
  a.veck = c->d_veck;
  a.rxyz = c->d_rxyz;
  a.uv = c->d_uv;
  a.mps = c->d_mps;
  a.natom = c->nlma > 0 ? c->natom : 0;
  a.split = kvec_split((long)a.natom * c->nk, c->cmax);
  a.atom_lma = c->d_atom_lma;
  a.entof = c->d_entof;
  a.zekr = c->d_zekr;
  a.zent = c->d_zent;
  a.nent = c->nent;
  a.cmax = c->cmax;
  a.kpar = c->d_kpar;
  memcpy(a.coef_nab, c->coef_nab, sizeof(a.coef_nab));
  a.coef_lap0 = c->coef_lap0;
  a.ax = vec_Ac ? vec_Ac[0] : 0.0;
  a.ay = vec_Ac ? vec_Ac[1] : 0.0;
  a.az = vec_Ac ? vec_Ac[2] : 0.0;
  a.actab = actab;
  a.itt = itt;
  a.tmax = tmax;
  a.nlma = c->nlma;
  a.nps = c->nps;
  a.nk = c->nk;
  return a;
}

static int update_kvector_impl(salmon_hip_t c, const double *vec_Ac, const double *actab, const int *itt,
                               int tmax = 0) {
  if (!actab && vec_Ac && c->staged && memcmp(vec_Ac, c->staged_A, sizeof(c->staged_A)) == 0) {
    // the table salmon_hip_current_next built ahead for this field becomes the active one
    std::swap(c->d_zekr, c->d_zekr_n);
    std::swap(c->d_zent, c->d_zent_n);
    std::swap(c->d_kpar, c->d_kpar_n);
    c->staged = false;
    if (c->pre_state == 1) c->pre_state = 2;
    c->have_k = true;
    return 0;
  }
  c->staged = false;
  c->pre_state = 0;
  const KvecArgs a = kvec_args(c, vec_Ac, actab, itt, tmax);
  dim3 grid(kvec_blocks(a), c->nk);
  hipLaunchKernelGGL(k_update_kvector, grid, dim3(kBlock), 0, c->stream, a);
  LAUNCHCHK("k_update_kvector");
  c->have_k = true;
  return 0;
}

int salmon_hip_update_kvector(salmon_hip_t c, const double *vec_Ac) {
  if (int rc = check(c)) return rc;
  if (!vec_Ac) return fail(SALMON_HIP_EINVAL, "vec_Ac is null");
  return update_kvector_impl(c, vec_Ac, nullptr, nullptr);
}

int salmon_hip_set_vec_ac(salmon_hip_t c, const double *vec_Ac) {
  if (int rc = check(c)) return rc;
  if (!vec_Ac) return fail(SALMON_HIP_EINVAL, "vec_Ac is null");
  if (c->nk > 1024) return fail(SALMON_HIP_EUNSUPPORTED, "nk=%d above 1024", c->nk);
  if (c->natom > 0 && !c->have_k) return fail(SALMON_HIP_ESTATE, "update_kvector not called yet");
  KvecArgs a;
  memset(&a, 0, sizeof(a));
  a.veck = c->d_veck;
  a.kpar = c->d_kpar;
  memcpy(a.coef_nab, c->coef_nab, sizeof(a.coef_nab));
  a.coef_lap0 = c->coef_lap0;
  a.ax = vec_Ac[0];
  a.ay = vec_Ac[1];
  a.az = vec_Ac[2];
  a.nk = c->nk;
  hipLaunchKernelGGL(k_set_kpar, dim3(1), dim3(1024), 0, c->stream, a);
  LAUNCHCHK("k_set_kpar");
  if (c->natom == 0) c->have_k = true;
  return 0;
}

// projection of psi into out (c(nb, nlma, nk) scaled by rinv, or the current moments)
// The projector count that the projection kernels of atoms with up to cmax projectors are built for.
static int proj_lm(int cmax) { return cmax <= 4 ? 4 : cmax <= 9 ? 9 : 16; }

static ProjArgs proj_args(salmon_hip_t c, const void *psi, double2 *out, int split) {
  ProjArgs a;
  a.psi = psi;
  a.zekr = c->d_zekr;
  a.rxyz = c->d_rxyz;
  a.jidx = c->d_jidx;
  a.mps = c->d_mps;
  a.atom_lma = c->d_atom_lma;
  a.rinv = c->d_rinv;
  a.out = out;
  a.osz = c->osz;
  a.nb = c->nb;
  a.nk = c->nk;
  a.natom = c->natom;
  a.nps = c->nps;
  a.nlma = c->nlma;
  a.ngrp = (c->nb + proj_orb(split) - 1) / proj_orb(split);
  a.skip = c->d_skip;
  a.zekr2 = nullptr;
  a.out2 = nullptr;
  return a;
}

// nw = 1: c of psi into d_c (skipped when salmon_hip_current_next left it there); 4: the current
// moments into d_curnl; 5: the moments and c of psi under the staged table into d_c
static int launch_proj(salmon_hip_t c, const void *psi, int nw, bool f32 = false) {
  if (nw == 1) {
    const bool pre = !f32 && c->pre_state == 2 && psi == c->pre_psi;
    c->pre_state = 0;
    if (pre) return 0;
  }
  const int lmx = proj_lm(c->cmax);
  const int split = proj_split(lmx, c->prec != SALMON_HIP_PREC_FP64);
  ProjArgs a = proj_args(c, psi, nw == 1 ? c->d_c : c->d_curnl, split);
  if (nw == 5) {
    a.zekr2 = c->d_zekr_n;
    a.out2 = c->d_c;
  }
  dim3 grid((unsigned)(a.ngrp * c->natom * c->nk));
  hipEvent_t e0, e1;
  prof_events(c, nw == 1 ? SALMON_HIP_KERNEL_PROJ : SALMON_HIP_KERNEL_PROJ_CURRENT, &e0, &e1);
  // with overlap: fork onto the side stream after everything enqueued on `stream` so far (the
  // producer of psi, the last reader of the projection buffer); joined before the scatter
  hipStream_t st = c->stream;
  if (c->overlap) {
    HIPCHK(hipEventRecord(c->ev_fork, c->stream));
    HIPCHK(hipStreamWaitEvent(c->side, c->ev_fork, 0));
    st = c->side;
  }
#define PROJ_LAUNCH_S(NWv, TPv, LMv, Sv) \
  hipExtLaunchKernelGGL((k_proj<NWv, TPv, LMv, Sv>), grid, dim3(kBlock), 0, st, e0, e1, 0, a)
#define PROJ_LAUNCH(NWv, TPv)                         \
  do {                                                \
    if (lmx == 4) PROJ_LAUNCH_S(NWv, TPv, 4, 1);      \
    else if (lmx == 9) PROJ_LAUNCH_S(NWv, TPv, 9, 1); \
    else PROJ_LAUNCH_S(NWv, TPv, 16, 1);              \
  } while (0)
  if (split == 4) {
    if (nw == 1) PROJ_LAUNCH_S(1, double2, 4, 4);
    else if (nw == 5) PROJ_LAUNCH_S(5, double2, 4, 4);
    else PROJ_LAUNCH_S(4, double2, 4, 4);
  } else
  if (nw == 1 && f32) PROJ_LAUNCH(1, float2);
  else if (nw == 1) PROJ_LAUNCH(1, double2);
  else if (nw == 5) PROJ_LAUNCH(5, double2);
  else PROJ_LAUNCH(4, double2);
#undef PROJ_LAUNCH
#undef PROJ_LAUNCH_S
  LAUNCHCHK("k_proj");
  if (c->overlap) {
    HIPCHK(hipEventRecord(c->ev_join, c->side));
    c->join_pending = true;
  }
  return 0;
}

// join: later work on `stream` waits for the last projection
static int join_proj(salmon_hip_t c) {
  if (!c->join_pending) return 0;
  HIPCHK(hipStreamWaitEvent(c->stream, c->ev_join, 0));
  c->join_pending = false;
  return 0;
}

}  // extern "C"

template <typename TI, int HC, int NC, int BS>
static size_t stencil_lds_bytes() {
  return sizeof(TI) * (kRingT * BS + kRingH * HC * BS) + sizeof(double2) * (NC >= 0 ? 2 * NC * BS : 0) +
         sizeof(double) * kRingH * BS;
}

// The dynamic-LDS limit of kernel f (hipFuncAttributeMaxDynamicSharedMemorySize), set once per
// device: the attribute belongs to the kernel on the device that is current when it is set.
static int lds_attr(const void *f, std::atomic<unsigned long long> &done, size_t bytes) {
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  const unsigned long long bit = 1ull << (dev & 63);
  if (done.load(std::memory_order_relaxed) & bit) return 0;
  HIPCHK(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
  done.fetch_or(bit);
  return 0;
}

template <typename TI, typename R, typename TO, int HC, int NC, int BS = kTile>
static int launch_stencil_t(salmon_hip_ctx *c, dim3 grid, hipEvent_t e0, hipEvent_t e1, const StencilArgs &a) {
  const size_t shmem = stencil_lds_bytes<TI, HC, NC, BS>();
  static std::atomic<unsigned long long> attr_dev{0};
  if (int rc = lds_attr((const void *)k_stencil<TI, R, TO, HC, NC, BS>, attr_dev, shmem)) return rc;
  hipExtLaunchKernelGGL((k_stencil<TI, R, TO, HC, NC, BS>), grid, dim3(BS), shmem, c->stream, e0, e1, 0, a);
  return 0;
}

// Stencil stages: plain FP64, and the three stages of the mixed-precision chain.
enum StencilStage { kStagePlain = 0, kStageMixedFirst = 1, kStageMixedMiddle = 2, kStageMixedFinal = 3 };

// Whole-plane tiles (no y halo) for the terms without the Taylor sum, nx * ny <= BS = 256.
template <int BS>
static int launch_stencil_plane(salmon_hip_ctx *c, int stage, dim3 grid, hipEvent_t e0, hipEvent_t e1,
                                const StencilArgs &a) {
  if (stage == kStageMixedFirst) return launch_stencil_t<double2, float, float2, 0, -1, BS>(c, grid, e0, e1, a);
  if (stage == kStageMixedMiddle) return launch_stencil_t<float2, float, float2, 0, -1, BS>(c, grid, e0, e1, a);
  return launch_stencil_t<double2, double, double2, 0, -1, BS>(c, grid, e0, e1, a);
}


// Whole planes of 256 < nx*ny <= 1024 points: 512 threads with PY points each (stencil_plane).
constexpr int kPlaneDepth = 2;  // look-ahead of the whole-plane kernel (planes; 3 measured no faster)

template <typename TI, typename R, typename TO, int PY>
static int launch_plane_t(salmon_hip_ctx *c, dim3 grid, hipEvent_t e0, hipEvent_t e1, const StencilArgs &a) {
  constexpr int BS = 512, D = kPlaneDepth;
  const size_t shmem = sizeof(TI) * (5 + D) * PY * BS + sizeof(double) * (D + 1) * PY * BS;
  static std::atomic<unsigned long long> attr_dev{0};
  if (int rc = lds_attr((const void *)k_stencil_plane<TI, R, TO, PY, BS, D>, attr_dev, shmem)) return rc;
  hipExtLaunchKernelGGL((k_stencil_plane<TI, R, TO, PY, BS, D>), grid, dim3(BS), shmem, c->stream, e0, e1, 0, a);
  return 0;
}

template <int PY>
static int launch_stencil_wp(salmon_hip_ctx *c, int stage, dim3 grid, hipEvent_t e0, hipEvent_t e1,
                             const StencilArgs &a) {
  if (stage == kStageMixedFirst) return launch_plane_t<double2, float, float2, PY>(c, grid, e0, e1, a);
  if (stage == kStageMixedMiddle) return launch_plane_t<float2, float, float2, PY>(c, grid, e0, e1, a);
  return launch_plane_t<double2, double, double2, PY>(c, grid, e0, e1, a);
}

// y tiles with the merged halo and compile-time ring slots (stencil_tile8): the middle terms of
// the mixed chain, rows of at most 64 points, (TY + 8) * nx <= 768 (slots of two or three
// 256-element chunks), z chunks of 8k planes.
static bool tile8_fits(const salmon_hip_ctx *c, int stage, int nc, const StencilArgs &a) {
  (void)nc;
  return stage == kStageMixedMiddle && a.nx <= 64 && (a.TY + 8) * a.nx <= 3 * kTile && a.TY * a.nx <= kTile &&
         a.TZ % 8 == 0 && a.nz % 8 == 0 && c->tile8;
}

// the paired dwordx4 DMAs need rows of even length and 16-byte aligned orbital blocks
static bool tile8_pairs(const StencilArgs &a) { return a.nx % 2 == 0 && a.osz % 2 == 0; }

// Taylor sums over up to 3 earlier terms (order 4): the slots of 4 or 5 would leave one block of
// stencil_tilez per CU (88 KB and more) where stencil_tile's shorter rings leave two.
constexpr int kTilezComb = 3;

// y tiles with the delayed z part (stencil_tilez): the FP64 terms on rows of up to 64 points and any
// number of planes; the mixed first term (FP64 input) on z chunks of 4k planes, elsewhere it keeps
// stencil_tile's order of the FP32 sum.  A plane's tile and halo rows fill a slot of 8, 10 or 12
// 64-element chunks (rows of up to 32 points; 48-point rows take 5 tile rows, 13 x 48 = 624
// elements in 10 chunks; up to 64 points).
static bool tilez_fits(int stage, int nc, const StencilArgs &a) {
  const bool fp64 = stage == kStagePlain && nc <= kTilezComb;
  return (fp64 || (stage == kStageMixedFirst && a.TZ % 4 == 0 && a.nz % 4 == 0)) && a.nx <= 64 &&
         (a.TY + 8) * a.nx <= 3 * kTile && a.TY * a.nx <= kTile;
}

template <typename TI, int NCK, int NC>
static constexpr size_t tilez_lds() {
  return sizeof(TI) * 4 * 64 * NCK + sizeof(double) * 4 * kTile + sizeof(double2) * 2 * (NC > 0 ? NC : 0) * kTile;
}

template <typename TI, typename R, typename TO, int NCK, bool XT, int NC>
static int launch_tilez_n(salmon_hip_ctx *c, dim3 grid, hipEvent_t e0, hipEvent_t e1, const StencilArgs &a) {
  const size_t shmem = tilez_lds<TI, NCK, NC>();
  static std::atomic<unsigned long long> attr_dev{0};
  if (int rc = lds_attr((const void *)k_stencilz<TI, R, TO, NCK, XT, NC>, attr_dev, shmem)) return rc;
  hipExtLaunchKernelGGL((k_stencilz<TI, R, TO, NCK, XT, NC>), grid, dim3(kTile), shmem, c->stream, e0, e1, 0, a);
  return 0;
}

// 64-element chunks per delayed-z slot for (TY + 8) rows of nx points: 8, 10 or 12
static int tilez_chunks(int TY, int nx) {
  const int need = (TY + 8) * nx;
  return need <= 8 * 64 ? 8 : (need <= 10 * 64 ? 10 : 12);
}

template <typename TI, typename R, typename TO, bool XT = false, int NC = -1>
static int launch_tilez_t(salmon_hip_ctx *c, dim3 grid, hipEvent_t e0, hipEvent_t e1, const StencilArgs &a) {
  switch (tilez_chunks(a.TY, XT ? a.TX + 8 : a.nx)) {
    case 8: return launch_tilez_n<TI, R, TO, 8, XT, NC>(c, grid, e0, e1, a);
    case 10: return launch_tilez_n<TI, R, TO, 10, XT, NC>(c, grid, e0, e1, a);
    default: return launch_tilez_n<TI, R, TO, 12, XT, NC>(c, grid, e0, e1, a);
  }
}

// z chunks of the FP64 terms in stencil_tilez: a chunk moves 8 planes beside its own, so as few as keep
// the chip busy.  With k blocks per CU a plane takes the larger of 0.65 us (one block's latency) and
// 0.49 us k; that is within 15% of what 14 shapes measured (13 to 48 points an axis, 16 to 512 orbitals) and
// picks the fastest of 1, 2, 3, 4 and 6 chunks for ten of them, the second for the rest.  Against 2048
// blocks or chunks of 8 planes at least: 32^3, 128 orbitals 48 and 42 us, 13 x 28 x 57, 128 orbitals 49 and 41 us.
static double tilez_planes(int nz, int nzt) {
  const int TZ = (nz + nzt - 1) / nzt;
  return (TZ + 7) / 4 * 4 + 4;
}

static void tilez_set_chunks(StencilArgs &a, int nzt) {
  a.TZ = (a.nz + nzt - 1) / nzt;
  a.nzt = (a.nz + a.TZ - 1) / a.TZ;
  a.nblk = a.nk * a.nb * a.nxt * a.nyt * a.nzt;
}

static void tilez_zchunks(StencilArgs &a) {
  const long tiles = (long)a.nk * a.nb * a.nxt * a.nyt;
  int best = 1;
  double tbest = 0.0;
  for (int n = 1; n <= std::max(1, a.nz / 8); ++n) {
    const double t = tilez_planes(a.nz, n) * std::max(0.65, 0.49 * ((tiles * n + 255) / 256));
    if (n > 1 && t >= tbest) continue;
    best = n;
    tbest = t;
  }
  tilez_set_chunks(a, best);
}

template <bool XT>
static int launch_tilez_fp64(salmon_hip_ctx *c, int nc, dim3 grid, hipEvent_t e0, hipEvent_t e1, const StencilArgs &a) {
  switch (nc) {
    case -1: return launch_tilez_t<double2, double, double2, XT>(c, grid, e0, e1, a);
    case 0: return launch_tilez_t<double2, double, double2, XT, 0>(c, grid, e0, e1, a);
    case 1: return launch_tilez_t<double2, double, double2, XT, 1>(c, grid, e0, e1, a);
    case 2: return launch_tilez_t<double2, double, double2, XT, 2>(c, grid, e0, e1, a);
    default: return launch_tilez_t<double2, double, double2, XT, 3>(c, grid, e0, e1, a);
  }
}

// Tiles of at most 256 points with a halo on x and y for rows above 64 points: the split of the plane
// that moves the fewest slot chunks.
static int tilez_xtiles(StencilArgs &a) {
  int best = INT_MAX;
  for (int nxt = 2; nxt <= 16; ++nxt) {
    const int TX = (a.nx + nxt - 1) / nxt;
    for (int nyt = 1; nyt <= a.ny; ++nyt) {
      const int TY = (a.ny + nyt - 1) / nyt;
      if (TX * TY > kTile || (TX + 8) * (TY + 8) > 12 * 64) continue;
      const int cost = ((a.nx + TX - 1) / TX) * ((a.ny + TY - 1) / TY) * tilez_chunks(TY, TX + 8);
      if (cost < best) {
        best = cost;
        a.TX = TX;
        a.TY = TY;
      }
      break;
    }
  }
  if (best == INT_MAX) return fail(SALMON_HIP_EINVAL, "no x/y tiles for a plane of %d x %d points", a.nx, a.ny);
  a.nxt = (a.nx + a.TX - 1) / a.TX;
  a.nyt = (a.ny + a.TY - 1) / a.TY;
  a.nblk = a.nk * a.nb * a.nxt * a.nyt * a.nzt;
  return 0;
}

template <typename TI, typename R, typename TO, int NCH, bool PR>
static int launch_tile8_n(salmon_hip_ctx *c, dim3 grid, hipEvent_t e0, hipEvent_t e1, const StencilArgs &a) {
  const size_t shmem = sizeof(TI) * 8 * NCH * kTile + sizeof(double) * 4 * kTile;
  static std::atomic<unsigned long long> attr_dev{0};
  if (int rc = lds_attr((const void *)k_stencil8<TI, R, TO, NCH, PR>, attr_dev, shmem)) return rc;
  hipExtLaunchKernelGGL((k_stencil8<TI, R, TO, NCH, PR>), grid, dim3(kTile), shmem, c->stream, e0, e1, 0, a);
  return 0;
}

template <typename TI, typename R, typename TO>
static int launch_tile8_t(salmon_hip_ctx *c, dim3 grid, hipEvent_t e0, hipEvent_t e1, const StencilArgs &a) {
  const bool pr = tile8_pairs(a);
  if ((a.TY + 8) * a.nx <= 2 * kTile)
    return pr ? launch_tile8_n<TI, R, TO, 2, true>(c, grid, e0, e1, a) : launch_tile8_n<TI, R, TO, 2, false>(c, grid, e0, e1, a);
  return pr ? launch_tile8_n<TI, R, TO, 3, true>(c, grid, e0, e1, a) : launch_tile8_n<TI, R, TO, 3, false>(c, grid, e0, e1, a);
}

template <int HC>
static int launch_stencil_hc(salmon_hip_ctx *c, int stage, int nc, dim3 grid, hipEvent_t e0, hipEvent_t e1,
                             const StencilArgs &a) {
  if (stage == kStageMixedFirst) return launch_stencil_t<double2, float, float2, HC, -1>(c, grid, e0, e1, a);
  if (stage == kStageMixedMiddle) return launch_stencil_t<float2, float, float2, HC, -1>(c, grid, e0, e1, a);
  if (stage == kStageMixedFinal) {
    switch (nc) {
      case 1: return launch_stencil_t<float2, float, double2, HC, 1>(c, grid, e0, e1, a);
      case 2: return launch_stencil_t<float2, float, double2, HC, 2>(c, grid, e0, e1, a);
      case 3: return launch_stencil_t<float2, float, double2, HC, 3>(c, grid, e0, e1, a);
      case 4: return launch_stencil_t<float2, float, double2, HC, 4>(c, grid, e0, e1, a);
      default: return launch_stencil_t<float2, float, double2, HC, 5>(c, grid, e0, e1, a);
    }
  }
  if (nc == 4) return launch_stencil_t<double2, double, double2, HC, 4>(c, grid, e0, e1, a);
  if (nc == 5) return launch_stencil_t<double2, double, double2, HC, 5>(c, grid, e0, e1, a);
  // the other FP64 terms are stencil_tilez's on every grid (tilez_fits, tilez_xtiles)
  return fail(SALMON_HIP_EINVAL, "no stencil form for %d earlier terms on rows of %d points", nc, a.nx);
}

extern "C" {

// shared_only: the touched points with several (atom, point) pairs (before k_proj_scatter);
// e0/e1 override the profiling events (nullptr: this launch's own)
// KB scatter hout += s * sum c zekr at the touched points (or only those several pairs cover)
static ScatterArgs scatter_args(salmon_hip_t c, void *hout, double2 s, const double2 *cbuf, bool shared_only, bool f32) {
  ScatterArgs a;
  a.hout = hout;
  a.c = cbuf;
  a.zent = c->d_zent;
  a.tp_info = shared_only ? c->d_tp_shared : c->d_tp_info;
  a.pt_lma = c->d_pt_lma;
  a.s = s;
  a.osz = c->osz;
  a.ntp = shared_only ? c->ntp_shared : c->ntp;
  a.nb = c->nb;
  a.nlma = c->nlma;
  a.nent = c->nent;
  a.cmax = c->cmax;
  a.skip = c->d_skip;
  const int G = f32 ? kScatG32 : kScatG;
  a.ngrp = (c->nb + G - 1) / G;
  return a;
}

static int launch_scatter(salmon_hip_t c, void *hout, double2 s, bool f32 = false, bool shared_only = false,
                          hipEvent_t ev0 = nullptr, hipEvent_t ev1 = nullptr, bool own_events = true) {
  if ((shared_only ? c->ntp_shared : c->ntp) == 0) return 0;
  const ScatterArgs a = scatter_args(c, hout, s, c->d_c, shared_only, f32);
  hipEvent_t e0 = ev0, e1 = ev1;
  if (own_events) prof_events(c, SALMON_HIP_KERNEL_NL_SCATTER, &e0, &e1);
  dim3 grid((unsigned)((a.ntp + kBlock - 1) / kBlock), (unsigned)(c->nk * a.ngrp));
  if (f32) {
    hipExtLaunchKernelGGL((k_nl_scatter<float2, kScatG32, kScatCM32>), grid, dim3(kBlock), 0, c->stream, e0, e1, 0, a);
  } else if (scat_plain(c->cmax, c->nb)) {
    hipExtLaunchKernelGGL((k_nl_scatter<double2, kScatG, 0>), grid, dim3(kBlock), 0, c->stream, e0, e1, 0, a);
  } else {
    hipExtLaunchKernelGGL((k_nl_scatter<double2, kScatG, kScatCM>), grid, dim3(kBlock), 0, c->stream, e0, e1, 0, a);
  }
  LAUNCHCHK("k_nl_scatter");
  return 0;
}

// the fused KB pass of hout (cin = c of the previous term, cout = c of hout)
static ProjScatArgs projscat_args(salmon_hip_t c, void *hout, const double2 *cin, double2 *cout, int split) {
  ProjScatArgs A;
  A.p = proj_args(c, hout, cout, split);
  A.cin = cin;
  A.jexcl = c->d_jexcl;
  A.s = make_double2(1.0, 0.0);
  A.cmax = c->cmax;
  return A;
}

// The KB term of hout = H in (c of `in` current in d_c) fused with the projection of hout: the
// points with several pairs by k_nl_scatter, then k_proj_scatter; afterwards d_c holds the c of
// hout.  Profiled as one SALMON_HIP_KERNEL_KB_FUSED interval.
static int launch_kb_fused(salmon_hip_t c, void *hout, bool f32) {
  hipEvent_t e0, e1;
  prof_events(c, SALMON_HIP_KERNEL_KB_FUSED, &e0, &e1);
  const bool shared = c->ntp_shared > 0;
  if (shared)
    if (int rc = launch_scatter(c, hout, make_double2(1.0, 0.0), f32, true, e0, nullptr, false)) return rc;
  const int lm = proj_lm(c->cmax);
  const int split = proj_split(lm, c->prec != SALMON_HIP_PREC_FP64);
  const ProjScatArgs A = projscat_args(c, hout, c->d_c, c->d_c2, split);
  const size_t shmem = sizeof(double2) * (size_t)c->cmax * proj_orb(split);
  dim3 grid((unsigned)(A.p.ngrp * c->natom * c->nk));
  hipEvent_t s0 = shared ? nullptr : e0;
  // LM: registers for the projector values of one point (s+p: 4, up to d: 9, up to f: 16)
#define KB_LAUNCH_S(TPv, LMv, Sv) \
  hipExtLaunchKernelGGL((k_proj_scatter<TPv, LMv, Sv>), grid, dim3(kBlock), shmem, c->stream, s0, e1, 0, A)
#define KB_LAUNCH(TPv)                        \
  do {                                        \
    if (lm == 4) KB_LAUNCH_S(TPv, 4, 1);      \
    else if (lm == 9) KB_LAUNCH_S(TPv, 9, 1); \
    else KB_LAUNCH_S(TPv, 16, 1);             \
  } while (0)
  if (split == 4) KB_LAUNCH_S(double2, 4, 4);
  else if (f32) KB_LAUNCH(float2);
  else KB_LAUNCH(double2);
#undef KB_LAUNCH
#undef KB_LAUNCH_S
  LAUNCHCHK("k_proj_scatter");
  std::swap(c->d_c, c->d_c2);
  c->pre_state = 0;
  return 0;
}

// The fused KB pass is used inside Taylor chains when the projections run on the handle's stream.
static bool kb_fused_on(const salmon_hip_ctx *c) { return c->kb_fused && !c->overlap && c->natom > 0 && c->nlma > 0; }

// One H application: hout = H in (fin = false), or the last Taylor term
// hout = psi + c1 h1 + ... + c_N H in (fin = true, comb = [psi, h1 .. h_{N-2}]).
// The projections c of `in` must be current (launch_proj).
// Stencil descriptor of one H application; *bs_out = whole-plane block size (0 = y tiles).
// tiled_only forces the y-tile shape (the batched step).
static StencilArgs stencil_args(salmon_hip_t c, const void *in, void *hout, bool fin, void *const *comb, int ncomb,
                                const double *zc, int *bs_out, bool tiled_only) {
  StencilArgs a;
  memset(&a, 0, sizeof(a));
  a.in = in;
  a.hout = hout;
  a.sink = c->d_sink;
  a.skip = tiled_only ? nullptr : c->d_skip;
  const int nc = fin ? ncomb : -1;
  for (int n = 0; n < (fin ? ncomb : 0); ++n) a.comb[n] = comb[n];
  if (fin)
    for (int n = 0; n <= ncomb; ++n) a.zc[n] = make_double2(zc[2 * n], zc[2 * n + 1]);
  a.V = c->d_V;
  a.kpar = c->d_kpar;
  memcpy(a.lap, c->coef_lap, sizeof(a.lap));
  a.osz = c->osz;
  a.nx = c->nx; a.ny = c->ny; a.nz = c->nz; a.ly = c->ly;
  a.nspin = c->nspin; a.nb = c->nb; a.nk = c->nk;
  a.TY = c->TY; a.TZ = c->TZ; a.nyt = c->nyt; a.nzt = c->nzt;
  a.TX = c->nx; a.nxt = 1;
  // terms without the Taylor sum use whole xy-plane tiles when a plane fits one block
  const int plane = c->nx * c->ny;
  // rule (tile_plane = -1): whole planes only up to 256 points (one 256-thread block); the
  // 1024-thread FP64 block spills and holds one block per CU (slower at 32x32, measured)
  const bool use_plane = !tiled_only && nc < 0 && plane <= 1024 &&
                         (c->tile_plane == 1 || (c->tile_plane == -1 && plane <= 256));
  const int bs = !use_plane ? 0 : (plane <= 256 ? 256 : (plane <= 512 ? 512 : 1024));
  if (bs) {
    a.TY = c->ny;
    a.nyt = 1;
    a.nzt = std::max(1, std::min((512 + c->norb - 1) / c->norb, c->nz / 8));
  }
  if (nc < 0 && c->mid_nzt > 0) a.nzt = std::min(c->mid_nzt, c->nz);
  if (bs || (nc < 0 && c->mid_nzt > 0)) {
    a.TZ = (c->nz + a.nzt - 1) / a.nzt;
    a.nzt = (c->nz + a.TZ - 1) / a.TZ;
  }
  a.nblk = c->norb * a.nyt * a.nzt;
  *bs_out = bs;
  return a;
}

// fuse_next: finish with the fused KB pass (hout's KB term and its projection) instead of the scatter.
static int launch_hpsi(salmon_hip_t c, int kind, const void *in, void *hout, bool fin, void *const *comb, int ncomb,
                       const double *zc, int stage = kStagePlain, bool fuse_next = false) {
  int bs = 0;
  const int nc = fin ? ncomb : -1;
  StencilArgs a = stencil_args(c, in, hout, fin, comb, ncomb, zc, &bs, false);
  dim3 grid((unsigned)a.nblk);
  hipEvent_t e0, e1;
  prof_events(c, kind, &e0, &e1);
  const int hc = (8 * c->nx + kTile - 1) / kTile;
  int rc = 0;
  if (bs == 256) rc = launch_stencil_plane<256>(c, stage, grid, e0, e1, a);
  else if (bs == 512) rc = launch_stencil_wp<1>(c, stage, grid, e0, e1, a);
  else if (bs == 1024) rc = launch_stencil_wp<2>(c, stage, grid, e0, e1, a);
  else if (tilez_fits(stage, nc, a) && stage == kStagePlain) {
    if (c->mid_nzt == 0 || nc >= 0) tilez_zchunks(a);
    rc = launch_tilez_fp64<false>(c, nc, dim3((unsigned)a.nblk), e0, e1, a);
  } else if (tilez_fits(stage, nc, a)) rc = launch_tilez_t<double2, float, float2>(c, grid, e0, e1, a);
  else if (tile8_fits(c, stage, nc, a)) rc = launch_tile8_t<float2, float, float2>(c, grid, e0, e1, a);
  else if (stage == kStagePlain && nc <= kTilezComb && a.nx > 64) {
    if (int rx = tilez_xtiles(a)) return rx;
    if (c->mid_nzt == 0 || nc >= 0) tilez_zchunks(a);
    rc = launch_tilez_fp64<true>(c, nc, dim3((unsigned)a.nblk), e0, e1, a);
  } else if (hc <= 1) rc = launch_stencil_hc<1>(c, stage, nc, grid, e0, e1, a);
  else if (hc <= 2) rc = launch_stencil_hc<2>(c, stage, nc, grid, e0, e1, a);
  else if (hc <= 4) rc = launch_stencil_hc<4>(c, stage, nc, grid, e0, e1, a);
  else rc = launch_stencil_hc<8>(c, stage, nc, grid, e0, e1, a);
  if (rc) return rc;
  LAUNCHCHK("k_stencil");
  const bool f32out = stage == kStageMixedFirst || stage == kStageMixedMiddle;
  if (int rc = join_proj(c)) return rc;
  if (fuse_next && !fin && kb_fused_on(c)) return launch_kb_fused(c, hout, f32out);
  if (c->natom > 0 && c->nlma > 0)
    return launch_scatter(c, hout, fin ? a.zc[ncomb] : make_double2(1.0, 0.0), f32out);
  return 0;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Whole-orbital launches for small grids (small_grid.h)
// ---------------------------------------------------------------------------
constexpr size_t kSmallLds = 156 * 1024;  // of the CU's 160 KB

// The launch of k_taylor_small for a handle's grid: template class (largest block, waves per SIMD that
// the registers allow), planes per thread, z chunks per column, threads, waves per atom.
struct SmallShape {
  int cls = -1, ppt = 0, zchunks = 0, bs = 0, nsub = 1;
  size_t lds = 0;
};

// Classes with the most planes per thread that each one's registers hold (more spill).
struct SmallClass {
  int bsmax, minw, pptmax;
};
constexpr SmallClass kSmallClass[] = {{512, 2, 8}, {512, 4, 4}, {768, 3, 10}, {1024, 4, 4}};

// The fewest wave-planes (waves x planes per thread, idle lanes included: the stencil is bound by the
// CU's LDS reads), weighted by what the launch needs beside: with up to two orbitals per CU the
// block's own latency counts, and the class with 256 registers issues its table loads ahead of their
// use; with more, blocks that share a CU hide each other's barriers and loads (few resident waves, or one
// block alone, cost as measured at 12^3).  Measured (one Taylor
// step of order 4, 8 atoms): 16^3, 16 orbitals: 51.6 us as {512, 2} with 8 planes, 56.7 as {768, 3},
// 73.8 as {512, 4}; 12^3, 1024 orbitals: 94 us as {512, 4} with 4 planes, 117 as {768, 3} with 3,
// 126 as {512, 2} with 4.
static SmallShape small_shape(const salmon_hip_ctx *c) {
  SmallShape best;
  const int ncol = c->nx * c->ny;
  double low = 0.0;
  for (int k = 0; k < 4; ++k) {
    const SmallClass &K = kSmallClass[k];
    for (int ppt = 2; ppt <= K.pptmax; ++ppt) {
      SmallShape s;
      s.cls = k;
      s.ppt = ppt;
      s.zchunks = (c->nz + ppt - 1) / ppt;
      if ((size_t)ncol * s.zchunks > (size_t)K.bsmax) continue;
      // at least one wave for each of the first eight atoms
      const int waves = std::max((ncol * s.zchunks + 63) / 64, std::min(c->natom, 8));
      s.bs = 64 * waves;
      if (c->natom > 0) s.nsub = std::max(1, waves / c->natom);
      s.lds = sizeof(double2) * (c->osz + 2 * (size_t)c->nlma * s.nsub + 2 * (size_t)c->ntp_shared);
      if (s.lds > kSmallLds) continue;
      double cost = (double)waves * ppt;
      if (c->norb <= 512) {
        cost *= K.minw == 2 ? 1.0 : 1.15;
      } else {
        const int blocks = std::min(std::max(1, 4 * K.minw / waves), (int)std::max<size_t>(1, (160 * 1024) / s.lds));
        cost *= std::sqrt(16.0 / std::min(16, blocks * waves)) * (blocks == 1 ? 1.2 : 1.0);
      }
      if (best.cls < 0 || cost < low) {
        best = s;
        low = cost;
      }
    }
  }
  return best;
}

// FP64 handles whose orbital block fits one CU's LDS; a launch shape set by hand
// (salmon_hip_set_launch_shape) and the overlapped projections select the per-term kernels.
static bool small_fits(const salmon_hip_ctx *c) {
  if (!c->small_grid || c->overlap || c->prec != SALMON_HIP_PREC_FP64) return false;
  if (c->osz * sizeof(double2) > kSmallLds || (size_t)c->nx * c->ly * sizeof(double2) > 65536 || c->ntp_shared > 65534)
    return false;
  return small_shape(c).cls >= 0;
}

// What a block of the whole-orbital kernels walks one after another in a KB pass: for the busiest wave, 64-point
// pieces of its atoms' spheres times groups of four projectors (with more than four, the points are completed in a
// pass of their own).
static double small_chain(const salmon_hip_ctx *c, const SmallShape &s) {
  if (c->natom == 0) return 0.0;
  const int ngroup = s.bs / 64 / s.nsub, pts = (int)std::ceil(c->kbval / c->nlma);
  const double pieces = (double)((c->natom + ngroup - 1) / ngroup) * ((pts + 64 * s.nsub - 1) / (64 * s.nsub));
  return pieces * ((c->cmax + 3) / 4 + (c->cmax > 4 ? 0.25 * c->cmax : 0.0));
}

// More than six planes per thread in 768 threads: the registers spill.
static bool small_spills(const SmallShape &s) { return kSmallClass[s.cls].bsmax == 768 && s.ppt > 6; }

// Where the whole-orbital step is the faster one on such a grid. A block reads all projector values of its orbital
// (kbval) in every term, k_proj and k_proj_scatter once for 16 or 64 orbitals, and the latter spread over more
// blocks with more atoms. Up to one orbital per CU, and with few values for any number of orbitals, one block per
// orbital won or tied wherever measured; else the line is drawn through 856 random cells (8 to 32 atoms of 1 to 16
// projectors, 240 to 4500 orbitals), of which 15 end 4 to 20% behind the better form; orders 2 and 3, whose
// orbitals are read and written for fewer terms, a little earlier (156 cells). Order 4, whole orbital against per
// term: 16^3, 8 atoms of 9 projectors (18 000 values), 4096 orbitals 1369 and 1385 us; 18^3, 9 projectors (26
// 000), 1024 orbitals 757 and 807 us, 2048 1573 and 1239 us; 12^3, 16 projectors (56 000), 512 orbitals 620 and
// 794 us, 2048 2336 and 1320 us; 12 x 12 x 24, 16 atoms of 16 (112 000), 320 orbitals 1310 and 718 us, 2048 6485
// and 2461 us.
static bool small_step(const salmon_hip_ctx *c, int n_hamil) {
  if (!small_fits(c)) return false;
  const double f = std::min(1.0, 0.3 + 0.175 * n_hamil);
  if (c->norb <= 256 || c->kbval <= 19e3 * f) return true;
  const SmallShape s = small_shape(c);
  return c->norb * std::sqrt(c->kbval * small_chain(c, s) * c->natom / 8) * (small_spills(s) ? 1.25 : 1.0) <= 1.44e6 * f;
}

// One application alone, whose three per-term launches are worth their cost above about a thousand orbitals
// (16^3, 1024 orbitals: 93 us in one launch, 112 per term; 15x17x14, 1600 orbitals: 150 and 126; 12x12x24, 2048
// orbitals: 171 and 158) and with many projector values or atoms earlier (18^3, 26 000 values, 512 orbitals 120
// and 147 us, 1024 235 and 200 us; 14 x 13 x 15, 86 000, 256 orbitals 148 and 172 us, 320 261 and 182 us; 10 x 20 x
// 30, 16 atoms, 320 orbitals 106 and 64 us).  Both forms' times in us, each within 10% (rms) of 538 random cells:
// one block costs its points, its shared points' projectors and its chain, per orbital and CU or round of
// resident blocks, and its projector values in the L2; the launches cost the points of all
// orbitals, the rounds of k_proj's blocks (32 sphere points at a time) and the gathers.
static bool small_hpsi(const salmon_hip_ctx *c) {
  if (c->norb > 1024 || !small_fits(c)) return false;
  if (c->norb <= 256 || c->natom == 0) return true;
  const SmallShape s = small_shape(c);
  const int waves = s.bs / 64, percu = (c->norb + 255) / 256;
  const int blocks = std::min(std::max(1, 4 * kSmallClass[s.cls].minw / waves), (int)std::max<size_t>(1, (160 * 1024) / s.lds));
  const int rounds = (percu + blocks - 1) / blocks;
  const double values = 1e-6 * c->norb * c->kbval, pts = c->kbval / c->nlma;
  const double whole = 5.0 + percu * (4.1e-3 * c->ngrid + 1.4e-3 * c->ntp_shared * c->cmax +
                                      (small_spills(s) ? 0.076 * waves * s.ppt : 0.0)) +
                       0.32 * rounds * small_chain(c, s) + 1.9 * values;
  const int pblk = c->natom * c->nk * ((c->nb + 63) / 64);
  const double terms = 25.0 + 14e-6 * c->norb * c->ngrid + 3.6e-6 * c->norb * c->natom * pts + 1.2 * values +
                       (c->cmax > 4 ? 4.9 * ((pblk + 511) / 512) * std::ceil(pts / 32) : 0.0);
  return whole <= 1.08 * terms;
}

static SmallArgs small_args(salmon_hip_t c, const void *psi, void *out, void *h1) {
  SmallArgs a;
  memset(&a, 0, sizeof(a));
  a.psi = (const double2 *)psi;
  a.out = (double2 *)out;
  a.h1 = (double2 *)h1;
  a.V = c->d_V;
  a.kpar = c->d_kpar;
  a.zekr = c->d_zekr;
  a.zent = c->d_zent;
  a.jidx = c->d_jidx;
  a.mps = c->d_mps;
  a.atom_lma = c->d_atom_lma;
  a.jexcl = c->d_jexcl;
  a.tp_shared = c->d_tp_shared;
  a.pt_lma = c->d_pt_lma;
  a.rinv = c->d_rinv;
  for (int i = 0; i < 12; ++i) a.lap[i] = -0.5 * c->coef_lap[i];
  a.osz = c->osz;
  a.nx = c->nx; a.ny = c->ny; a.nz = c->nz; a.ly = c->ly;
  a.nspin = c->nspin; a.nb = c->nb; a.nk = c->nk;
  a.nterm = a.first = 1;
  a.natom = c->natom; a.nps = c->nps; a.nlma = c->nlma;
  a.nent = c->nent; a.cmax = c->cmax; a.ntp_shared = c->ntp_shared;
  a.skip = c->d_skip;
  return a;
}

template <int PPT, int BSMAX, int MINW>
static int launch_taylor_small_t(salmon_hip_ctx *c, const SmallShape &s, const SmallArgs &a, hipEvent_t e0, hipEvent_t e1) {
  static std::atomic<unsigned long long> attr_dev{0};
  if (int rc = lds_attr((const void *)k_taylor_small<PPT, BSMAX, MINW>, attr_dev, kSmallLds)) return rc;
  hipExtLaunchKernelGGL((k_taylor_small<PPT, BSMAX, MINW>), dim3((unsigned)c->norb), dim3(s.bs), s.lds, c->stream, e0, e1, 0,
                        a);
  LAUNCHCHK("k_taylor_small");
  return 0;
}

template <int K>
static int launch_taylor_small_c(salmon_hip_ctx *c, const SmallShape &s, const SmallArgs &a, hipEvent_t e0, hipEvent_t e1) {
  constexpr int BSMAX = kSmallClass[K].bsmax, MINW = kSmallClass[K].minw, PM = kSmallClass[K].pptmax;
  switch (s.ppt) {
    case 2: return launch_taylor_small_t<2, BSMAX, MINW>(c, s, a, e0, e1);
    case 3: return launch_taylor_small_t<3, BSMAX, MINW>(c, s, a, e0, e1);
    case 4: return launch_taylor_small_t<4, BSMAX, MINW>(c, s, a, e0, e1);
    case 5: return launch_taylor_small_t<std::min(5, PM), BSMAX, MINW>(c, s, a, e0, e1);
    case 6: return launch_taylor_small_t<std::min(6, PM), BSMAX, MINW>(c, s, a, e0, e1);
    case 7: return launch_taylor_small_t<std::min(7, PM), BSMAX, MINW>(c, s, a, e0, e1);
    case 8: return launch_taylor_small_t<std::min(8, PM), BSMAX, MINW>(c, s, a, e0, e1);
    case 9: return launch_taylor_small_t<std::min(9, PM), BSMAX, MINW>(c, s, a, e0, e1);
    default: return launch_taylor_small_t<std::min(10, PM), BSMAX, MINW>(c, s, a, e0, e1);
  }
}

static int launch_taylor_small(salmon_hip_ctx *c, int kind, SmallArgs &a) {
  const SmallShape s = small_shape(c);
  a.zchunks = s.zchunks;
  a.nsub = s.nsub;
  c->pre_state = 0;
  hipEvent_t e0, e1;
  prof_events(c, kind, &e0, &e1);
  switch (s.cls) {
    case 0: return launch_taylor_small_c<0>(c, s, a, e0, e1);
    case 1: return launch_taylor_small_c<1>(c, s, a, e0, e1);
    case 2: return launch_taylor_small_c<2>(c, s, a, e0, e1);
    default: return launch_taylor_small_c<3>(c, s, a, e0, e1);
  }
}

extern "C" {

static int ready(salmon_hip_t c) {
  if (!c->have_V) return fail(SALMON_HIP_ESTATE, "V_local not set");
  if (!c->have_k) return fail(SALMON_HIP_ESTATE, "update_kvector (vec_Ac) not set");
  return 0;
}

int salmon_hip_hpsi(salmon_hip_t c, const void *tpsi, void *htpsi) {
  if (int rc = check(c)) return rc;
  if (!tpsi || !htpsi || tpsi == htpsi) return fail(SALMON_HIP_EINVAL, "tpsi/htpsi invalid or aliased");
  if (int rc = ready(c)) return rc;
  if (small_hpsi(c)) {
    SmallArgs a = small_args(c, tpsi, nullptr, htpsi);
    return launch_taylor_small(c, SALMON_HIP_KERNEL_HPSI0, a);
  }
  if (c->natom > 0)
    if (int rc = launch_proj(c, tpsi, 1)) return rc;
  return launch_hpsi(c, SALMON_HIP_KERNEL_HPSI0, tpsi, htpsi, false, nullptr, 0, nullptr);
}

// Mixed-precision Taylor step: h_n = H^n psi in complex FP32 (stencil and
// local-potential products in FP32; projections, the KB term and the Taylor sum
// in FP64), out = psi + sum_n zc(n) h_n formed in FP64 by the last stencil pass.
// first = 1: the whole chain; first = 2: h_1 (the handle's FP32 H psi) is already current
static int taylor_mixed(salmon_hip_t c, const double *zc, int n_hamil, void *tin, void *tout, int first = 1) {
  if (n_hamil < 2) return fail(SALMON_HIP_EUNSUPPORTED, "mixed precision needs n_hamil >= 2");
  while ((int)c->tscr32.size() < n_hamil - 1) {
    float2 *p = nullptr;
    if (int rc = dalloc(&p, c->osz * c->norb)) return rc;
    c->tscr32.push_back(p);
  }
  void *h[kMaxComb + 1];
  h[0] = tin;
  for (int n = 1; n < n_hamil; ++n) h[n] = c->tscr32[n - 1];
  // with the fused KB pass each term's projection comes out of the previous term's KB pass
  const bool fuse = kb_fused_on(c);
  bool have_c = false;
  for (int n = first; n < n_hamil; ++n) {
    if (c->natom > 0 && !have_c)
      if (int rc = launch_proj(c, h[n - 1], 1, n > 1)) return rc;
    const int kind = n == 1 ? SALMON_HIP_KERNEL_HPSI_TAYLOR1 : SALMON_HIP_KERNEL_HPSI_TAYLOR;
    const int stage = n == 1 ? kStageMixedFirst : kStageMixedMiddle;
    if (int rc = launch_hpsi(c, kind, h[n - 1], h[n], false, nullptr, 0, nullptr, stage, fuse)) return rc;
    have_c = fuse;
  }
  if (c->natom > 0 && !have_c)
    if (int rc = launch_proj(c, h[n_hamil - 1], 1, true)) return rc;
  return launch_hpsi(c, SALMON_HIP_KERNEL_HPSI_TAYLOR_LAST, h[n_hamil - 1], tout, true, h, n_hamil - 1, zc,
                     kStageMixedFinal);
}

int salmon_hip_set_precision(salmon_hip_t c, int mode) {
  if (int rc = check(c)) return rc;
  if (mode != SALMON_HIP_PREC_FP64 && mode != SALMON_HIP_PREC_MIXED)
    return fail(SALMON_HIP_EINVAL, "precision mode %d", mode);
  c->prec = mode;
  return 0;
}

// h_1 += dv psi (salmon_hip_taylor_reuse)
}  // extern "C"
template <typename TH>
static int launch_vshift(salmon_hip_ctx *c, void *h1, const void *psi, const double *dv) {
  const size_t ntot = c->osz * c->norb;
  const dim3 grid((unsigned)((ntot + kBlock - 1) / kBlock));
  hipLaunchKernelGGL(k_vshift<TH>, grid, dim3(kBlock), 0, c->stream, (TH *)h1, (const double2 *)psi, dv, c->osz, c->nx,
                     c->ny, c->ly, c->nz, c->nspin, ntot, c->d_skip);
  LAUNCHCHK("k_vshift");
  return 0;
}
extern "C" {

// first = 1: the whole chain; first = 2: h_1 = sshtpsi is H psi of a previous call, to be shifted by dv
static int taylor_fp64(salmon_hip_t c, const double *zc, int n_hamil, void *tspsi_in, void *tspsi_out, void *sshtpsi,
                       int first, const double *dv = nullptr) {
  if (small_step(c, n_hamil)) {
    SmallArgs a = small_args(c, tspsi_in, tspsi_out, n_hamil >= 2 ? sshtpsi : nullptr);
    for (int n = 0; n < n_hamil; ++n) a.zc[n] = make_double2(zc[2 * n], zc[2 * n + 1]);
    a.nterm = n_hamil;
    a.first = first;
    a.dv = dv;
    return launch_taylor_small(c, SALMON_HIP_KERNEL_HPSI_TAYLOR_LAST, a);
  }
  if (dv)
    if (int rc = launch_vshift<double2>(c, sshtpsi, tspsi_in, dv)) return rc;
  // h_1 = H psi -> sshtpsi, h_2 .. h_{N-1} -> internal scratch
  const int nscr = std::max(0, n_hamil - 2);
  while ((int)c->tscr.size() < nscr) {
    double2 *p = nullptr;
    if (int rc = dalloc(&p, c->osz * c->norb)) return rc;
    c->tscr.push_back(p);
  }
  void *h[kMaxComb + 1];
  h[0] = tspsi_in;
  if (n_hamil >= 2) h[1] = sshtpsi;
  for (int n = 2; n < n_hamil; ++n) h[n] = c->tscr[n - 2];
  const bool fuse = kb_fused_on(c);
  bool have_c = false;
  for (int n = first; n < n_hamil; ++n) {
    if (c->natom > 0 && !have_c)
      if (int rc = launch_proj(c, h[n - 1], 1)) return rc;
    const int kind = n == 1 ? SALMON_HIP_KERNEL_HPSI_TAYLOR1 : SALMON_HIP_KERNEL_HPSI_TAYLOR;
    if (int rc = launch_hpsi(c, kind, h[n - 1], h[n], false, nullptr, 0, nullptr, kStagePlain, fuse)) return rc;
    have_c = fuse;
  }
  if (c->natom > 0 && !have_c)
    if (int rc = launch_proj(c, h[n_hamil - 1], 1)) return rc;
  return launch_hpsi(c, SALMON_HIP_KERNEL_HPSI_TAYLOR_LAST, h[n_hamil - 1], tspsi_out, true, h, n_hamil - 1, zc);
}

int salmon_hip_taylor(salmon_hip_t c, const double *zc, int n_hamil, void *tspsi_in, void *tspsi_out,
                      void *sshtpsi) {
  if (int rc = check(c)) return rc;
  if (!zc || n_hamil < 1 || n_hamil > kMaxComb + 1)
    return fail(SALMON_HIP_EINVAL, "zc null or n_hamil=%d outside 1..%d", n_hamil, kMaxComb + 1);
  if (!tspsi_in || !tspsi_out || !sshtpsi || tspsi_in == tspsi_out || tspsi_in == sshtpsi || tspsi_out == sshtpsi)
    return fail(SALMON_HIP_EINVAL, "taylor buffers invalid or aliased");
  if (int rc = ready(c)) return rc;
  if (c->prec == SALMON_HIP_PREC_MIXED) return taylor_mixed(c, zc, n_hamil, tspsi_in, tspsi_out);
  return taylor_fp64(c, zc, n_hamil, tspsi_in, tspsi_out, sshtpsi, 1);
}

int salmon_hip_taylor_reuse(salmon_hip_t c, const double *zc, int n_hamil, void *tspsi_in, void *tspsi_out,
                            void *sshtpsi, const double *dv_dev) {
  if (int rc = check(c)) return rc;
  if (!zc || n_hamil < 2 || n_hamil > kMaxComb + 1)
    return fail(SALMON_HIP_EINVAL, "zc null or n_hamil=%d outside 2..%d", n_hamil, kMaxComb + 1);
  if (!tspsi_in || !tspsi_out || !dv_dev || tspsi_in == tspsi_out)
    return fail(SALMON_HIP_EINVAL, "taylor_reuse buffers invalid or aliased");
  if (int rc = ready(c)) return rc;
  const bool mixed = c->prec == SALMON_HIP_PREC_MIXED;
  void *h1 = mixed ? (c->tscr32.empty() ? nullptr : (void *)c->tscr32[0]) : sshtpsi;
  if (!h1 || (!mixed && (sshtpsi == tspsi_in || sshtpsi == tspsi_out)))
    return fail(SALMON_HIP_ESTATE, "taylor_reuse needs H psi of a previous taylor call (sshtpsi, or the FP32 chain)");
  if (mixed) {
    if (int rc = launch_vshift<float2>(c, h1, tspsi_in, dv_dev)) return rc;
    return taylor_mixed(c, zc, n_hamil, tspsi_in, tspsi_out, 2);
  }
  return taylor_fp64(c, zc, n_hamil, tspsi_in, tspsi_out, sshtpsi, 2, dv_dev);
}



int salmon_hip_autotune(salmon_hip_t c, int reps, int *choice, double *best_ms) {
  if (int rc = check(c)) return rc;
  if (int rc = ready(c)) return rc;
  if (reps < 1) reps = 3;
  // two orbital buffers of scratch (zero orbitals: the timing does not depend on the values)
  double2 *bin = nullptr, *bout = nullptr;
  int rc = dalloc(&bin, c->osz * c->norb);
  if (!rc) rc = dalloc(&bout, c->osz * c->norb);
  if (rc) { dfree(bin); return rc; }
  (void)hipMemsetAsync(bin, 0, sizeof(double2) * c->osz * c->norb, c->stream);
  struct Cand { int plane, nzt; };
  const bool save_small = c->small_grid;
  const int save_plane = c->tile_plane, save_nzt = c->mid_nzt;
  // the rule first: it stays unless another shape beats it by more than two runs of one shape differ.  Where the
  // rule takes the whole-orbital kernels it is the only candidate (and H psi in one of them what is timed): the
  // shapes are the per-term kernels'.
  std::vector<Cand> cands{{-1, 0}};
  c->small_grid = true;
  const bool whole = small_step(c, 4) || small_hpsi(c);
  if (!whole) {
    if (c->nx * c->ny <= 1024)
      for (int n : {1, 2}) cands.push_back({1, n});
    for (int n : {1, 2, 4})
      if (n <= std::max(1, c->nz / 8)) cands.push_back({0, n});
  }
  SmallArgs sa = small_args(c, bin, nullptr, bout);
  auto launch = [&]() {
    return whole ? launch_taylor_small(c, SALMON_HIP_KERNEL_HPSI0, sa)
                 : launch_hpsi(c, SALMON_HIP_KERNEL_HPSI0, bin, bout, false, nullptr, 0, nullptr);
  };
  hipEvent_t e0, e1;
  HIPCHK(hipEventCreate(&e0));
  HIPCHK(hipEventCreate(&e1));
  const bool save_prof = c->prof;
  c->prof = false;
  double best = 1e30;
  int besti = 0;
  for (size_t i = 0; i < cands.size() && !rc; ++i) {
    c->tile_plane = cands[i].plane;
    c->mid_nzt = cands[i].nzt;
    // local stencil only (the KB scatter does not depend on the tile shape)
    const int nat = c->natom;
    if (!whole) c->natom = 0;
    rc = launch();
    if (!rc && hipEventRecord(e0, c->stream) != hipSuccess) rc = fail(SALMON_HIP_EHIP, "event record");
    for (int r = 0; r < reps && !rc; ++r) rc = launch();
    c->natom = nat;
    if (rc) break;
    float ms = 0.f;
    if (hipEventRecord(e1, c->stream) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
        hipEventElapsedTime(&ms, e0, e1) != hipSuccess) {
      rc = fail(SALMON_HIP_EHIP, "autotune timing failed");
      break;
    }
    const double t = ms / reps;
    if (t < (besti == 0 ? 0.98 : 1.0) * best) { best = t; besti = (int)i; }
  }
  c->prof = save_prof;
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  (void)hipStreamSynchronize(c->stream);
  dfree(bin);
  dfree(bout);
  if (rc) {
    c->tile_plane = save_plane;
    c->mid_nzt = save_nzt;
    c->small_grid = save_small;
    return rc;
  }
  c->tile_plane = cands[besti].plane;
  c->mid_nzt = cands[besti].nzt;
  if (choice) *choice = 10 * cands[besti].plane + cands[besti].nzt;
  if (best_ms) *best_ms = best;
  return 0;
}

int salmon_hip_set_overlap(salmon_hip_t c, int on) {
  if (int rc = check(c)) return rc;
  if (int rc = join_proj(c)) return rc;
  c->overlap = on != 0;
  return 0;
}

int salmon_hip_set_launch_shape(salmon_hip_t c, int whole_plane, int z_chunks) {
  if (int rc = check(c)) return rc;
  if (whole_plane < -1 || whole_plane > 1 || z_chunks < 0) return fail(SALMON_HIP_EINVAL, "launch shape");
  c->tile_plane = whole_plane;
  c->mid_nzt = z_chunks;
  c->small_grid = whole_plane == -1 && z_chunks == 0;
  return 0;
}

static DensArgs dens_args(salmon_hip_t c, const void *psi, double *rho_dev, double *part) {
  DensArgs a;
  a.psi = (const double2 *)psi;
  a.rocc = c->d_rocc;
  a.wtk = c->d_wtk;
  a.part = part;
  a.rho = rho_dev;
  a.osz = c->osz;
  a.nx = c->nx; a.ny = c->ny; a.nz = c->nz; a.ly = c->ly;
  a.nspin = c->nspin; a.no = c->no; a.nk = c->nk;
  a.ngrp = c->dens_ngrp;
  a.gsz = kDensGroup;
  a.skip = c->d_skip;
  return a;
}

static int density_impl(salmon_hip_t c, const void *psi, double *rho_dev, double *part) {
  const DensArgs a = dens_args(c, psi, rho_dev, part);
  dim3 grid((unsigned)((c->ngrid + kBlock - 1) / kBlock), a.ngrp, c->nspin);
  hipLaunchKernelGGL(k_density_part, grid, dim3(kBlock), 0, c->stream, a);
  LAUNCHCHK("k_density_part");
  if (a.ngrp > 1) {
    dim3 g2((unsigned)((c->ngrid * c->nspin + kBlock - 1) / kBlock));
    hipLaunchKernelGGL(k_density_sum, g2, dim3(kBlock), 0, c->stream, a);
    LAUNCHCHK("k_density_sum");
  }
  return 0;
}

int salmon_hip_density(salmon_hip_t c, const void *psi, double *rho_dev) {
  if (int rc = check(c)) return rc;
  if (!psi || !rho_dev) return fail(SALMON_HIP_EINVAL, "null pointer");
  return density_impl(c, psi, rho_dev, c->d_denspart);
}

int salmon_hip_density_noalloc(salmon_hip_t c, const void *psi, double *rho_dev) {
  if (int rc = check(c)) return rc;
  if (!psi || !rho_dev) return fail(SALMON_HIP_EINVAL, "null pointer");
  if (!c->d_scratch) return fail(SALMON_HIP_ESTATE, "device scratch not resolved");
  const size_t need = c->dens_ngrp > 1 ? c->ngrid * (size_t)c->nspin * (size_t)c->dens_ngrp : 0;
  if (need > kNoAllocScratch)
    return fail(SALMON_HIP_EINVAL,
                "density_noalloc: %zu partial sums (%d groups of %d orbitals x %zu points x %d spins) exceed the "
                "device scratch of %zu doubles",
                need, c->dens_ngrp, kDensGroup, c->ngrid, c->nspin, kNoAllocScratch);
  return density_impl(c, psi, rho_dev, c->d_scratch);
}

static CurArgs cur_args(salmon_hip_t c, const void *psi) {
  CurArgs a;
  a.psi = (const double2 *)psi;
  a.part = c->d_curpart;
  memcpy(a.coef_nab, c->coef_nab, sizeof(a.coef_nab));
  a.osz = c->osz;
  a.nx = c->nx; a.ny = c->ny; a.nz = c->nz; a.ly = c->ly;
  a.TY = c->TY;
  a.nyt = c->nyt;
  return a;
}

static size_t cur_shmem(salmon_hip_t c) { return sizeof(double2) * 2 * (size_t)(c->TY + 4) * c->nx; }

static CurFinArgs curfin_args(salmon_hip_t c, const double *vec_Ac, const double *actab, const int *itt,
                              double *curr_dev, int tmax) {
  CurFinArgs f;
  f.part = c->d_curpart;
  f.nl = c->natom > 0 ? c->d_curnl : nullptr;
  f.rinv = c->d_rinv;
  f.veck = c->d_veck;
  f.rocc = c->d_rocc;
  f.wtk = c->d_wtk;
  f.contrib = c->d_contrib;
  f.curr = curr_dev;
  f.ax = vec_Ac ? vec_Ac[0] : 0.0;
  f.ay = vec_Ac ? vec_Ac[1] : 0.0;
  f.az = vec_Ac ? vec_Ac[2] : 0.0;
  f.actab = actab;
  f.itt = itt;
  f.tmax = tmax;
  f.inv_ngrid = 1.0 / (double)c->ngrid;
  f.nslab = c->nyt;
  f.nspin = c->nspin;
  f.no = c->no;
  f.nk = c->nk;
  f.nlma = c->nlma;
  return f;
}

static size_t small_current_lds(const salmon_hip_ctx *c, int nsub) {
  return sizeof(double2) * c->osz + sizeof(double) * (8 * (size_t)c->nlma * nsub + 4 * (kSmallCurBs / 64));
}

// Whole-orbital current of a small grid; false where its moments do not fit the LDS beside the orbital.
static bool small_current_args(salmon_hip_t c, const void *psi, const CurFinArgs &f, SmallCurArgs &a) {
  a.f = f;
  a.psi = (const double2 *)psi;
  a.zekr = c->d_zekr;
  a.rxyz = c->d_rxyz;
  a.jidx = c->d_jidx;
  a.mps = c->d_mps;
  a.atom_lma = c->d_atom_lma;
  memcpy(a.coef_nab, c->coef_nab, sizeof(a.coef_nab));
  a.osz = c->osz;
  a.nx = c->nx; a.ny = c->ny; a.nz = c->nz; a.ly = c->ly;
  a.natom = c->natom; a.nps = c->nps; a.nlma = c->nlma;
  a.nsub = c->natom > 0 ? std::max(1, kSmallCurBs / 64 / c->natom) : 1;
  return small_current_lds(c, a.nsub) <= kSmallLds;
}

// Where the whole-orbital current is the faster one: a block walks its orbital's points and its atoms' spheres (two
// projectors at a time), which the per-term kernels spread over the chip once the orbitals are many.  The line is
// drawn through 828 random cells (5 of them left more than 5% slower).  Whole orbital against per term: 16^3, 2048
// orbitals of 4, 9 and 16 projectors per atom 81 and 83, 113 and 126, 146 and 159 us, 4096 166 and 146, 241 and 172,
// 319 and 208 us; 18^3, 16 projectors, 1024 orbitals 136 and 172 us, 4096 647 and 335 us; 12^3, 4 projectors, 4096
// orbitals 77 and 101 us.
static bool small_current(const salmon_hip_ctx *c) {
  if (!small_fits(c)) return false;
  if (c->natom == 0) return true;
  const int nsub = std::max(1, kSmallCurBs / 64 / c->natom), ngroup = kSmallCurBs / 64 / nsub;
  const int pts = (int)std::ceil(c->kbval / c->nlma);
  const double chain = (double)((c->natom + ngroup - 1) / ngroup) * ((pts + 64 * nsub - 1) / (64 * nsub)) * ((c->cmax + 1) / 2);
  return c->norb * std::sqrt(chain) * c->ngrid * c->natom / 8 <= 1e8;
}

static int launch_current_small(salmon_hip_t c, const SmallCurArgs &a) {
  static std::atomic<unsigned long long> attr_dev{0};
  if (int rc = lds_attr((const void *)k_current_small, attr_dev, kSmallLds)) return rc;
  hipEvent_t e0, e1;
  prof_events(c, SALMON_HIP_KERNEL_PROJ_CURRENT, &e0, &e1);
  hipExtLaunchKernelGGL(k_current_small, dim3((unsigned)c->norb), dim3(kSmallCurBs), small_current_lds(c, a.nsub), c->stream,
                        e0, e1, 0, a);
  LAUNCHCHK("k_current_small");
  return 0;
}

static int current_impl(salmon_hip_t c, const double *vec_Ac, const double *actab, const int *itt, const void *psi,
                        double *curr_dev, int tmax = 0, bool next = false) {
  if (!actab && !next && small_current(c)) {
    SmallCurArgs a;
    if (small_current_args(c, psi, curfin_args(c, vec_Ac, actab, itt, curr_dev, tmax), a)) {
      if (int rc = launch_current_small(c, a)) return rc;
      for (int is = 0; is < c->nspin; ++is) {
        hipLaunchKernelGGL(k_current_sum, dim3(1), dim3(kBlock), 0, c->stream, a.f, is);
        LAUNCHCHK("k_current_sum");
      }
      return 0;
    }
  }
  const CurArgs a = cur_args(c, psi);
  // the projector moments run on the side stream, overlapping the local part
  if (c->natom > 0)
    if (int rc = launch_proj(c, psi, next ? 5 : 4)) return rc;
  hipLaunchKernelGGL(k_current_local, dim3((unsigned)(c->norb * c->nyt)), dim3(kBlock), cur_shmem(c), c->stream, a);
  LAUNCHCHK("k_current_local");
  if (int rc = join_proj(c)) return rc;
  const CurFinArgs f = curfin_args(c, vec_Ac, actab, itt, curr_dev, tmax);
  const int M = c->no * c->nk;
  for (int is = 0; is < c->nspin; ++is) {
    hipLaunchKernelGGL(k_current_orb, dim3((unsigned)((M + 3) / 4)), dim3(kBlock), 0, c->stream, f, is);
    LAUNCHCHK("k_current_orb");
    hipLaunchKernelGGL(k_current_sum, dim3(1), dim3(kBlock), 0, c->stream, f, is);
    LAUNCHCHK("k_current_sum");
  }
  return 0;
}

int salmon_hip_current(salmon_hip_t c, const double *vec_Ac, const void *psi, double *curr_dev) {
  if (int rc = check(c)) return rc;
  if (!vec_Ac || !psi || !curr_dev) return fail(SALMON_HIP_EINVAL, "null pointer");
  if (c->natom > 0 && !c->have_k) return fail(SALMON_HIP_ESTATE, "update_kvector not called");
  return current_impl(c, vec_Ac, nullptr, nullptr, psi, curr_dev);
}

static DipArgs dip_args(salmon_hip_t c, const double *rho_dev, double *out_dev) {
  DipArgs a;
  a.rho = rho_dev;
  a.part = c->d_dippart;
  a.out = out_dev;
  a.nx = c->nx; a.ny = c->ny; a.nz = c->nz; a.nspin = c->nspin;
  a.hx = c->hgs[0]; a.hy = c->hgs[1]; a.hz = c->hgs[2]; a.hvol = c->hvol;
  return a;
}

int salmon_hip_current_next(salmon_hip_t c, const double *vec_Ac, const void *psi, double *curr_dev,
                            const double *vec_Ac_next) {
  if (int rc = check(c)) return rc;
  if (!vec_Ac || !psi || !curr_dev || !vec_Ac_next) return fail(SALMON_HIP_EINVAL, "null pointer");
  if (c->natom > 0 && !c->have_k) return fail(SALMON_HIP_ESTATE, "update_kvector not called");
  if (c->in_batch) return fail(SALMON_HIP_ESTATE, "current_next on a handle of a batch");
  if (c->natom == 0 || c->nlma == 0) return current_impl(c, vec_Ac, nullptr, nullptr, psi, curr_dev);
  if (!c->d_zekr_n) {
    int rc = dalloc(&c->d_zekr_n, (size_t)c->nps * c->nlma * c->nk);
    if (!rc) rc = dalloc(&c->d_zent_n, (size_t)c->cmax * std::max(c->nent, 1) * c->nk);
    if (!rc && !c->d_kpar_n) rc = dalloc(&c->d_kpar_n, 16 * (size_t)c->nk);
    if (rc) return rc;
  }
  // the next step's phase table and stencil terms into the staging buffers
  KvecArgs ka = kvec_args(c, vec_Ac_next, nullptr, nullptr, 0);
  ka.zekr = c->d_zekr_n;
  ka.zent = c->d_zent_n;
  ka.kpar = c->d_kpar_n;
  hipLaunchKernelGGL(k_update_kvector, dim3(kvec_blocks(ka), c->nk), dim3(kBlock), 0, c->stream, ka);
  LAUNCHCHK("k_update_kvector");
  c->staged = true;
  memcpy(c->staged_A, vec_Ac_next, sizeof(c->staged_A));
  // (the whole-orbital kernels of a small grid form no projection ahead and use none)
  const void *pre = small_step(c, 4) || small_current(c) ? nullptr : psi;
  if (int rc = current_impl(c, vec_Ac, nullptr, nullptr, psi, curr_dev, 0, pre != nullptr)) return rc;
  c->pre_state = pre ? 1 : 0;
  c->pre_psi = pre;
  return 0;
}

int salmon_hip_dipole(salmon_hip_t c, const double *rho_dev, double *out_dev) {
  if (int rc = check(c)) return rc;
  if (!rho_dev || !out_dev) return fail(SALMON_HIP_EINVAL, "null pointer");
  const DipArgs a = dip_args(c, rho_dev, out_dev);
  hipLaunchKernelGGL(k_dipole_part, dim3(kDipBlocks), dim3(256), 0, c->stream, a);
  LAUNCHCHK("k_dipole_part");
  hipLaunchKernelGGL(k_dipole_sum, dim3(1), dim3(256), 0, c->stream, a);
  LAUNCHCHK("k_dipole_sum");
  return 0;
}

int salmon_hip_set_poisson(salmon_hip_t c, const double *al) {
  if (int rc = check(c)) return rc;
  if (!al) return fail(SALMON_HIP_EINVAL, "null pointer");
  for (int d = 0; d < 3; ++d)
    if (!(al[d] > 0.0)) return fail(SALMON_HIP_EINVAL, "cell length al[%d]=%g", d, al[d]);
  const int n[3] = {c->nx, c->ny, c->nz};
  for (int d = 0; d < 3; ++d)
    if (n[d] > kDftMaxN) return fail(SALMON_HIP_EUNSUPPORTED, "grid extent %d above %d", n[d], kDftMaxN);
  const double pi = 3.141592653589793238462643383279502884;
  int rc = 0;
  for (int d = 0; d < 3; ++d) {
    std::vector<double2> tw(n[d]);
    for (int m = 0; m < n[d]; ++m) {
      const double ang = 2.0 * pi * (double)m / (double)n[d];
      tw[m] = make_double2(cos(ang), sin(ang));
    }
    if (!c->d_tw[d] && (rc = dalloc(&c->d_tw[d], tw.size()))) return rc;
    HIPCHK(hipMemcpy(c->d_tw[d], tw.data(), sizeof(double2) * tw.size(), hipMemcpyHostToDevice));
  }
  // fg%coef (src/common/initialization.f90:705-724): index i -> i - n for i >= (n+1)/2
  std::vector<double> coef(c->ngrid);
  for (int kz = 0; kz < c->nz; ++kz)
    for (int ky = 0; ky < c->ny; ++ky)
      for (int kx = 0; kx < c->nx; ++kx) {
        const int ik[3] = {kx, ky, kz};
        double g2 = 0.0;
        for (int d = 0; d < 3; ++d) {
          const int ii = ik[d] >= (n[d] + 1) / 2 ? ik[d] - n[d] : ik[d];
          const double g = (double)ii * (2.0 * pi / al[d]);
          g2 = g2 + g * g;
        }
        coef[(size_t)kx + (size_t)c->nx * ((size_t)ky + (size_t)c->ny * kz)] =
            (kx == 0 && ky == 0 && kz == 0) ? 0.0 : 4.0 * pi / g2;
      }
  if (!c->d_gcoef && (rc = dalloc(&c->d_gcoef, c->ngrid))) return rc;
  HIPCHK(hipMemcpy(c->d_gcoef, coef.data(), sizeof(double) * c->ngrid, hipMemcpyHostToDevice));
  const size_t half = (size_t)c->nx * c->ny * (c->nz / 2 + 1);
  for (double2 *&p : c->d_fft)
    if (!p && (rc = dalloc(&p, half))) return rc;
  c->have_cell = true;
  return 0;
}

}  // extern "C"

// Columns per block of the complex passes: 8 (whole 128-byte lines) while their tile fits, else 4.
static int dft_cols(int n) { return n <= 128 ? 8 : 4; }

// Few columns of many planes: 4 of them per block in the z passes too (16 in the first and 8 in the last leave
// most CUs idle and a thread several rounds of outputs).  Potential update, one and two spins: 12 x 12 x 96 34 and 39
// us with 16 and 8, 23 and 26 us with 4; 16 x 16 x 256 87 and 94 us, 54 and 61 us; 64^3 44 us both, 128^3 200 us
// with 16 and 8, 214 us with 4; 31 x 37 x 41, two spins, 28 and 30 us.
static bool dft_few(int n, int plane) { return n >= 64 && plane <= 4096; }

template <typename F8, typename F4>
static void launch_dft(hipStream_t st, const DftArgs &a, int tiles, int cols, F8 f8, F4 f4) {
  const size_t shm = sizeof(double2) * (size_t)a.n * (1 + tiles * cols);
  const dim3 grid((unsigned)((a.ncols + cols - 1) / cols));
  if (cols == 8) hipLaunchKernelGGL(f8, grid, dim3(256), shm, st, a);
  else hipLaunchKernelGGL(f4, grid, dim3(256), shm, st, a);
}

static VlocArgs vloc_args(salmon_hip_t c, const double *vpsl, const double *vh, const double *vxc, const double *rho,
                          const double *vmix, double *vout) {
  VlocArgs a;
  a.vpsl = vpsl; a.vh = vh; a.vxc = vxc; a.rho = rho; a.vmix = vmix;
  a.V = c->d_V;
  a.vout = vout;
  a.n = c->ngrid;
  a.nspin = c->nspin;
  a.skip = c->d_skip;
  return a;
}

// Hartree potential of rho (+ rho2 when not null: the total density of two spin channels,
// rho_s(1) + rho_s(2), src/rt/time_evolution_step.f90:166-169, formed in the first pass) into vh_dev, or
// where that is null straight into the local potential (v)
static int hartree_impl(salmon_hip_t c, const double *rho_dev, const double *rho2_dev, double *vh_dev, const VlocArgs *v) {
  const int plane = c->nx * c->ny, nkz = c->nz / 2 + 1;
  DftArgs a;
  memset(&a, 0, sizeof(a));
  a.skip = c->d_skip;
  a.coef = c->d_gcoef;
  a.rn = 1.0 / (double)c->ngrid;
  a.sg = -1.0;
  a.rho = rho_dev;
  a.rho2 = rho2_dev;
  a.out = c->d_fft[0];
  a.tw = c->d_tw[2];
  a.n = c->nz; a.inner = plane; a.ncols = plane;
  const bool few = dft_few(c->nz, plane);
  if (few)
    hipLaunchKernelGGL(k_dft_zr<4>, dim3((unsigned)((plane + 3) / 4)), dim3(256), sizeof(double2) * c->nz * 3, c->stream, a);
  else
    hipLaunchKernelGGL(k_dft_zr<16>, dim3((unsigned)((plane + 15) / 16)), dim3(256), sizeof(double2) * c->nz * 9, c->stream, a);
  LAUNCHCHK("k_dft_zr");
  a.in = c->d_fft[0]; a.out = c->d_fft[1];
  a.tw = c->d_tw[1];
  a.n = c->ny; a.inner = c->nx; a.ncols = nkz * c->nx;
  launch_dft(c->stream, a, 1, dft_cols(a.n), k_dft_y<8>, k_dft_y<4>);
  LAUNCHCHK("k_dft_y");
  a.in = a.out = c->d_fft[1];
  a.tw = c->d_tw[0];
  a.n = c->nx; a.inner = 1; a.ncols = nkz * c->ny;
  launch_dft(c->stream, a, 2, dft_cols(a.n), k_dft_x<8>, k_dft_x<4>);
  LAUNCHCHK("k_dft_x");
  a.sg = 1.0;
  a.in = c->d_fft[1]; a.out = c->d_fft[0];
  a.tw = c->d_tw[1];
  a.n = c->ny; a.inner = c->nx; a.ncols = nkz * c->nx;
  launch_dft(c->stream, a, 1, dft_cols(a.n), k_dft_y<8>, k_dft_y<4>);
  LAUNCHCHK("k_dft_y");
  a.in = c->d_fft[0]; a.out = nullptr;
  a.tw = c->d_tw[2];
  a.n = c->nz; a.inner = plane; a.ncols = plane;
  a.vh = vh_dev;
  if (!vh_dev) a.v = *v;
  launch_dft(c->stream, a, 1, few ? 4 : dft_cols(a.n), k_dft_zi<8>, k_dft_zi<4>);
  LAUNCHCHK("k_dft_zi");
  return 0;
}

extern "C" {

int salmon_hip_hartree(salmon_hip_t c, const double *rho_dev, double *vh_dev) {
  if (int rc = check(c)) return rc;
  if (!rho_dev || !vh_dev) return fail(SALMON_HIP_EINVAL, "null pointer");
  if (!c->have_cell) return fail(SALMON_HIP_ESTATE, "set_poisson not called");
  return hartree_impl(c, rho_dev, nullptr, vh_dev, nullptr);
}

int salmon_hip_xc_pz(salmon_hip_t c, const double *rho_dev, double *vxc_dev, double *exc_dev) {
  if (int rc = check(c)) return rc;
  if (!rho_dev || !vxc_dev) return fail(SALMON_HIP_EINVAL, "null pointer");
  hipLaunchKernelGGL(k_xc_pz, dim3((unsigned)((c->ngrid + 255) / 256)), dim3(256), 0, c->stream, rho_dev,
                     vxc_dev, exc_dev, c->ngrid, c->nspin);
  LAUNCHCHK("k_xc_pz");
  return 0;
}

int salmon_hip_update_vlocal(salmon_hip_t c, const double *vpsl_dev, const double *vh_dev, const double *vxc_dev,
                             const double *vmix_dev, double *vout_dev) {
  if (int rc = check(c)) return rc;
  if (!vpsl_dev || !vh_dev || !vxc_dev) return fail(SALMON_HIP_EINVAL, "null pointer");
  const VlocArgs a = vloc_args(c, vpsl_dev, vh_dev, vxc_dev, nullptr, vmix_dev, vout_dev);
  hipLaunchKernelGGL(k_update_vlocal, dim3((unsigned)((c->ngrid + 255) / 256)), dim3(256), 0, c->stream, a);
  LAUNCHCHK("k_update_vlocal");
  c->have_V = true;
  return 0;
}

int salmon_hip_vlocal_extrapolate(salmon_hip_t c, double *vold1_dev, double *vold2_dev, double *vout_dev) {
  if (int rc = check(c)) return rc;
  if (!vold1_dev || !vold2_dev) return fail(SALMON_HIP_EINVAL, "null pointer");
  if (!c->have_V) return fail(SALMON_HIP_ESTATE, "V_local not set");
  const size_t n = c->ngrid * (size_t)c->nspin;
  hipLaunchKernelGGL(k_vextrap, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream, c->d_V, vold1_dev,
                     vold2_dev, vout_dev, n);
  LAUNCHCHK("k_vextrap");
  return 0;
}

int salmon_hip_update_potential(salmon_hip_t c, const double *rho_dev, const double *vpsl_dev,
                                const double *vmix_dev, double *vout_dev) {
  if (int rc = check(c)) return rc;
  if (!rho_dev || !vpsl_dev) return fail(SALMON_HIP_EINVAL, "null pointer");
  if (!c->have_cell) return fail(SALMON_HIP_ESTATE, "set_poisson not called");
  const VlocArgs v = vloc_args(c, vpsl_dev, nullptr, nullptr, rho_dev, vmix_dev, vout_dev);
  if (int rc = hartree_impl(c, rho_dev, c->nspin == 2 ? rho_dev + c->ngrid : nullptr, nullptr, &v)) return rc;
  c->have_V = true;
  return 0;
}

// ---------------------------------------------------------------------------
// Batched step over many independent systems (no counterpart in the reference).
// ---------------------------------------------------------------------------
}  // extern "C"

namespace {

// record the per-step observables at the device step counter, advance it
__global__ void k_record(const double *const *csrc, double *const *cdst, const int *cw, const double *const *dsrc,
                         double *const *ddst, const int *nt, int nsys, int *itt) {
  const int i = threadIdx.x;
  const int t = *itt;
  if (i < nsys && t >= 1 && t <= nt[i]) {
    for (int k = 0; k < cw[i]; ++k) cdst[i][(size_t)(t - 1) * cw[i] + k] = csrc[i][k];
    for (int k = 0; k < 4; ++k) ddst[i][(size_t)(t - 1) * 4 + k] = dsrc[i][k];
  }
  __syncthreads();
  if (i == 0) *itt = t + 1;
}

__global__ void k_set_itt(int *itt, int v) { *itt = v; }

template <int HC, int NC>
int launch_packed_t(hipStream_t st, const StencilArgs *sys, const int2 *tiles, int ntiles, int grid) {
  const size_t shmem = stencil_lds_bytes<double2, HC, NC, kTile>();
  static std::atomic<unsigned long long> attr_dev{0};
  if (int rc = lds_attr((const void *)k_stencil_packed<double2, double, double2, HC, NC, kTile>, attr_dev, shmem))
    return rc;
  hipLaunchKernelGGL((k_stencil_packed<double2, double, double2, HC, NC, kTile>), dim3(grid), dim3(kTile), shmem, st,
                     sys, tiles, ntiles);
  LAUNCHCHK("k_stencil_packed");
  return 0;
}

template <int HC>
int launch_packed_hc(hipStream_t st, int nc, const StencilArgs *sys, const int2 *tiles, int ntiles, int grid) {
  if (nc == 4) return launch_packed_t<HC, 4>(st, sys, tiles, ntiles, grid);
  if (nc == 5) return launch_packed_t<HC, 5>(st, sys, tiles, ntiles, grid);
  if constexpr (HC > 2) {  // rows of up to 64 points take the delayed-z tiles there
    switch (nc) {
      case -1: return launch_packed_t<HC, -1>(st, sys, tiles, ntiles, grid);
      case 1: return launch_packed_t<HC, 1>(st, sys, tiles, ntiles, grid);
      case 2: return launch_packed_t<HC, 2>(st, sys, tiles, ntiles, grid);
      case 3: return launch_packed_t<HC, 3>(st, sys, tiles, ntiles, grid);
    }
  }
  return fail(SALMON_HIP_EINVAL, "batch stencil form");
}

int launch_packed(hipStream_t st, int hc, int nc, const StencilArgs *sys, const int2 *tiles, int ntiles, int grid) {
  if (hc <= 1) return launch_packed_hc<1>(st, nc, sys, tiles, ntiles, grid);
  if (hc <= 2) return launch_packed_hc<2>(st, nc, sys, tiles, ntiles, grid);
  if (hc <= 4) return launch_packed_hc<4>(st, nc, sys, tiles, ntiles, grid);
  return launch_packed_hc<8>(st, nc, sys, tiles, ntiles, grid);
}

template <int NCK, int NC>
int launch_packed_z_t(hipStream_t st, const StencilArgs *sys, const int2 *tiles, int ntiles) {
  const size_t shmem = tilez_lds<double2, NCK, NC>();
  static std::atomic<unsigned long long> attr_dev{0};
  if (int rc = lds_attr((const void *)k_stencilz_packed<double2, double, double2, NCK, NC>, attr_dev, shmem))
    return rc;
  hipLaunchKernelGGL((k_stencilz_packed<double2, double, double2, NCK, NC>), dim3(ntiles), dim3(kTile), shmem, st, sys,
                     tiles);
  LAUNCHCHK("k_stencilz_packed");
  return 0;
}

// the delayed-z y tiles, slots of nck 64-element chunks
template <int NC>
int launch_packed_z_n(hipStream_t st, int nck, const StencilArgs *sys, const int2 *tiles, int ntiles) {
  switch (nck) {
    case 8: return launch_packed_z_t<8, NC>(st, sys, tiles, ntiles);
    case 10: return launch_packed_z_t<10, NC>(st, sys, tiles, ntiles);
    default: return launch_packed_z_t<12, NC>(st, sys, tiles, ntiles);
  }
}

int launch_packed_z(hipStream_t st, int nck, int nc, const StencilArgs *sys, const int2 *tiles, int ntiles) {
  switch (nc) {
    case -1: return launch_packed_z_n<-1>(st, nck, sys, tiles, ntiles);
    case 1: return launch_packed_z_n<1>(st, nck, sys, tiles, ntiles);
    case 2: return launch_packed_z_n<2>(st, nck, sys, tiles, ntiles);
    default: return launch_packed_z_n<3>(st, nck, sys, tiles, ntiles);
  }
}

}  // namespace

// ---------------------------------------------------------------------------
// Packed launches of the batched step: one launch runs a kernel body for every system of the
// batch.  The systems' argument records sit in a device array and system s owns the blocks
// [off[s], off[s+1]) of the launch; a block finds its system by binary search over off (block-
// uniform, scalar loads), copies the record and runs the body with its local block index.  The
// ranges of the bodies that order their blocks for the XCDs (projections, fused KB pass) are
// padded to multiples of 8 blocks, so a local block index keeps its XCD (block b runs on XCD
// b % 8); padding blocks return.  The per-system kernels and these run the same bodies on the
// same records (a packed step differs from the per-system one only by the rounding of members that
// take another form there).
// ---------------------------------------------------------------------------
__device__ __forceinline__ int pack_find(const int *off, int nsys, int b) {
  int lo = 0, hi = nsys;  // off[lo] <= b < off[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (off[mid] <= b) lo = mid;
    else hi = mid;
  }
  return lo;
}

__global__ __launch_bounds__(kBlock) void kp_update_kvector(const KvecArgs *args, const int *off, int nsys) {
  const int s = pack_find(off, nsys, blockIdx.x);
  const KvecArgs a = args[s];
  const int lb = (int)blockIdx.x - off[s], gx = max(1, a.natom * a.split);
  update_kvector_body(a, lb % gx, lb / gx);
}

template <int NW, int LMX>
__global__ __launch_bounds__(kBlock, LMX == 4 ? 4 : 2) void kp_proj(const ProjArgs *args, const int *off, int nsys) {
  const int s = pack_find(off, nsys, blockIdx.x);
  const ProjArgs a = args[s];
  const int item = xcd_order((int)blockIdx.x - off[s], off[s + 1] - off[s]);
  if (item >= a.ngrp * a.natom * a.nk) return;
  proj_body<NW, double2, LMX, proj_split(LMX, false)>(a, item);
}

template <int LM>
__global__ __launch_bounds__(kBlock, LM == 4 ? 3 : 2) void kp_proj_scatter(const ProjScatArgs *args, const int *off, int nsys) {
  const int s = pack_find(off, nsys, blockIdx.x);
  const ProjScatArgs A = args[s];
  const int item = xcd_order((int)blockIdx.x - off[s], off[s + 1] - off[s]);
  if (item >= A.p.ngrp * A.p.natom * A.p.nk) return;
  proj_scatter_body<double2, LM, proj_split(LM, false)>(A, item);
}

template <int CM>
__global__ __launch_bounds__(kBlock) void kp_nl_scatter(const ScatterArgs *args, const int *off, int nsys) {
  const int s = pack_find(off, nsys, blockIdx.x);
  const ScatterArgs a = args[s];
  const int lb = (int)blockIdx.x - off[s], gx = (a.ntp + kBlock - 1) / kBlock;
  nl_scatter_body<double2, kScatG, CM>(a, lb % gx, lb / gx);
}

__global__ __launch_bounds__(kBlock) void kp_density_part(const DensArgs *args, const int *off, int nsys) {
  const int s = pack_find(off, nsys, blockIdx.x);
  const DensArgs a = args[s];
  const int lb = (int)blockIdx.x - off[s];
  const int gx = (a.nx * a.ny * a.nz + kBlock - 1) / kBlock;
  density_part_body(a, lb % gx, (lb / gx) % a.ngrp, lb / (gx * a.ngrp));
}

__global__ __launch_bounds__(kBlock) void kp_density_sum(const DensArgs *args, const int *off, int nsys) {
  const int s = pack_find(off, nsys, blockIdx.x);
  const DensArgs a = args[s];
  density_sum_body(a, (int)blockIdx.x - off[s]);
}

__global__ __launch_bounds__(kBlock) void kp_current_local(const CurArgs *args, const int *off, int nsys) {
  const int s = pack_find(off, nsys, blockIdx.x);
  const CurArgs a = args[s];
  current_local_body(a, (int)blockIdx.x - off[s]);
}

__global__ __launch_bounds__(kBlock) void kp_current_orb(const CurFinArgs *args, const int *off, int nsys) {
  const int s = pack_find(off, nsys, blockIdx.x);
  const CurFinArgs a = args[s];
  const int lb = (int)blockIdx.x - off[s], gx = (a.no * a.nk + 3) / 4;
  current_orb_body(a, lb % gx, lb / gx);
}

__global__ __launch_bounds__(kBlock) void kp_current_sum(const CurFinArgs *args, const int *off, int nsys) {
  const int s = pack_find(off, nsys, blockIdx.x);
  const CurFinArgs a = args[s];
  current_sum_body(a, (int)blockIdx.x - off[s]);
}

__global__ __launch_bounds__(256) void kp_dipole_part(const DipArgs *args, const int *off, int nsys) {
  const int s = pack_find(off, nsys, blockIdx.x);
  const DipArgs a = args[s];
  dipole_part_body(a, (int)blockIdx.x - off[s]);
}

__global__ __launch_bounds__(256) void kp_dipole_sum(const DipArgs *args, const int *off, int nsys) {
  const int s = pack_find(off, nsys, blockIdx.x);
  const DipArgs a = args[s];
  dipole_sum_body(a);
}

// one packed launch: device records, block offsets, grid, dynamic LDS
struct Packed {
  void *args = nullptr;
  int *off = nullptr;
  int nblk = 0;
  size_t shmem = 0;
};

struct salmon_hip_batch {
  std::vector<salmon_hip_t> h;
  hipStream_t stream = nullptr;
  struct Sys {
    void *psi[2] = {nullptr, nullptr};
    void *work = nullptr;
    double *rho = nullptr, *curr_t = nullptr, *dip_t = nullptr;
    const double *actab = nullptr;
    int nt = 0;
    double *curr_s = nullptr, *dip_s = nullptr;  // this step's observables (scratch)
  };
  std::vector<Sys> sys;
  struct Group {
    int hc = 1;
    std::vector<int> mem;               // systems of this halo class
    int2 *d_tiles[2] = {nullptr, nullptr};  // middle terms, last term (different z-chunking)
    int ntiles[2] = {0, 0}, grid[2] = {0, 0};
    StencilArgs *d_args = nullptr;      // [parity][term][member]
    int zch = 0;                        // middle terms on the delayed-z kernel, slots of zch 64-element chunks (0: no)
  };
  std::vector<Group> groups;
  int n_hamil = 0;
  std::vector<double> zc;
  int z_chunks = 0;                     // 0: each system's own rule
  int grid_mult = 4;                    // persistent blocks = grid_mult x 256 (capped at the tile count)
  int *d_itt = nullptr;
  int itt = 1;                          // host copy of the step counter (the next step's index)
  int nt_min = 0;                       // steps the shortest field table covers
  // k_record tables
  double **d_csrc = nullptr, **d_cdst = nullptr, **d_dsrc = nullptr, **d_ddst = nullptr;
  int *d_cw = nullptr, *d_nt = nullptr;
  int parity = 0;
  bool prepared = false;
  std::vector<void *> allocs;
  // the per-system kernels of a phase (projections, scatters, observables) run on kLanes side
  // streams forked from and joined back to `stream`, so small systems overlap (captured as
  // parallel branches of the graph)
  std::vector<hipStream_t> lanes;
  std::vector<hipEvent_t> lane_ev;
  hipEvent_t fork_ev = nullptr;
  // packed launches of the per-system phases ([parity] = which orbital buffer is the input;
  // [term] for the fused KB passes); used when every system with projectors runs the fused
  // KB pass, else the step forks per-system launches onto the lanes
  bool packed = false;
  int lm = 4, cm = kScatCM;               // template choices common to the systems
  Packed p_kvec, p_proj[2], p_kbsh[2][kMaxComb], p_kbf[2][kMaxComb], p_last[2];
  Packed p_dpart[2], p_dsum[2], p_proj4[2], p_curl[2], p_curo, p_curs, p_dipp, p_dips;
};

namespace {

constexpr int kLanes = 4;  // side streams of a batch

template <typename T>
int balloc(salmon_hip_batch *b, T **p, size_t n) {
  if (int rc = dalloc(p, std::max<size_t>(n, 1))) return rc;
  b->allocs.push_back((void *)*p);
  return 0;
}

// Taylor buffers of system i at parity p: h[0] = input, h[1] = work, h[2..] = handle scratch, out
void batch_buffers(salmon_hip_batch *b, int i, int p, void **hh, void **out) {
  salmon_hip_t c = b->h[i];
  hh[0] = b->sys[i].psi[p];
  hh[1] = b->sys[i].work;
  for (int n = 2; n < b->n_hamil; ++n) hh[n] = c->tscr[n - 2];
  *out = b->sys[i].psi[1 - p];
}

// (re)build tile lists and descriptor tables for the current z_chunks / grid_mult
int batch_tables(salmon_hip_batch *b) {
  for (auto &g : b->groups) {
    // rows of up to 64 points (hc <= 2) run on the delayed-z tiles, whose slots they fit, with any number of
    // planes (the last term up to order 4); the group takes its largest member's chunk count
    g.zch = 0;
    if (g.hc <= 2)
      for (int i : g.mem) g.zch = std::max(g.zch, tilez_chunks(b->h[i]->TY, b->h[i]->nx));
    // the members' common number of z chunks by tilez_zchunks' measure of the whole group
    int gz = 1;
    double tbest = 0.0;
    for (int n = 1; n <= 16; ++n) {
      double sum = 0.0, lat = 0.0;
      bool fits = n == 1;
      for (int i : g.mem) {
        const salmon_hip_t c = b->h[i];
        const int ni = std::min(n, std::max(1, c->nz / 8));
        fits = fits || ni == n;
        sum += tilez_planes(c->nz, ni) * ((double)c->norb * c->nyt * ni);
        lat = std::max(lat, tilez_planes(c->nz, ni));
      }
      const double t = std::max(0.65 * lat, 0.49 / 256 * sum);
      if (!fits || (n > 1 && t >= tbest)) continue;
      gz = n;
      tbest = t;
    }
    std::vector<int2> tiles[2];
    std::vector<StencilArgs> args;
    for (int p = 0; p < 2; ++p)
      for (int n = 1; n <= b->n_hamil; ++n)
        for (size_t m = 0; m < g.mem.size(); ++m) {
          const int i = g.mem[m];
          salmon_hip_t c = b->h[i];
          void *hh[kMaxComb + 1], *out;
          batch_buffers(b, i, p, hh, &out);
          const bool fin = n == b->n_hamil;
          int bs = 0;
          const int save = c->mid_nzt;
          c->mid_nzt = b->z_chunks;
          StencilArgs a = stencil_args(c, hh[n - 1], fin ? out : hh[n], fin, hh, n - 1, b->zc.data(), &bs, true);
          c->mid_nzt = save;
          if (g.zch) {
            if (b->z_chunks == 0) tilez_set_chunks(a, std::min(gz, std::max(1, a.nz / 8)));
            a.TZ = (a.TZ + 3) / 4 * 4;  // whole groups of four planes (the kernel's loop) but in the last chunk
            a.nzt = (a.nz + a.TZ - 1) / a.TZ;
            a.nblk = c->norb * a.nyt * a.nzt;
          }
          args.push_back(a);
          if (p == 0 && (n == 1 || fin))
            for (int t = 0; t < a.nblk; ++t) {
              // neighbouring tiles on one XCD, as in the per-system launches
              const int n8 = a.nblk / 8, u = t < n8 * 8 ? (t % 8) * n8 + t / 8 : t;
              tiles[fin ? 1 : 0].push_back(make_int2((int)m, u));
            }
        }
    for (int k = 0; k < 2; ++k) {
      dfree(g.d_tiles[k]);
      if (int rc = dalloc(&g.d_tiles[k], tiles[k].size())) return rc;
      HIPCHK(hipMemcpy(g.d_tiles[k], tiles[k].data(), sizeof(int2) * tiles[k].size(), hipMemcpyHostToDevice));
      g.ntiles[k] = (int)tiles[k].size();
      g.grid[k] = std::min(g.ntiles[k], b->grid_mult * 256);
    }
    dfree(g.d_args);
    if (int rc = dalloc(&g.d_args, args.size())) return rc;
    HIPCHK(hipMemcpy(g.d_args, args.data(), sizeof(StencilArgs) * args.size(), hipMemcpyHostToDevice));
  }
  return 0;
}

int batch_stencil(salmon_hip_batch *b, int p, int n) {
  const int nc = n == b->n_hamil ? b->n_hamil - 1 : -1;
  for (auto &g : b->groups) {
    const StencilArgs *args = g.d_args + ((size_t)p * b->n_hamil + (n - 1)) * g.mem.size();
    const int k = nc >= 0 ? 1 : 0;
    const int rc = (nc <= kTilezComb && g.zch) ? launch_packed_z(b->stream, g.zch, nc, args, g.d_tiles[k], g.ntiles[k])
                                               : launch_packed(b->stream, g.hc, nc, args, g.d_tiles[k], g.ntiles[k], g.grid[k]);
    if (rc) return rc;
  }
  return 0;
}

// fork: system i's kernels go to lane i % kLanes after all work enqueued on the batch stream
int batch_fork(salmon_hip_batch *b) {
  HIPCHK(hipEventRecord(b->fork_ev, b->stream));
  for (size_t k = 0; k < b->lanes.size(); ++k) HIPCHK(hipStreamWaitEvent(b->lanes[k], b->fork_ev, 0));
  for (size_t i = 0; i < b->h.size(); ++i) b->h[i]->stream = b->lanes[i % b->lanes.size()];
  return 0;
}

// join: later work on the batch stream waits for every lane
int batch_join(salmon_hip_batch *b) {
  for (size_t i = 0; i < b->h.size(); ++i) b->h[i]->stream = b->stream;
  for (size_t k = 0; k < b->lanes.size(); ++k) {
    HIPCHK(hipEventRecord(b->lane_ev[k], b->lanes[k]));
    HIPCHK(hipStreamWaitEvent(b->stream, b->lane_ev[k], 0));
  }
  return 0;
}

int batch_step(salmon_hip_batch *b, int p) {
  const int N = b->n_hamil;
  const size_t ns = b->h.size();
  int rc = batch_fork(b);
  for (size_t i = 0; i < ns && !rc; ++i) rc = update_kvector_impl(b->h[i], nullptr, b->sys[i].actab, b->d_itt, b->sys[i].nt + 1);
  if (int r2 = batch_join(b)) return r2;
  if (rc) return rc;
  // the KB term of every term but the last runs fused with the next term's projection, so a
  // system's projection phase runs only for the first term (or without the fused pass)
  for (int n = 1; n <= N; ++n) {
    bool any = false;
    for (size_t i = 0; i < ns; ++i) any = any || (b->h[i]->natom > 0 && (n == 1 || !kb_fused_on(b->h[i])));
    if (any) {
      rc = batch_fork(b);
      for (size_t i = 0; i < ns && !rc; ++i) {
        salmon_hip_t c = b->h[i];
        void *hh[kMaxComb + 1], *out;
        batch_buffers(b, (int)i, p, hh, &out);
        if (c->natom > 0 && (n == 1 || !kb_fused_on(c))) rc = launch_proj(c, hh[n - 1], 1);
      }
      if (int r2 = batch_join(b)) return r2;
      if (rc) return rc;
    }
    if (int r2 = batch_stencil(b, p, n)) return r2;
    rc = batch_fork(b);
    for (size_t i = 0; i < ns && !rc; ++i) {
      salmon_hip_t c = b->h[i];
      void *hh[kMaxComb + 1], *out;
      batch_buffers(b, (int)i, p, hh, &out);
      rc = join_proj(c);
      if (!rc && n < N && kb_fused_on(c)) {
        rc = launch_kb_fused(c, hh[n], false);
      } else if (!rc && c->natom > 0 && c->nlma > 0) {
        const double2 sc = n == N ? make_double2(b->zc[2 * (N - 1)], b->zc[2 * (N - 1) + 1]) : make_double2(1.0, 0.0);
        rc = launch_scatter(c, n == N ? out : hh[n], sc);
      }
    }
    if (int r2 = batch_join(b)) return r2;
    if (rc) return rc;
  }
  rc = batch_fork(b);
  for (size_t i = 0; i < ns && !rc; ++i) {
    salmon_hip_t c = b->h[i];
    void *out = b->sys[i].psi[1 - p];
    rc = salmon_hip_density(c, out, b->sys[i].rho);
    if (!rc) rc = current_impl(c, nullptr, b->sys[i].actab, b->d_itt, out, b->sys[i].curr_s, b->sys[i].nt + 1);
    if (!rc) rc = salmon_hip_dipole(c, b->sys[i].rho, b->sys[i].dip_s);
  }
  if (int r2 = batch_join(b)) return r2;
  if (rc) return rc;
  hipLaunchKernelGGL(k_record, dim3(1), dim3(std::max<size_t>(64, (ns + 63) / 64 * 64)), 0, b->stream, b->d_csrc,
                     b->d_cdst, b->d_cw, b->d_dsrc, b->d_ddst, b->d_nt, (int)ns, b->d_itt);
  LAUNCHCHK("k_record");
  return 0;
}

template <typename A>
int pack_make(salmon_hip_batch *b, Packed &P, const std::vector<A> &recs, const std::vector<int> &cnt, bool pad8,
              size_t shmem = 0) {
  const int n = (int)recs.size();
  std::vector<int> off(n + 1, 0);
  for (int i = 0; i < n; ++i) off[i + 1] = off[i] + (pad8 ? (cnt[i] + 7) / 8 * 8 : cnt[i]);
  A *da = nullptr;
  int *doff = nullptr;
  if (int rc = balloc(b, &da, (size_t)n)) return rc;
  if (int rc = balloc(b, &doff, (size_t)n + 1)) return rc;
  HIPCHK(hipMemcpy(da, recs.data(), sizeof(A) * n, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(doff, off.data(), sizeof(int) * (n + 1), hipMemcpyHostToDevice));
  P.args = da;
  P.off = doff;
  P.nblk = off[n];
  P.shmem = shmem;
  return 0;
}

// Records of the packed launches for both buffer parities.  The two c buffers of each handle
// alternate over the Taylor terms exactly as in launch_kb_fused: the first projection writes X,
// the fused pass of term n reads (n odd ? X : Y) and writes the other, the last scatter reads
// what the pass of term N-1 wrote.
int batch_packed_tables(salmon_hip_batch *b) {
  b->packed = false;
  const int ns = (int)b->h.size(), N = b->n_hamil;
  int cmax = 0;
  for (int i = 0; i < ns; ++i) {
    salmon_hip_t c = b->h[i];
    if (c->natom > 0 && c->nlma > 0 && !kb_fused_on(c)) return 0;  // per-system launches on the lanes
    cmax = std::max(cmax, c->natom > 0 ? c->cmax : 0);
  }
  if (cmax > kMaxLmaPerAtom) return 0;
  b->lm = proj_lm(cmax);
  b->cm = cmax > kScatCM ? 0 : kScatCM;  // 0 where it is every larger system's form
  for (salmon_hip_t c : b->h)
    if (c->natom > 0 && c->cmax > kScatCM && !scat_plain(c->cmax, c->nb)) b->cm = kScatCM;
  auto kb = [&](salmon_hip_t c) { return kb_fused_on(c); };
  auto scat_blocks = [&](salmon_hip_t c, int ntp) {
    return ntp > 0 ? ((ntp + kBlock - 1) / kBlock) * c->nk * ((c->nb + kScatG - 1) / kScatG) : 0;
  };
  auto proj_blocks = [&](const ProjArgs &a) { return a.ngrp * a.natom * a.nk; };
  std::vector<int> cnt(ns);
  {
    std::vector<KvecArgs> r(ns);
    long atoms = 0;
    for (int i = 0; i < ns; ++i) {
      r[i] = kvec_args(b->h[i], nullptr, b->sys[i].actab, b->d_itt, b->sys[i].nt + 1);
      atoms += (long)r[i].natom * r[i].nk;
    }
    for (int i = 0; i < ns; ++i) {
      r[i].split = kvec_split(atoms, r[i].cmax);
      cnt[i] = kvec_blocks(r[i]) * r[i].nk;
    }
    if (int rc = pack_make(b, b->p_kvec, r, cnt, false)) return rc;
  }
  size_t kb_shm = 0, cur_shm = 0;
  for (int i = 0; i < ns; ++i) {
    kb_shm = std::max(kb_shm, sizeof(double2) * (size_t)b->h[i]->cmax * proj_orb(proj_split(b->lm, false)));
    cur_shm = std::max(cur_shm, cur_shmem(b->h[i]));
  }
  for (int p = 0; p < 2; ++p) {
    std::vector<ProjArgs> pr(ns), p4(ns);
    std::vector<ScatterArgs> last(ns);
    std::vector<DensArgs> de(ns);
    std::vector<CurArgs> cl(ns);
    std::vector<int> c4(ns), cl_n(ns), cd(ns), cs(ns), cls(ns);
    for (int i = 0; i < ns; ++i) {
      salmon_hip_t c = b->h[i];
      void *hh[kMaxComb + 1], *out;
      batch_buffers(b, i, p, hh, &out);
      pr[i] = proj_args(c, hh[0], c->d_c, proj_split(b->lm, false));
      cnt[i] = kb(c) ? proj_blocks(pr[i]) : 0;
      const double2 *cl_buf = ((N - 1) % 2 == 1) ? c->d_c2 : c->d_c;
      last[i] = scatter_args(c, out, make_double2(b->zc[2 * (N - 1)], b->zc[2 * (N - 1) + 1]), cl_buf, false, false);
      cls[i] = kb(c) ? scat_blocks(c, c->ntp) : 0;
      de[i] = dens_args(c, out, b->sys[i].rho, c->d_denspart);
      const int gx = (int)((c->ngrid + kBlock - 1) / kBlock);
      cd[i] = gx * c->dens_ngrp * c->nspin;
      cs[i] = c->dens_ngrp > 1 ? (int)((c->ngrid * c->nspin + kBlock - 1) / kBlock) : 0;
      p4[i] = proj_args(c, out, c->d_curnl, proj_split(b->lm, false));
      c4[i] = c->natom > 0 ? proj_blocks(p4[i]) : 0;
      cl[i] = cur_args(c, out);
      cl_n[i] = c->norb * c->nyt;
    }
    if (int rc = pack_make(b, b->p_proj[p], pr, cnt, true)) return rc;
    if (int rc = pack_make(b, b->p_last[p], last, cls, false)) return rc;
    if (int rc = pack_make(b, b->p_dpart[p], de, cd, false)) return rc;
    if (int rc = pack_make(b, b->p_dsum[p], de, cs, false)) return rc;
    if (int rc = pack_make(b, b->p_proj4[p], p4, c4, true)) return rc;
    if (int rc = pack_make(b, b->p_curl[p], cl, cl_n, false, cur_shm)) return rc;
    for (int n = 1; n < N; ++n) {
      std::vector<ScatterArgs> sh(ns);
      std::vector<ProjScatArgs> fu(ns);
      std::vector<int> shn(ns), fun(ns);
      for (int i = 0; i < ns; ++i) {
        salmon_hip_t c = b->h[i];
        void *hh[kMaxComb + 1], *out;
        batch_buffers(b, i, p, hh, &out);
        const double2 *cin = (n % 2 == 1) ? c->d_c : c->d_c2;
        double2 *cout = (n % 2 == 1) ? c->d_c2 : c->d_c;
        sh[i] = scatter_args(c, hh[n], make_double2(1.0, 0.0), cin, true, false);
        shn[i] = kb(c) ? scat_blocks(c, c->ntp_shared) : 0;
        fu[i] = projscat_args(c, hh[n], cin, cout, proj_split(b->lm, false));
        fun[i] = kb(c) ? proj_blocks(fu[i].p) : 0;
      }
      if (int rc = pack_make(b, b->p_kbsh[p][n - 1], sh, shn, false)) return rc;
      if (int rc = pack_make(b, b->p_kbf[p][n - 1], fu, fun, true, kb_shm)) return rc;
    }
  }
  std::vector<CurFinArgs> cf(ns);
  std::vector<DipArgs> dp(ns);
  std::vector<int> co(ns), csum(ns), dpn(ns, kDipBlocks), dsn(ns, 1);
  for (int i = 0; i < ns; ++i) {
    salmon_hip_t c = b->h[i];
    cf[i] = curfin_args(c, nullptr, b->sys[i].actab, b->d_itt, b->sys[i].curr_s, b->sys[i].nt + 1);
    co[i] = ((c->no * c->nk + 3) / 4) * c->nspin;
    csum[i] = c->nspin;
    dp[i] = dip_args(c, b->sys[i].rho, b->sys[i].dip_s);
  }
  if (int rc = pack_make(b, b->p_curo, cf, co, false)) return rc;
  if (int rc = pack_make(b, b->p_curs, cf, csum, false)) return rc;
  if (int rc = pack_make(b, b->p_dipp, dp, dpn, false)) return rc;
  if (int rc = pack_make(b, b->p_dips, dp, dsn, false)) return rc;
  b->packed = true;
  return 0;
}

#define PACKED_LAUNCH(kern, P, A)                                                                      \
  do {                                                                                                 \
    if ((P).nblk > 0) {                                                                                \
      hipLaunchKernelGGL(kern, dim3((unsigned)(P).nblk), dim3(kBlock), (P).shmem, b->stream,          \
                         (const A *)(P).args, (const int *)(P).off, ns);                               \
      LAUNCHCHK(#kern);                                                                                \
    }                                                                                                  \
  } while (0)

// One step of every system with one launch per phase (the packed stencil per halo class and term).
int batch_step_packed(salmon_hip_batch *b, int p) {
  const int N = b->n_hamil;
  const int ns = (int)b->h.size();
  PACKED_LAUNCH(kp_update_kvector, b->p_kvec, KvecArgs);
  if (b->lm == 4) PACKED_LAUNCH((kp_proj<1, 4>), b->p_proj[p], ProjArgs);
  else if (b->lm == 9) PACKED_LAUNCH((kp_proj<1, 9>), b->p_proj[p], ProjArgs);
  else PACKED_LAUNCH((kp_proj<1, 16>), b->p_proj[p], ProjArgs);
  for (int n = 1; n <= N; ++n) {
    if (int rc = batch_stencil(b, p, n)) return rc;
    const Packed &S = n < N ? b->p_kbsh[p][n - 1] : b->p_last[p];
    if (b->cm == kScatCM) PACKED_LAUNCH(kp_nl_scatter<kScatCM>, S, ScatterArgs);
    else PACKED_LAUNCH(kp_nl_scatter<0>, S, ScatterArgs);
    if (n < N) {
      const Packed &F = b->p_kbf[p][n - 1];
      if (b->lm == 4) PACKED_LAUNCH(kp_proj_scatter<4>, F, ProjScatArgs);
      else if (b->lm == 9) PACKED_LAUNCH(kp_proj_scatter<9>, F, ProjScatArgs);
      else PACKED_LAUNCH(kp_proj_scatter<16>, F, ProjScatArgs);
    }
  }
  PACKED_LAUNCH(kp_density_part, b->p_dpart[p], DensArgs);
  PACKED_LAUNCH(kp_density_sum, b->p_dsum[p], DensArgs);
  if (b->lm == 4) PACKED_LAUNCH((kp_proj<4, 4>), b->p_proj4[p], ProjArgs);
  else if (b->lm == 9) PACKED_LAUNCH((kp_proj<4, 9>), b->p_proj4[p], ProjArgs);
  else PACKED_LAUNCH((kp_proj<4, 16>), b->p_proj4[p], ProjArgs);
  PACKED_LAUNCH(kp_current_local, b->p_curl[p], CurArgs);
  PACKED_LAUNCH(kp_current_orb, b->p_curo, CurFinArgs);
  PACKED_LAUNCH(kp_current_sum, b->p_curs, CurFinArgs);
  PACKED_LAUNCH(kp_dipole_part, b->p_dipp, DipArgs);
  PACKED_LAUNCH(kp_dipole_sum, b->p_dips, DipArgs);
  hipLaunchKernelGGL(k_record, dim3(1), dim3(std::max<size_t>(64, (ns + 63) / 64 * 64)), 0, b->stream, b->d_csrc,
                     b->d_cdst, b->d_cw, b->d_dsrc, b->d_ddst, b->d_nt, ns, b->d_itt);
  LAUNCHCHK("k_record");
  return 0;
}

int bcheck(salmon_hip_batch_t b) {
  if (!b) return fail(SALMON_HIP_EINVAL, "null batch");
  return 0;
}

}  // namespace

extern "C" {

int salmon_hip_batch_create(const salmon_hip_t *handles, int n, void *stream, salmon_hip_batch_t *out) {
  if (!out || !handles || n < 1 || n > 1024) return fail(SALMON_HIP_EINVAL, "batch of %d systems", n);
  *out = nullptr;
  salmon_hip_batch *b = new salmon_hip_batch();
  for (int i = 0; i < n; ++i)
    if (!handles[i]) { delete b; return fail(SALMON_HIP_EINVAL, "handle %d is null", i); }
  for (int i = 0; i < n; ++i) {
    handles[i]->in_batch = true;
    handles[i]->staged = false;
    handles[i]->pre_state = 0;
  }
  // the null stream cannot be captured into a graph: NULL selects the first handle's own stream
  b->stream = stream ? (hipStream_t)stream : handles[0]->own;
  for (int i = 0; i < n; ++i) {
    b->h.push_back(handles[i]);
    handles[i]->stream = b->stream;
  }
  b->sys.resize(n);
  for (int k = 0; k < std::min(n, kLanes); ++k) {
    hipStream_t st = nullptr;
    hipEvent_t ev = nullptr;
    if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess) {
      salmon_hip_batch_destroy(b);
      return fail(SALMON_HIP_EHIP, "batch lane stream");
    }
    b->lanes.push_back(st);
    if (hipEventCreateWithFlags(&ev, hipEventDisableTiming) != hipSuccess) {
      salmon_hip_batch_destroy(b);
      return fail(SALMON_HIP_EHIP, "batch lane event");
    }
    b->lane_ev.push_back(ev);
  }
  if (hipEventCreateWithFlags(&b->fork_ev, hipEventDisableTiming) != hipSuccess) {
    salmon_hip_batch_destroy(b);
    return fail(SALMON_HIP_EHIP, "batch fork event");
  }
  int rc = balloc(b, &b->d_itt, 1);
  if (!rc) rc = balloc(b, &b->d_csrc, n);
  if (!rc) rc = balloc(b, &b->d_cdst, n);
  if (!rc) rc = balloc(b, &b->d_dsrc, n);
  if (!rc) rc = balloc(b, &b->d_ddst, n);
  if (!rc) rc = balloc(b, &b->d_cw, n);
  if (!rc) rc = balloc(b, &b->d_nt, n);
  for (int i = 0; i < n && !rc; ++i) {
    rc = balloc(b, &b->sys[i].curr_s, 3 * (size_t)handles[i]->nspin);
    if (!rc) rc = balloc(b, &b->sys[i].dip_s, 4);
  }
  if (rc) { salmon_hip_batch_destroy(b); return rc; }
  *out = b;
  return 0;
}

int salmon_hip_batch_destroy(salmon_hip_batch_t b) {
  if (!b) return 0;
  if (b->stream) (void)hipStreamSynchronize(b->stream);
  for (hipStream_t st : b->lanes) (void)hipStreamSynchronize(st);
  for (auto &g : b->groups) { dfree(g.d_tiles[0]); dfree(g.d_tiles[1]); dfree(g.d_args); }
  for (void *p : b->allocs) (void)hipFree(p);
  for (hipStream_t st : b->lanes) (void)hipStreamDestroy(st);
  for (hipEvent_t ev : b->lane_ev) (void)hipEventDestroy(ev);
  if (b->fork_ev) (void)hipEventDestroy(b->fork_ev);
  for (salmon_hip_t c : b->h) {
    c->stream = b->stream;
    c->in_batch = false;
  }
  delete b;
  return 0;
}

int salmon_hip_batch_set_system(salmon_hip_batch_t b, int i, void *psi_a, void *psi_b, void *work, double *rho_dev,
                                const double *ac_dev, int nt, double *curr_t_dev, double *dip_t_dev) {
  if (int rc = bcheck(b)) return rc;
  if (i < 0 || i >= (int)b->h.size()) return fail(SALMON_HIP_EINVAL, "system %d of %zu", i, b->h.size());
  if (!psi_a || !psi_b || !work || !rho_dev || !ac_dev || !curr_t_dev || !dip_t_dev || nt < 1)
    return fail(SALMON_HIP_EINVAL, "system %d: null buffer or nt < 1", i);
  auto &y = b->sys[i];
  y.psi[0] = psi_a; y.psi[1] = psi_b; y.work = work; y.rho = rho_dev; y.actab = ac_dev; y.nt = nt;
  y.curr_t = curr_t_dev; y.dip_t = dip_t_dev;
  b->prepared = false;
  return 0;
}

int salmon_hip_batch_prepare(salmon_hip_batch_t b, const double *zc, int n_hamil) {
  if (int rc = bcheck(b)) return rc;
  if (!zc || n_hamil < 2 || n_hamil > kMaxComb + 1)
    return fail(SALMON_HIP_EINVAL, "zc null or n_hamil=%d outside 2..%d", n_hamil, kMaxComb + 1);
  const int ns = (int)b->h.size();
  for (int i = 0; i < ns; ++i) {
    salmon_hip_t c = b->h[i];
    if (!b->sys[i].psi[0]) return fail(SALMON_HIP_ESTATE, "system %d: set_system not called", i);
    if (!c->have_V) return fail(SALMON_HIP_ESTATE, "system %d: V_local not set", i);
    if (c->prec != SALMON_HIP_PREC_FP64) return fail(SALMON_HIP_EUNSUPPORTED, "batched step is FP64");
    while ((int)c->tscr.size() < n_hamil - 2) {
      double2 *q = nullptr;
      if (int rc = dalloc(&q, c->osz * c->norb)) return rc;
      c->tscr.push_back(q);
    }
    c->have_k = true;  // the phase table is rebuilt from the device field table every step
  }
  b->n_hamil = n_hamil;
  b->zc.assign(zc, zc + 2 * n_hamil);
  for (auto &g : b->groups) { dfree(g.d_tiles[0]); dfree(g.d_tiles[1]); dfree(g.d_args); }
  b->groups.clear();
  for (int i = 0; i < ns; ++i) {
    const int hc = (8 * b->h[i]->nx + kTile - 1) / kTile;
    const int cls = hc <= 1 ? 1 : hc <= 2 ? 2 : hc <= 4 ? 4 : 8;
    salmon_hip_batch::Group *g = nullptr;
    for (auto &q : b->groups)
      if (q.hc == cls) g = &q;
    if (!g) {
      b->groups.push_back(salmon_hip_batch::Group());
      g = &b->groups.back();
      g->hc = cls;
    }
    g->mem.push_back(i);
  }
  if (int rc = batch_tables(b)) return rc;
  if (int rc = batch_packed_tables(b)) return rc;
  std::vector<const double *> cs(ns), ds(ns);
  std::vector<double *> cd(ns), dd(ns);
  std::vector<int> cw(ns), nt(ns);
  for (int i = 0; i < ns; ++i) {
    cs[i] = b->sys[i].curr_s; ds[i] = b->sys[i].dip_s; cd[i] = b->sys[i].curr_t; dd[i] = b->sys[i].dip_t;
    cw[i] = 3 * b->h[i]->nspin; nt[i] = b->sys[i].nt;
  }
  HIPCHK(hipMemcpy(b->d_csrc, cs.data(), sizeof(double *) * ns, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(b->d_dsrc, ds.data(), sizeof(double *) * ns, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(b->d_cdst, cd.data(), sizeof(double *) * ns, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(b->d_ddst, dd.data(), sizeof(double *) * ns, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(b->d_cw, cw.data(), sizeof(int) * ns, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(b->d_nt, nt.data(), sizeof(int) * ns, hipMemcpyHostToDevice));
  b->nt_min = nt[0];
  for (int i = 1; i < ns; ++i) b->nt_min = std::min(b->nt_min, nt[i]);
  b->prepared = true;
  b->parity = 0;
  return salmon_hip_batch_set_time(b, 1);
}

int salmon_hip_batch_set_time(salmon_hip_batch_t b, int itt) {
  if (int rc = bcheck(b)) return rc;
  if (itt < 1 || (b->prepared && itt > b->nt_min + 1))
    return fail(SALMON_HIP_EINVAL, "step index %d outside 1..%d (the field tables cover %d steps)", itt,
                b->nt_min + 1, b->nt_min);
  b->itt = itt;
  hipLaunchKernelGGL(k_set_itt, dim3(1), dim3(1), 0, b->stream, b->d_itt, itt);
  LAUNCHCHK("k_set_itt");
  b->parity = (itt - 1) & 1;
  return 0;
}

int salmon_hip_batch_step(salmon_hip_batch_t b) {
  if (int rc = bcheck(b)) return rc;
  if (!b->prepared) return fail(SALMON_HIP_ESTATE, "batch_prepare not called");
  if (b->itt > b->nt_min)
    return fail(SALMON_HIP_EINVAL, "step %d past the field tables (%d steps)", b->itt, b->nt_min);
  if (int rc = b->packed ? batch_step_packed(b, b->parity) : batch_step(b, b->parity)) return rc;
  b->parity ^= 1;
  b->itt += 1;
  return 0;
}

// Graph capture of the batched step is switched off: one capture (stream capture of the step
// with the per-system launches forked onto side streams and joined by events) ended in a host
// segmentation fault inside the capture whose cause was not found.  Both entry points report
// SALMON_HIP_EUNSUPPORTED; salmon_hip_batch_step runs the same step with eager launches.
int salmon_hip_batch_capture(salmon_hip_batch_t b) {
  if (int rc = bcheck(b)) return rc;
  return fail(SALMON_HIP_EUNSUPPORTED, "graph capture of the batched step is switched off (use batch_step)");
}

int salmon_hip_batch_replay(salmon_hip_batch_t b, int npairs) {
  if (int rc = bcheck(b)) return rc;
  (void)npairs;
  return fail(SALMON_HIP_EUNSUPPORTED, "graph capture of the batched step is switched off (use batch_step)");
}

int salmon_hip_batch_autotune(salmon_hip_batch_t b, int reps, int *choice, double *best_ms) {
  if (int rc = bcheck(b)) return rc;
  if (!b->prepared) return fail(SALMON_HIP_ESTATE, "batch_prepare not called");
  if (reps < 1) reps = 3;
  hipEvent_t e0, e1;
  HIPCHK(hipEventCreate(&e0));
  HIPCHK(hipEventCreate(&e1));
  double best = 1e30;
  int bz = 0, bg = 4;
  int rc = 0;
  // the persistent grid matters only to groups outside the delayed-z form (one block per tile there); without
  // such a group the timed terms are the same launch for every grid, and the default stays
  bool mid = false, last = b->n_hamil - 1 > kTilezComb;  // persistent middle terms; last terms
  for (const auto &g : b->groups) mid = mid || g.zch == 0;
  const std::vector<int> grids = mid ? std::vector<int>{1, 2, 4, 8, 1 << 20} : std::vector<int>{bg};
  for (int z : {0, 1, 2}) {
    for (int gm : grids) {
      b->z_chunks = z;
      b->grid_mult = gm;
      if ((rc = batch_tables(b))) break;
      // middle-term packed stencil of every group (parity 0, term 2: reads h1, writes h2)
      if ((rc = batch_stencil(b, 0, 2))) break;
      if (hipEventRecord(e0, b->stream) != hipSuccess) { rc = fail(SALMON_HIP_EHIP, "event"); break; }
      for (int r = 0; r < reps && !rc; ++r) rc = batch_stencil(b, 0, 2);
      float ms = 0.f;
      if (rc || hipEventRecord(e1, b->stream) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
          hipEventElapsedTime(&ms, e0, e1) != hipSuccess) {
        if (!rc) rc = fail(SALMON_HIP_EHIP, "autotune timing");
        break;
      }
      if (ms / reps < best) { best = ms / reps; bz = z; bg = gm; }
    }
    if (rc) break;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (rc) return rc;
  b->z_chunks = bz;
  b->grid_mult = bg;
  if (int rc2 = batch_tables(b)) return rc2;
  if (choice) *choice = 100 * bz + (bg > 64 || !(mid || last) ? 99 : bg);
  if (best_ms) *best_ms = best;
  return 0;
}

int salmon_hip_prof_start(salmon_hip_t c, int max_launches) {
  if (int rc = check(c)) return rc;
  if (max_launches < 1) return fail(SALMON_HIP_EINVAL, "max_launches=%d", max_launches);
  HIPCHK(hipStreamSynchronize(c->stream));
  while (c->ev.size() < 2 * (size_t)max_launches) {
    hipEvent_t e;
    HIPCHK(hipEventCreate(&e));
    c->ev.push_back(e);
  }
  c->ev_kind.assign(c->ev.size() / 2, -1);
  c->ev_used = 0;
  c->prof = true;
  return 0;
}

int salmon_hip_prof_stop(salmon_hip_t c, int kind, double *total_ms, int *count) {
  if (int rc = check(c)) return rc;
  if (!total_ms || !count) return fail(SALMON_HIP_EINVAL, "null output");
  HIPCHK(hipStreamSynchronize(c->stream));
  double tot = 0.0;
  int n = 0;
  for (size_t i = 0; i < c->ev_used; ++i) {
    if (c->ev_kind[i] != kind) continue;
    float ms = 0.f;
    HIPCHK(hipEventElapsedTime(&ms, c->ev[2 * i], c->ev[2 * i + 1]));
    tot += ms;
    n += 1;
  }
  *total_ms = tot;
  *count = n;
  return 0;
}

int salmon_hip_prof_end(salmon_hip_t c) {
  if (int rc = check(c)) return rc;
  HIPCHK(hipStreamSynchronize(c->stream));
  c->prof = false;
  c->ev_used = 0;
  return 0;
}

int salmon_hip_synchronize(salmon_hip_t c) {
  if (int rc = check(c)) return rc;
  HIPCHK(hipStreamSynchronize(c->side));
  HIPCHK(hipStreamSynchronize(c->stream));
  return 0;
}

int salmon_hip_malloc(void **dptr, size_t bytes) {
  if (!dptr) return fail(SALMON_HIP_EINVAL, "dptr is null");
  hipError_t e = hipMalloc(dptr, bytes);
  if (e != hipSuccess) return fail(SALMON_HIP_ENOMEM, "hipMalloc(%zu): %s", bytes, hipGetErrorString(e));
  return 0;
}

int salmon_hip_free(void *dptr) {
  HIPCHK(hipFree(dptr));
  return 0;
}

int salmon_hip_memcpy_htod(salmon_hip_t c, void *dst, const void *src, size_t bytes) {
  if (int rc = check(c)) return rc;
  HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, c->stream));
  HIPCHK(hipStreamSynchronize(c->stream));
  return 0;
}

int salmon_hip_memcpy_dtoh(salmon_hip_t c, void *dst, const void *src, size_t bytes) {
  if (int rc = check(c)) return rc;
  HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(hipStreamSynchronize(c->stream));
  return 0;
}

}  // extern "C"
