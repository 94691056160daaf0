// Whole-orbital kernels for small grids (included by salmon_hip.hip inside its namespace).
//
// An orbital block of up to 7680 points (one 8-atom cell: 12^3 .. 18^3; the most that the launch classes' threads
// and planes cover) fits the 160 KB of LDS of one CU, so the complete Taylor step of an orbital -- every stencil application, KB projection,
// KB scatter and the Taylor sum -- runs in ONE workgroup without leaving the CU: the orbital is read
// once and written once (plus H psi), instead of one stencil, one projection and one scatter launch
// per term.  Orbitals do not couple inside a Taylor step, so no block waits for another.
//
// Half of it is the stencil (17 LDS reads per point, 11 to 13 cycles per wave read against the 8 of 128 bytes a
// cycle, beside the FP64 sums), a third the latency of the KB tables between the barriers, the rest loads and
// stores: 12^3 x 1024 orbitals 90 us = 48 for the four applications + 26 for the KB passes + 16; 16^3 x 16
// 52 us = 27 + 19 + 6 (orders 1 to 4 with and without projectors).  Measured, one Taylor
// step of order 4 (per-term kernels -> here): 16^3 x 16 orbitals 145 -> 52 us, 12^3 x 1024 225 -> 90 us,
// 16^3 x 1024 446 -> 223 us, 18^3 x 1024 700 -> 428 us; the current: 16^3 x 16 118 -> 13 us, 12^3 x 1024
// 85 -> 24 us.  Where many orbitals carry many projector values the per-term kernels are the faster ones
// (small_step, small_hpsi, small_current).

// ---------------------------------------------------------------------------
// Work split: thread t owns the column (x, y) = t % (nx ny) over PPT consecutive planes from
// PPT (t / (nx ny)), marching in z with the z neighbours in registers; x and y neighbours come from
// LDS, which holds the orbital in its own (padded) layout, so the sphere tables' offsets apply to it
// unchanged.  The KB projection gives one atom to a wave (lanes on sphere points, four projectors at a
// time, sums combined over the lanes in a fixed tree); the KB scatter puts lanes on touched points.
// ---------------------------------------------------------------------------
struct SmallArgs {
  const double2 *psi;      // input orbitals
  double2 *out;            // propagated orbitals, or null (H psi only)
  double2 *h1;             // H psi, written when not null (read instead with first = 2)
  const double *dv;        // first = 2: h1 += dv psi before the later terms (else null)
  const double *V;         // (nx, ny, nz, nspin)
  const double *kpar;      // (16, nk)
  const double2 *zekr;     // (nps, nlma, nk)
  const double2 *zent;     // (cmax, nent, nk)
  const int *jidx;         // (nps, natom)
  const int *mps;          // (natom)
  const int2 *atom_lma;    // (natom)
  const int *jexcl;        // (nps, natom): jidx where one pair covers the point, else -1
  const int4 *tp_shared;   // (ntp_shared): the points that several pairs cover
  const int *pt_lma;       // (nent)
  const double *rinv;      // (nlma)
  double2 zc[kMaxComb + 1];
  double lap[12];          // -coef_lap / 2 (no scalar FP64 multiply: scaled on the host to stay in SGPRs)
  size_t osz;
  int nx, ny, nz, ly, nspin, nb, nk;
  int nterm, first;        // Taylor terms first .. nterm
  int zchunks;             // z chunks of PPT planes per column
  int natom, nps, nlma, nent, cmax, ntp_shared;
  int nsub;                // waves sharing one atom's sphere
  const int *skip;         // device flag: the launch does nothing when it is set (null: never)
};

// v of another lane of the 16-lane row through a DPP move (no LDS traffic)
template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
constexpr int kDppMirror = 0x140, kDppHalfMirror = 0x141, kDppXor2 = 0x4e, kDppXor1 = 0xb1;

// a + a of the lane 32 (ROW = 16: 16) away in the lower half, b + b of it in the upper half
template <int OFF>
__device__ __forceinline__ double swap_add(double a, double b) {
  unsigned al = __double2loint(a), ah = __double2hiint(a), bl = __double2loint(b), bh = __double2hiint(b);
  if constexpr (OFF == 32) {
    const auto l = __builtin_amdgcn_permlane32_swap(al, bl, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(ah, bh, false, false);
    return __hiloint2double(h[0], l[0]) + __hiloint2double(h[1], l[1]);
  } else {
    const auto l = __builtin_amdgcn_permlane16_swap(al, bl, false, false);
    const auto h = __builtin_amdgcn_permlane16_swap(ah, bh, false, false);
    return __hiloint2double(h[0], l[0]) + __hiloint2double(h[1], l[1]);
  }
}

// Sums v[0 .. 7] over the 64 lanes: lane L returns the total of v[4 (L >> 5) + 2 (L >> 4 & 1) + (L >> 3 & 1)]:
// three steps halve the number of live values each, three add the rest of the lanes (partners are the
// mirrored lanes of the 16- and 8-lane rows: every lane is counted once).
__device__ __forceinline__ double wave_sum8(const double (&v)[8]) {
  double a[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) a[i] = swap_add<32>(v[i], v[i + 4]);
  const double b0 = swap_add<16>(a[0], a[2]), b1 = swap_add<16>(a[1], a[3]);
  const bool hi = threadIdx.x & 8;
  double r = (hi ? b1 : b0) + dpp<kDppMirror>(hi ? b0 : b1);
  r += dpp<kDppHalfMirror>(r);
  r += dpp<kDppXor2>(r);
  r += dpp<kDppXor1>(r);
  return r;
}

// element at byte offset o (32 bits: one orbital's block) from a wave-uniform base
template <typename T>
__device__ __forceinline__ T &at(T *base, unsigned o) {
  return *(T *)((char *)base + o);
}
template <typename T>
__device__ __forceinline__ const T &at(const T *base, unsigned o) {
  return *(const T *)((const char *)base + o);
}

// The value, hidden from loop-invariant motion: the addresses derived from it inside a loop are
// recomputed there (one add each) instead of being kept in registers across the loop.
__device__ __forceinline__ unsigned opaque(unsigned v) {
  asm volatile("" : "+v"(v));
  return v;
}

__device__ __forceinline__ void cmac(double2 &acc, const double2 &c, const double2 &z) {
  acc.x += c.x * z.x - c.y * z.y;
  acc.y += c.x * z.y + c.y * z.x;
}

// One 64-point chunk of an atom's sphere and the table values of up to four projectors (point 0's past
// the sphere, the last projector's past theirs): loads alone, not waited for, so that they can be
// issued ahead of a barrier.
struct SmallChunk {
  unsigned jo;  // the point's offset in the orbital block
  int jw;       // the same where this (atom, point) pair covers the point alone, else -1
  double2 z[4];
};
template <typename A>
__device__ __forceinline__ SmallChunk small_chunk(const A &a, const double2 *zk, int ia, int j, int m, int nl) {
  SmallChunk c;
  const unsigned jc = j < m ? j : 0;
  c.jo = at(a.jidx + (size_t)a.nps * ia, 4u * jc);
  c.jw = at(a.jexcl + (size_t)a.nps * ia, 4u * jc);
#pragma unroll
  for (int l = 0; l < 4; ++l) c.z[l] = at(zk + (size_t)a.nps * min(l, nl - 1), 16u * jc);
  return c;
}

// The wave's place in the KB pass: one atom per group of nsub waves, groups taking atoms in turn.
struct SmallWave {
  int lane, sub, ia, ngroup;
};
template <typename A>
__device__ __forceinline__ SmallWave small_wave(const A &a) {
  const unsigned tid = opaque(threadIdx.x);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  SmallWave w;
  w.lane = tid & 63;
  w.sub = wave % a.nsub;
  w.ngroup = (int)(blockDim.x >> 6) / a.nsub;
  w.ia = wave < w.ngroup * a.nsub ? wave / a.nsub : a.natom;  // waves left over have no atom
  return w;
}

// The chunk a wave's KB pass starts with.
template <typename A>
__device__ __forceinline__ SmallChunk small_first(const A &a, int ik) {
  const SmallWave w = small_wave(a);
  const int ia = min(w.ia, a.natom - 1);
  const int2 al = a.atom_lma[ia];
  const double2 *zk = a.zekr + (size_t)a.nps * ((size_t)a.nlma * ik + al.x);
  return small_chunk(a, zk, ia, 64 * w.sub + w.lane, al.y > 0 ? a.mps[ia] : 0, max(1, min(4, al.y)));
}

// c of projector ilma: the sum of the waves' shares
template <typename A>
__device__ __forceinline__ double2 small_c(const A &a, const double2 *part, int ilma) {
  double2 c = part[ilma];
  for (int u = 1; u < a.nsub; ++u) {
    const double2 v = part[u * a.nlma + ilma];
    c.x += v.x;
    c.y += v.y;
  }
  return c;
}

// KB pass on the orbital in LDS.  add: first completes h at the points that this (atom, point) pair
// covers alone, h += sum_lma c zekr in ascending ilma (the points that several pairs cover are complete
// already, SmallShared).  proj: projects the completed h, pnew(sub, l) = rinv(l) sum over the wave's
// share of conj(zekr(j, l)) h(j).  With up to four projectors per atom a point's table values are
// loaded once for both.  PRE: those of the first chunk (k) were loaded ahead of the barrier before, the
// next chunk's are in flight while a chunk is worked on.
template <bool PRE, typename A>
__device__ __forceinline__ void small_kb(const A &a, int ik, double2 *hs, const double2 *part, double2 *pnew, bool add,
                                         bool proj, SmallChunk k) {
  const SmallWave w = small_wave(a);
  const double2 *zk0 = a.zekr + (size_t)a.nps * a.nlma * ik;
  for (int ia = w.ia; ia < a.natom; ia += w.ngroup) {
    const int2 al = a.atom_lma[ia];
    const int m = a.mps[ia];
    const bool one = al.y <= 4;
    if (add && !one) {
      const int *je = a.jexcl + (size_t)a.nps * ia;
      for (int j = 64 * w.sub + w.lane; j < m; j += 64 * a.nsub) {
        const int o = je[j];
        if (o < 0) continue;
        double2 sum = make_double2(0.0, 0.0);
        for (int l = 0; l < al.y; ++l) cmac(sum, small_c(a, part, al.x + l), zk0[(size_t)j + (size_t)a.nps * (al.x + l)]);
        double2 h = hs[o];
        h.x += sum.x;
        h.y += sum.y;
        hs[o] = h;
      }
    }
    if (!proj && !one) continue;
    for (int l0 = 0; l0 < al.y; l0 += 4) {
      const double2 *zk = zk0 + (size_t)a.nps * (al.x + l0);
      const int nl = min(4, al.y - l0);
      const int ival = w.lane >> 3;  // the value of wave_sum8 this lane holds: 2 l + component
      const double rinv = a.rinv[al.x + l0 + min(ival >> 1, nl - 1)];
      double2 c[4];
      if (PRE && add && one) {
#pragma unroll
        for (int l = 0; l < 4; ++l) c[l] = small_c(a, part, al.x + min(l, nl - 1));
      }
      double s[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) s[i] = 0.0;
      if (PRE && (ia != w.ia || l0 > 0)) k = small_chunk(a, zk, ia, 64 * w.sub + w.lane, m, nl);
      for (int j0 = 64 * w.sub; j0 < m; j0 += 64 * a.nsub) {
        const SmallChunk x = PRE ? k : small_chunk(a, zk, ia, j0 + w.lane, m, nl);
        if (PRE && j0 + 64 * a.nsub < m) k = small_chunk(a, zk, ia, j0 + 64 * a.nsub + w.lane, m, nl);
        double2 v = at(hs, 16u * x.jo);
        const bool in = j0 + w.lane < m;
        if (add && one && in && x.jw >= 0) {
          double2 sum = make_double2(0.0, 0.0);
#pragma unroll
          for (int l = 0; l < 4; ++l)
            if (l < nl) cmac(sum, PRE ? c[l] : small_c(a, part, al.x + l), x.z[l]);
          v.x += sum.x;
          v.y += sum.y;
          at(hs, 16u * x.jw) = v;
        }
        if (proj) {
          if (!in) v = make_double2(0.0, 0.0);
#pragma unroll
          for (int l = 0; l < 4; ++l) {
            s[2 * l] += x.z[l].x * v.x + x.z[l].y * v.y;
            s[2 * l + 1] += x.z[l].x * v.y - x.z[l].y * v.x;
          }
        }
      }
      if (proj) {
        const double r = wave_sum8(s);
        if ((w.lane & 7) == 0 && (ival >> 1) < nl)
          ((double *)(pnew + w.sub * a.nlma + al.x + l0 + (ival >> 1)))[ival & 1] = r * rinv;
      }
    }
  }
}

// KB sums of the points that several (atom, point) pairs cover: sum_lma c(lma) zent in ascending ilma
// into ksum (one per point), added to h by the thread that owns the point.  PRE: the loads of a thread's
// first point (its first two entries) were issued before the barrier that completes c.
struct SmallShared {
  int4 inf;
  int lc1;
  double2 z[2][4];
};
template <typename A>
__device__ __forceinline__ void small_shared_load(const A &a, int ik, const int4 *rec, SmallShared &x) {
  const unsigned i = opaque(threadIdx.x);
  if ((int)i >= a.ntp_shared) return;
  x.inf = rec[i];
  const double2 *ze = a.zent + ((size_t)ik * a.nent + x.inf.y) * a.cmax;
  x.lc1 = a.pt_lma[x.inf.y + 1];
  // values past an entry's own count lie within its cmax and are not used
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int l = 0; l < 4; ++l) x.z[q][l] = ze[q * a.cmax + min(l, a.cmax - 1)];
}
template <bool PRE, typename A>
__device__ __forceinline__ void small_shared_sum(const A &a, int ik, const int4 *rec, const double2 *part, double2 *ksum,
                                                 const SmallShared &x) {
  const double2 *zb = a.zent + (size_t)ik * a.nent * a.cmax;
  for (int i = opaque(threadIdx.x); i < a.ntp_shared; i += blockDim.x) {
    const bool pre = PRE && i < (int)blockDim.x;
    const int4 inf = pre ? x.inf : rec[i];
    double2 acc = make_double2(0.0, 0.0);
    auto entry = [&](int lc, const double2 *ze, const double2 (&z)[4]) __attribute__((always_inline)) {
      const int ilma0 = lc & 0xffffff;
      const int cnt = lc >> 24;
#pragma unroll
      for (int l = 0; l < 4; ++l)
        if (l < cnt) cmac(acc, small_c(a, part, ilma0 + l), z[l]);
      for (int l = 4; l < cnt; ++l) cmac(acc, small_c(a, part, ilma0 + l), ze[l]);
    };
    int q = 0;
    if (pre) {
      entry(inf.w, zb + (size_t)inf.y * a.cmax, x.z[0]);
      entry(x.lc1, zb + (size_t)(inf.y + 1) * a.cmax, x.z[1]);
      q = 2;
    }
    for (; q < inf.z; ++q) {
      const double2 *ze = zb + (size_t)(inf.y + q) * a.cmax;
      const int lc = a.pt_lma[inf.y + q];
      double2 z[4];
#pragma unroll
      for (int l = 0; l < 4; ++l) z[l] = ze[min(l, a.cmax - 1)];
      entry(lc, ze, z);
    }
    ksum[i] = acc;
  }
}

// Forms r here and starts no later read before: the compiler otherwise sinks a plane's sum below the
// next planes' LDS reads, whose registers then spill.
__device__ __forceinline__ void pin(double2 &r) {
  asm volatile("" : "+v"(r.x), "+v"(r.y));
  __builtin_amdgcn_sched_barrier(0);
}

// The kernel's arguments read anew: scalars of one phase then need not stay in SGPRs through the
// others (the stencil's 25 coefficients fill half of them).
typedef const SmallArgs __attribute__((address_space(4))) SmallConst;
__device__ __forceinline__ SmallConst *args_again(SmallConst *p) {
  asm volatile("" : "+s"(p));
  return p;
}

template <int PPT, int BSMAX, int MINW>
__global__ __launch_bounds__(BSMAX, MINW) void k_taylor_small(SmallArgs a) {
  extern __shared__ double2 lds[];
  // with 256 registers per lane (two waves per SIMD) table loads are issued ahead of their use
  constexpr bool PRE = MINW == 2;
  SmallConst *args = (SmallConst *)__builtin_amdgcn_kernarg_segment_ptr();
  if (a.skip && *a.skip) return;  // a device-side gate switched this launch off
  double2 *hs = lds;              // osz: h_{n-1}, then h_n
  double2 *part = lds + a.osz;            // nsub x nlma: the waves' shares of the projections of h_{n-1}
  double2 *pnew = part + a.nsub * a.nlma;  // the same of h_n
  double2 *ksum = pnew + a.nsub * a.nlma;  // ntp_shared
  int4 *rec = (int4 *)(ksum + a.ntp_shared);
  // the blocks of one XCD take consecutive orbitals, so that they share a k-point's phase tables
  const int b = xcd_order(blockIdx.x, gridDim.x);
  const int ik = b / a.nb;
  const int ispin = b % a.nspin;
  const int nx = a.nx, ny = a.ny, nz = a.nz;
  const int ncol = nx * ny;
  const bool on = (int)threadIdx.x < ncol * a.zchunks;  // threads without a column repeat the first
  const int zc = on ? threadIdx.x / ncol : 0;
  const int col = on ? threadIdx.x - zc * ncol : 0;
  const int tx = col % nx, ty = col / nx;
  const int z0 = zc * PPT;
  const int npl = on ? min(PPT, nz - z0) : 0;  // this thread's planes
  const size_t orb = (size_t)b * a.osz;
  const double *kp = a.kpar + 16 * ik;
  const double klap0 = kp[0];
  double nab[12], lap[12];
#pragma unroll
  for (int i = 0; i < 12; ++i) {
    nab[i] = kp[1 + i];
    lap[i] = a.lap[i];
  }
  // byte offsets within the orbital block (LDS and global alike) and within V's grid
  const unsigned zs = 16u * nx * a.ly, pend = zs * nz;
  const unsigned p0 = 16u * (tx + nx * ty) + zs * z0, vz = 8u * ncol, v0 = 8u * col + vz * z0;
  // neighbours relative to the own plane's first point: +n in the low, -n in the high half (a plane
  // has at most 64 KB)
  unsigned xo[4], yo[4];
#pragma unroll
  for (int n = 1; n <= 4; ++n) {
    const int xp = tx + n < nx ? tx + n : tx + n - nx, xm = tx >= n ? tx - n : tx - n + nx;
    const int yp = ty + n < ny ? ty + n : ty + n - ny, ym = ty >= n ? ty - n : ty - n + ny;
    xo[n - 1] = 16u * (xp + nx * ty) | 16u * (xm + nx * ty) << 16;
    yo[n - 1] = 16u * (tx + nx * yp) | 16u * (tx + nx * ym) << 16;
  }
  const bool kb = a.natom > 0, shared = a.ntp_shared > 0;
  unsigned slot[(PPT + 1) / 2];  // the own points' places in ksum, plus one (two per word; 0: none)
#pragma unroll
  for (int i = 0; i < (PPT + 1) / 2; ++i) slot[i] = 0;
  if (shared) {
    // found by marking the points in the (still empty) orbital
    unsigned p = opaque(p0);
#pragma unroll
    for (int i = 0; i < PPT; ++i) {
      if (i < npl) at((unsigned *)hs, p) = 0;
      p += zs;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < a.ntp_shared; i += blockDim.x) {
      const int4 t = a.tp_shared[i];
      rec[i] = t;
      at((unsigned *)hs, 16u * t.x) = i + 1;
    }
    __syncthreads();
    p = opaque(p0);
#pragma unroll
    for (int i = 0; i < PPT; ++i) {
      if (i < npl) slot[i / 2] |= at((unsigned *)hs, p) << 16 * (i & 1);
      p += zs;
    }
  }
  double2 acc[PPT];  // the Taylor sum of the own points
  {
    const double2 *psi = a.psi + orb;
    double2 *h1 = a.h1 + orb;
    const double *dv = a.dv + (size_t)ispin * ncol * nz;
    unsigned p = opaque(p0), v = opaque(v0);
#pragma unroll
    for (int i = 0; i < PPT; ++i) {
      acc[i] = make_double2(0.0, 0.0);
      if (i < npl) {
        acc[i] = at(psi, p);
        double2 h = acc[i];
        if (a.first == 2) {  // h_1 from the given H psi with the changed potential
          const double d = at(dv, v);
          h = at(h1, p);
          h.x += d * acc[i].x;
          h.y += d * acc[i].y;
          at(h1, p) = h;
          acc[i].x += a.zc[0].x * h.x - a.zc[0].y * h.y;
          acc[i].y += a.zc[0].x * h.y + a.zc[0].y * h.x;
        }
        at(hs, p) = h;
        p += zs;
        v += vz;
      }
    }
  }
  SmallChunk k;
  if (PRE && kb) k = small_first(*args_again(args), ik);
  __syncthreads();
  for (int n = a.first - 1;; ++n) {
    // here h_n lacks the KB term at the points one pair covers (but for the chain's first orbital)
    if (kb) {
      small_kb<PRE>(*args_again(args), ik, hs, part, pnew, n >= a.first, n < a.nterm, k);
      double2 *t = part;
      part = pnew;
      pnew = t;
    }
    if (n == a.nterm) break;
    SmallShared x;
    if (PRE && shared) small_shared_load(*args_again(args), ik, rec, x);
    __syncthreads();
    if (shared) small_shared_sum<PRE>(*args_again(args), ik, rec, part, ksum, x);
    // h_{n+1} = H_loc h_n; h_n joins the Taylor sum as it is read
    const bool prev = n >= a.first;
    const double2 cp = a.zc[prev ? n - 1 : 0];
    double2 *h1 = prev && n == 1 && a.h1 ? a.h1 + orb : nullptr;
    double2 hn[PPT];
    {
      const double *Vb = a.V + (size_t)ispin * ncol * nz;
      unsigned p = opaque(p0), v = opaque(v0);
      unsigned pl = opaque(zs * z0);  // the plane's first point
      double2 q[PPT + 8];  // own column, planes z0 - 4 .. z0 + PPT + 3
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        unsigned o = p + zs * i - 4 * zs;  // below the first plane: wraps modulo 2^32, above pend
        o += i < 4 && z0 < 4 - i ? pend : 0;
        o -= i > 4 && z0 + i - 4 >= nz ? pend : 0;
        q[i] = at(hs, o);
      }
      double vnext = at(Vb, v);  // V of the plane, loaded one plane ahead
#pragma unroll
      for (int i = 0; i < PPT; ++i) {
        unsigned o = p + 4 * zs;
        o -= o >= pend ? pend : 0;
        q[i + 8] = at(hs, o);
        const bool more = i + 1 < npl;  // planes past the chunk's last repeat it (their values are not stored)
        const double vl = vnext + klap0;
        v += more ? vz : 0;
        if (i + 1 < PPT) vnext = at(Vb, v);
        const double2 t = q[i + 4];
        if (prev) cmac(acc[i], cp, t);
        if (h1 && i < npl) at(h1, p) = t;
        double2 r = make_double2(vl * t.x, vl * t.y);
        // a neighbour at +n adds (lap - i nab) times it, at -n (lap + i nab)
        auto add = [&](const double2 &u, double l, double w) __attribute__((always_inline)) {
          r.x += l * u.x;
          r.y += l * u.y;
          r.x += w * u.y;
          r.y -= w * u.x;
        };
        // eight neighbours' LDS reads are issued together, ahead of the sums that wait on them
        double2 u[8];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          u[m] = at(hs, pl + (xo[m] & 0xffff));
          u[4 + m] = at(hs, pl + (xo[m] >> 16));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          add(u[m], lap[m], nab[m]);
          add(u[4 + m], lap[m], -nab[m]);
        }
        pin(r);
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          u[m] = at(hs, pl + (yo[m] & 0xffff));
          u[4 + m] = at(hs, pl + (yo[m] >> 16));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          add(u[m], lap[4 + m], nab[4 + m]);
          add(u[4 + m], lap[4 + m], -nab[4 + m]);
        }
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          add(q[i + 5 + m], lap[8 + m], nab[8 + m]);
          add(q[i + 3 - m], lap[8 + m], -nab[8 + m]);
        }
        pin(r);
        hn[i] = r;
        p += more ? zs : 0;
        pl += more ? zs : 0;
      }
    }
    __syncthreads();
    {
      unsigned p = opaque(p0);
#pragma unroll
      for (int i = 0; i < PPT; ++i) {
        if (i < npl) {
          const unsigned t = slot[i / 2] >> 16 * (i & 1) & 0xffff;
          if (t) {
            hn[i].x += ksum[t - 1].x;
            hn[i].y += ksum[t - 1].y;
          }
          at(hs, p) = hn[i];
        }
        p += zs;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (PRE && kb) k = small_first(*args_again(args), ik);
    __syncthreads();
  }
  __syncthreads();
  const double2 c = a.zc[a.nterm - 1];
  double2 *out = a.out ? a.out + orb : a.h1 + orb;
  unsigned p = opaque(p0);
#pragma unroll
  for (int i = 0; i < PPT; ++i) {
    if (i < npl) {
      double2 t = at(hs, p);
      if (a.out) {
        cmac(acc[i], c, t);
        t = acc[i];
      }
      at(out, p) = t;
      p += zs;
    }
  }
}

// ---------------------------------------------------------------------------
// Current of one orbital per block (stencil_current and calc_current_nonlocal,
// density_matrix.f90:465-591): the orbital is read once into LDS; the local part takes its forward
// neighbours from there, the nonlocal part forms the four moments of every projector (one wave per
// atom, lanes on sphere points).  Writes the orbital's weighted current to contrib, which
// k_current_sum adds up.  One launch for the moments, the local part and the per-orbital sums.
// ---------------------------------------------------------------------------
struct SmallCurArgs {
  CurFinArgs f;            // weights, fields and the output of the orbital contributions
  const double2 *psi;
  const double2 *zekr;     // (nps, nlma, nk)
  const double *rxyz;      // (3, nps, natom)
  const int *jidx;         // (nps, natom)
  const int *mps;          // (natom)
  const int2 *atom_lma;    // (natom)
  double coef_nab[12];
  size_t osz;
  int nx, ny, nz, ly, natom, nps, nlma, nsub;
};

constexpr int kSmallCurBs = 512;

__global__ __launch_bounds__(kSmallCurBs, 4) void k_current_small(SmallCurArgs a) {
  extern __shared__ double2 lds[];
  double2 *hs = lds;                                   // osz
  double *mom = (double *)(lds + a.osz);               // (8, nlma, nsub): u and u_x, u_y, u_z
  double *red = mom + 8 * (size_t)a.nlma * a.nsub;     // (4, waves)
  const int b = xcd_order(blockIdx.x, gridDim.x);
  const int nb = a.f.no * a.f.nspin;
  const int ik = b / nb, ispin = b % a.f.nspin, io = (b % nb) / a.f.nspin;
  const int nx = a.nx, ny = a.ny, nz = a.nz;
  const int ncol = nx * ny, n = ncol * nz;
  const unsigned zs = 16u * nx * a.ly, pend = zs * nz;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const double2 *psi = a.psi + (size_t)b * a.osz;
  for (int g = tid; g < n; g += kSmallCurBs) {
    const int z = g / ncol, c = g - z * ncol;
    const unsigned p = 16u * c + zs * z;
    at(hs, p) = at(psi, p);
  }
  __syncthreads();
  // moments: sums over the wave's share of conj(zekr) psi and conj(zekr) r psi
  const int ngroup = (kSmallCurBs / 64) / a.nsub, sub = wave % a.nsub;
  for (int ia = wave < ngroup * a.nsub ? wave / a.nsub : a.natom; ia < a.natom; ia += ngroup) {
    const int2 al = a.atom_lma[ia];
    const int m = a.mps[ia];
    const int *jx = a.jidx + (size_t)a.nps * ia;
    const double *rx = a.rxyz + 3 * (size_t)a.nps * ia;
    for (int l0 = 0; l0 < al.y; l0 += 2) {
      const double2 *zk = a.zekr + (size_t)a.nps * ((size_t)a.nlma * ik + al.x + l0);
      const int nl = min(2, al.y - l0);
      double s[2][8];
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i >> 3][i & 7] = 0.0;
      for (int j0 = 64 * sub; j0 < m; j0 += 64 * a.nsub) {
        const bool in = j0 + lane < m;
        const unsigned jc = in ? j0 + lane : 0;
        const unsigned jo = at(jx, 4u * jc);
        const double r[3] = {at(rx, 24u * jc), at(rx, 24u * jc + 8u), at(rx, 24u * jc + 16u)};
        double2 z[2];
#pragma unroll
        for (int l = 0; l < 2; ++l) z[l] = at(zk + (size_t)a.nps * min(l, nl - 1), 16u * jc);
        double2 v = at(hs, 16u * jo);
        if (!in) v = make_double2(0.0, 0.0);
#pragma unroll
        for (int l = 0; l < 2; ++l) {
          const double ux = z[l].x * v.x + z[l].y * v.y, uy = z[l].x * v.y - z[l].y * v.x;
          s[l][0] += ux;
          s[l][1] += uy;
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            s[l][2 + 2 * d] += r[d] * ux;
            s[l][3 + 2 * d] += r[d] * uy;
          }
        }
      }
#pragma unroll
      for (int l = 0; l < 2; ++l) {
        const double r = wave_sum8(s[l]);
        if ((lane & 7) == 0 && l < nl) mom[8 * ((size_t)sub * a.nlma + al.x + l0 + l) + (lane >> 3)] = r;
      }
    }
  }
  // local part
  double s[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  for (int g = tid; g < n; g += kSmallCurBs) {
    const int z = g / ncol, c = g - z * ncol, y = c / nx, x = c - y * nx;
    const unsigned pl = zs * z, p = 16u * c + pl;
    const double2 t = at(hs, p);
    s[0] += t.x * t.x + t.y * t.y;
#pragma unroll
    for (int k = 1; k <= 4; ++k) {
      const unsigned xo = x + k < nx ? 16u * k : 16u * k - 16u * nx;
      const unsigned yo = y + k < ny ? 16u * nx * k : 16u * nx * k - 16u * ncol;
      const unsigned zo = p + zs * k;
      const double2 px = at(hs, p + xo), py = at(hs, p + yo), pz = at(hs, zo < pend ? zo : zo - pend);
      s[1] += a.coef_nab[k - 1] * (t.x * px.y - t.y * px.x);
      s[2] += a.coef_nab[3 + k] * (t.x * py.y - t.y * py.x);
      s[3] += a.coef_nab[7 + k] * (t.x * pz.y - t.y * pz.x);
    }
  }
  {
    const double r = wave_sum8(s);
    if ((lane & 7) == 0 && lane < 32) red[4 * wave + (lane >> 3)] = r;
  }
  __syncthreads();
  if (wave > 0) return;
  // jNL = 2 sum_lma Im(conj(uVpsi_r) uVpsi): lanes on projectors
  double jw[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  for (int l = lane; l < a.nlma; l += 64) {
    double u[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      u[i] = mom[8 * l + i];
      for (int k = 1; k < a.nsub; ++k) u[i] += mom[8 * ((size_t)k * a.nlma + l) + i];
    }
    const double rv = a.f.rinv[l];
#pragma unroll
    for (int d = 0; d < 3; ++d) jw[d] += rv * (u[2 + 2 * d] * u[1] - u[3 + 2 * d] * u[0]);
  }
  // lanes 8 d hold component d's sum
  const double nl = wave_sum8(jw);
  const int d = lane >> 3;
  if ((lane & 7) == 0 && d < 3) {
    double rt = 0.0, sd = 0.0;
    for (int w = 0; w < kSmallCurBs / 64; ++w) {
      rt += red[4 * w];
      sd += red[4 * w + 1 + d];
    }
    double A = d == 0 ? a.f.ax : d == 1 ? a.f.ay : a.f.az;
    if (a.f.actab) A = a.f.actab[3 * min(max(*a.f.itt, 0), a.f.tmax) + d];
    const double j1 = (a.f.veck[3 * ik + d] + A) * rt;
    const double occ = a.f.rocc[io + (size_t)a.f.no * (ik + (size_t)a.f.nk * ispin)];
    const size_t mm = io + (size_t)a.f.no * ik, M = (size_t)a.f.no * a.f.nk;
    a.f.contrib[3 * (mm + M * ispin) + d] = (((j1 + 2.0 * sd) + 2.0 * nl) * occ) * a.f.wtk[ik];
  }
}
