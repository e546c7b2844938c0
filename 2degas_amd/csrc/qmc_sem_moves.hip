// qmc_sem_moves.hip -- the single-electron move kernels (no backflow): see
// qmc_sem.hip for the move, its ratio and the update.
//
// One block of W wavefronts per walker, for the whole call and both spins.  The
// walker's inverse stays in registers, thread (l, c) = (tid / CG, tid % CG)
// holding row l at every CG-th column (MR rows x CG threads).  Three kinds of
// row:
//   RealRow        FP64, real orbitals (spins whose plane waves come with their
//                  opposites): X = R^-1 of the real matrix R (rows cos(g.r),
//                  sin(g.r); qmc_gjr.hip), with the ratio sum_pairs X_c(j)
//                  cos(g.r') + X_s(j) sin(g.r') and the same rank-one update: a
//                  quarter of the complex arithmetic in half of the registers.
//                  A^-1(l, +-g) = (X_c(l) -+ i X_s(l)) / 2, so the caller's
//                  complex inverse is read from the columns of g and written
//                  to both (exactly: the factors are powers of two).
//   CplxRow<double2>, CplxRow<float2>  the complex inverse, FP64 or FP32.
// Every wavefront forms the new orbital column for itself (one sin/cos per
// lane), thread p takes the Jastrow terms of partner p, whose position and
// three-body vector stay in its registers, and what crosses wavefronts (row j',
// the ratio, the Jastrow sums) goes through LDS buffers that alternate between
// moves, so that a move costs one barrier, or none where W is 1 (up to 32 rows
// x 2 threads).  The chain of a move bounds the kernel (new column, table
// loads, sums, exp, decision: waits take 58% of the wavefronts' cycles at N=122
// in FP64, vector issue 47%), so what counts is its length and how many walkers
// a CU holds.  A block of 256 threads with two barriers per move, one launch
// per spin, took 1.99 ms for a sweep of 4096 walkers of N=122 in FP64 and 0.27
// ms for one of 2048 walkers of N=58 with FP32 inverses and u3.  One wavefront
// with whole real rows (64 x 1 threads) needs 128 registers for the row, spilled
// inside the loop and was slower than that.
#include <type_traits>

#include "qmc_sem.h"

// Value of a table's cubic at the pair's grid index and remainder.  (FMAs are
// written out in this file where a sum has two products to choose from or a
// block boundary may part them: the kernels' variants must agree to the bit, as
// a job's results do not depend on the variant its launch takes.)
__device__ __forceinline__ double sem_spline(const DevSys& s, TabRef t, const PairGeo& p) {
  const double4 c = tab_row(s.tab, t, p.ind);
  const double rm = p.rem * s.drti;
  return fma(rm, fma(rm, fma(rm, c.w, c.z), c.y), c.x);
}

__device__ __forceinline__ void sem_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}


// 1/d: hardware reciprocal and two Newton steps (5 instructions where the
// division takes a dozen in one chain).
__device__ __forceinline__ double sem_rcp(double d) {
  double y = __builtin_amdgcn_rcp(d);
  y = fma(y, fma(-d, y, 1.0), y);
  return fma(y, fma(-d, y, 1.0), y);
}

// x plus the neighbouring lanes' x, over the CG threads of a row.
template <int CG>
__device__ __forceinline__ double row_sum(double x) {
  if (CG > 1) x += dpp_f64<0xB1>(x);
  if (CG > 2) x += dpp_f64<0x4E>(x);
  return x;
}
template <int CG>
__device__ __forceinline__ float row_sum(float x) {
  if (CG > 1) x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0xB1, 0xF, 0xF, false));
  if (CG > 2) x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x4E, 0xF, 0xF, false));
  return x;
}

// The spin a block moves: sizes and orbital tables.
struct SemSpin {
  int m, nslot, zero;
  const double* g;   // per lane's column entry: pairs (RealRow) or g-vectors
  const int2* kpm;
};

// Row l of X at pairs cg, cg + CG, ...
template <int MR_, int CG_>
struct RealRow {
  static constexpr int MR = MR_, CG = CG_, EPT = MR / 2 / CG;
  typedef double2 Z;     // the caller's inverse
  typedef double2 Col;   // (cos, sin) of a pair
  typedef double Ratio;
  static constexpr int NCOL = 32;
  double c[EPT], v[EPT];
  double t;

  static __device__ __forceinline__ SemSpin spin(const DevSys& s, int sp) {
    return SemSpin{pick2(s.np, sp), pick2(s.nslot, sp), pick2(s.zslot, sp), sp ? s.gpair[1] : s.gpair[0],
                   sp ? s.kpm[1] : s.kpm[0]};
  }
  static __device__ __forceinline__ int ncol(const SemSpin& q) { return q.nslot; }
  // rows and pairs beyond the spin's read a valid entry and are zeroed
  __device__ __forceinline__ void load(const SemSpin& q, const Z* in, int mm, int l, int cg) {
    in += (int64_t)(l < q.m ? l : 0) * mm;
#pragma unroll
    for (int i = 0; i < EPT; i++) {
      const int sl = cg + CG * i;
      const Z a = in[q.kpm[sl < q.nslot ? sl : 0].x];
      const double f = l < q.m && sl < q.nslot ? (q.zero && sl == 0 ? 1.0 : 2.0) : 0.0;
      c[i] = f * a.x;
      v[i] = q.zero && sl == 0 ? 0.0 : -f * a.y;
    }
  }
  __device__ __forceinline__ void store(const SemSpin& q, Z* out, int mm, int l, int cg) const {
    if (l >= q.m) return;
    out += (int64_t)l * mm;
#pragma unroll
    for (int i = 0; i < EPT; i++) {
      const int sl = cg + CG * i;
      if (sl < q.nslot) {
        const int2 k = q.kpm[sl];
        const bool z = q.zero && sl == 0;
        const double a = z ? c[i] : 0.5 * c[i], b = 0.5 * v[i];
        out[k.x] = make_double2(a, -b);
        if (!z) out[k.y] = make_double2(a, b);
      }
    }
  }
  // t = (X a')_l
  __device__ __forceinline__ Ratio dot(const Col* ap, int cg) {
    double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int i = 0; i < EPT; i++) {
      const Col a = ap[cg + CG * i];
      s[2 * (i & 1)] = fma(c[i], a.x, s[2 * (i & 1)]);
      s[2 * (i & 1) + 1] = fma(v[i], a.y, s[2 * (i & 1) + 1]);
    }
    return t = row_sum<CG>((s[0] + s[1]) + (s[2] + s[3]));
  }
  __device__ __forceinline__ void put(Col* row, int cg) const {
#pragma unroll
    for (int i = 0; i < EPT; i++) row[cg + CG * i] = make_double2(c[i], v[i]);
  }
  static __device__ __forceinline__ double mod2(Ratio r) { return r * r; }
  // X -= (t - e_j') (row j' of X) / R
  __device__ __forceinline__ void update(const Col* row, Ratio r, double, bool mine, int cg) {
    const double f = -(mine ? t - 1.0 : t) * sem_rcp(r);
#pragma unroll
    for (int i = 0; i < EPT; i++) {
      const Col q = row[cg + CG * i];
      c[i] = fma(f, q.x, c[i]);
      v[i] = fma(f, q.y, v[i]);
    }
  }
};

// Row l of A^-1 at columns cg, cg + CG, ...
template <typename Z_, int MR_, int CG_>
struct CplxRow {
  static constexpr int MR = MR_, CG = CG_, EPT = MR / CG;
  typedef Z_ Z;
  typedef Z_ Col;
  typedef Z_ Ratio;
  typedef decltype(Z::x) R;
  static constexpr int NCOL = 64;
  Z b[EPT];
  R tr, ti;

  static __device__ __forceinline__ SemSpin spin(const DevSys& s, int sp) {
    return SemSpin{pick2(s.np, sp), 0, 0, s.gvec, nullptr};
  }
  static __device__ __forceinline__ int ncol(const SemSpin& q) { return q.m; }
  __device__ __forceinline__ void load(const SemSpin& q, const Z* in, int mm, int l, int cg) {
#pragma unroll
    for (int i = 0; i < EPT; i++) {
      const int k = cg + CG * i;
      b[i] = (l < q.m && k < q.m) ? in[l * mm + k] : Z{(R)0, (R)0};
    }
  }
  __device__ __forceinline__ void store(const SemSpin& q, Z* out, int mm, int l, int cg) const {
#pragma unroll
    for (int i = 0; i < EPT; i++) {
      const int k = cg + CG * i;
      if (l < q.m && k < q.m) out[l * mm + k] = b[i];
    }
  }
  // t = (A^-1 a')_l, explicit FMAs into two accumulator pairs (even and odd
  // entries)
  __device__ __forceinline__ Ratio dot(const Col* ap, int cg) {
    R ur = 0, ui = 0;
    tr = ti = 0;
#pragma unroll
    for (int i = 0; i < EPT; i += 2) {
      const Z a = ap[cg + CG * i], a2 = ap[cg + CG * (i + 1)];
      tr = fma(b[i].x, a.x, tr);
      tr = fma(-b[i].y, a.y, tr);
      ti = fma(b[i].x, a.y, ti);
      ti = fma(b[i].y, a.x, ti);
      ur = fma(b[i + 1].x, a2.x, ur);
      ur = fma(-b[i + 1].y, a2.y, ur);
      ui = fma(b[i + 1].x, a2.y, ui);
      ui = fma(b[i + 1].y, a2.x, ui);
    }
    tr = row_sum<CG>(tr + ur);
    ti = row_sum<CG>(ti + ui);
    return Z{tr, ti};
  }
  __device__ __forceinline__ void put(Col* row, int cg) const {
#pragma unroll
    for (int i = 0; i < EPT; i++) row[cg + CG * i] = b[i];
  }
  static __device__ __forceinline__ double mod2(Ratio r) {
    return fma((double)r.x, (double)r.x, (double)r.y * (double)r.y);
  }
  // A^-1 -= (t - e_j') (row j' of A^-1) / R, 1/R as conj(R) / |R|^2
  __device__ __forceinline__ void update(const Col* row, Ratio rz, double m2, bool mine, int cg) {
    const R inv2 = (R)(1.0 / m2);
    const R vr = mine ? tr - (R)1 : tr;
    const R fr = -fma(vr, rz.x, ti * rz.y) * inv2, fi = -fma(ti, rz.x, -(vr * rz.y)) * inv2;
#pragma unroll
    for (int i = 0; i < EPT; i++) {
      const Z q = row[cg + CG * i];
      b[i].x = fma(fr, q.x, b[i].x);
      b[i].x = fma(-fi, q.y, b[i].x);
      b[i].y = fma(fr, q.y, b[i].y);
      b[i].y = fma(fi, q.x, b[i].y);
    }
  }
};

// LDS of a walker; the pairs of buffers alternate between moves.
template <class Row, int W>
struct SemShared {
  typename Row::Col ap[W][Row::NCOL];  // per wavefront: the column at the proposed position
  typename Row::Col row[2][Row::NCOL]; // row j' before the update
  typename Row::Ratio ratio[2];        // R
  double2 gj[2];                       // three-body vector of electron j
  double red[2][W][3];                 // the wavefronts' Jastrow sums
  double2 g[Row::NCOL];                // the columns' plane waves
  double2 step[64];                    // move i's displacement
  double uacc[64];                     // move i's acceptance uniform
  uint64_t rng;                        // the walker's stream
};

// The thread's partner electron (N <= 64 W): position, three-body vector.
struct SemWalk {
  double px, py, gx, gy;
};

template <int W>
__device__ __forceinline__ void sem_sync() {
  if (W > 1) block_sync();
  else sem_wave_sync();
}

// The index of wavefront wv's thread, formed anew at each call: kept from one
// phase to the next, it and what follows from it took the registers of the row.
__device__ __forceinline__ int sem_tid(int wv) {
  int l = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  __asm__ volatile("" : "+v"(l));
  return 64 * wv + l;
}

// Moves of electrons j0..j1-1 of spin sp, in order.  The proposals come first:
// thread i jumps the walker's stream 3i draws ahead and forms move i's Gaussian
// step (Box-Muller) and acceptance uniform.  The log|R| of the accepted moves
// are summed as a product kept as mantissa and exponent (frexp), one log at the
// end.
template <class Row, int W, bool U3, class Sh>
__device__ __forceinline__ void sem_spin(const DevSys& s, Sh& sh, const double* __restrict__ xs, SemWalk& wk, int w,
                                         int wv, int sp, int j0, int j1, const SemJob& jb) {
  typedef typename Row::Col Col;
  int tid = sem_tid(wv);
  const int lane = tid & 63, N = __builtin_amdgcn_readfirstlane(s.nptot);
  const SemSpin q = Row::spin(s, sp);
  const int p0 = pick2(s.ipf, sp), nc = Row::ncol(q);
  const int l = tid / Row::CG, cg = tid % Row::CG;
  const int nmv = j1 - j0;
  sem_sync<W>();
  const uint64_t st0 = sh.rng;
  if (tid < Row::NCOL) sh.g[tid] = tid < nc ? make_double2(q.g[2 * tid], q.g[2 * tid + 1]) : make_double2(0.0, 0.0);
  if (tid < nmv) {
    uint64_t st = (st0 * lcg_pow(3 * tid)) & ((1ULL << 48) - 1ULL);
    const double u1 = rannyu(st), u2 = rannyu(st), ua = rannyu(st);
    double sv, cv;
    qsincos_sreg(6.283185307179586 * u2, &sv, &cv);
    const double rad = jb.sigma * sqrt(-2.0 * sem_log(u1));
    sh.step[tid] = make_double2(rad * cv, rad * sv);
    sh.uacc[tid] = ua;
  }
  Row r;
  r.load(q, (const typename Row::Z*)jb.ainv + ((int64_t)w * 2 + sp) * jb.mm * jb.mm, jb.mm, l, cg);
  // tables of the thread's partner
  const int tp = tpair(sp, ptype(s, tid));
  const TabRef t2 = tabref<TK_U2>(s, tp), t3 = tabref<TK_U3>(s, tp);
  double du_acc = 0.0, pm = 1.0;
  int pe = 0, na = 0;
  sem_sync<W>();
  if (tid == 0) sh.rng = (st0 * lcg_pow(3 * nmv)) & ((1ULL << 48) - 1ULL);
  // (electron j has not moved before its own move: xs holds its position)
  for (int j = j0; j < j1; j++) {
    const int jj = j - p0, b = (j - j0) & 1;
    const double2 dx = sh.step[j - j0], xo = ld2(xs, j);
    const double ua = sh.uacc[j - j0];
    const double xn = xo.x + dx.x, yn = xo.y + dx.y;
    if (lane < Row::NCOL) {
      double sv, cv;
      const double2 g = sh.g[lane];
      qsincos_sreg(fma(g.x, xn, g.y * yn), &sv, &cv);
      sh.ap[wv][lane] = Col{(decltype(Col::x))cv, (decltype(Col::x))sv};
    }
    // the Jastrow change of partner tid: the u2 term and, with U3, the
    // three-body factor's pair term (xi r)^2 and its share of -1/2 sum_p |G_p|^2
    // (G_p changes by dG_p = xi' u' - xi u, u = x_j - x_p folded; G_j becomes
    // -sum_p xi' u')
    double du = 0.0, gjx = 0.0, gjy = 0.0, dgx = 0.0, dgy = 0.0;
    if (tid < N && tid != j) {
      const PairGeo pn = pair_geo(s, xn, yn, wk.px, wk.py), po = pair_geo(s, xo.x, xo.y, wk.px, wk.py);
      if (t2.row0 >= 0) du = sem_spline(s, t2, pn) - sem_spline(s, t2, po);
      if (U3 && t3.row0 >= 0) {
        const double fn = sem_spline(s, t3, pn), fo = sem_spline(s, t3, po);
        const double an = fn * pn.r, ao = fo * po.r;
        dgx = fn * pn.ux - fo * po.ux;
        dgy = fn * pn.uy - fo * po.uy;
        du += (an * an - ao * ao) - (wk.gx * dgx + wk.gy * dgy) - 0.5 * (dgx * dgx + dgy * dgy);
        gjx = -(fn * pn.ux);
        gjy = -(fn * pn.uy);
      }
    }
    sem_wave_sync();
    const typename Row::Ratio tl = r.dot(sh.ap[wv], cg);
    if (l == jj) {
      r.put(sh.row[b], cg);
      if (cg == 0) sh.ratio[b] = tl;
    }
    if (U3 && tid == j) sh.gj[b] = make_double2(wk.gx, wk.gy);
    du = wave_sum(du);
    if (U3) {
      gjx = wave_sum(gjx);
      gjy = wave_sum(gjy);
    }
    if (W > 1 && lane == 0) {
      sh.red[b][wv][0] = du;
      if (U3) {
        sh.red[b][wv][1] = gjx;
        sh.red[b][wv][2] = gjy;
      }
    }
    sem_sync<W>();
    const typename Row::Ratio rr = sh.ratio[b];
    const double mod2 = Row::mod2(rr);
    if (W > 1) {
      // partners are the threads below N: the first two wavefronts
      du = sh.red[b][0][0] + sh.red[b][1 % W][0];
      if (U3) {
        gjx = sh.red[b][0][1] + sh.red[b][1 % W][1];
        gjy = sh.red[b][0][2] + sh.red[b][1 % W][2];
      }
    }
    if (U3) {
      const double2 g = sh.gj[b];
      du -= 0.5 * ((gjx * gjx + gjy * gjy) - (g.x * g.x + g.y * g.y));
    }
    // (the same on every lane: a scalar branch)
    if (__builtin_amdgcn_readfirstlane(ua < mod2 * sem_exp(-2.0 * du))) {
      r.update(sh.row[b], rr, mod2, l == jj, cg);
      if (tid == j) {
        wk.px = xn;
        wk.py = yn;
      }
      if (U3) {
        wk.gx = tid == j ? gjx : wk.gx + dgx;
        wk.gy = tid == j ? gjy : wk.gy + dgy;
      }
      int e;
      pm = frexp(pm * mod2, &e);
      pe += __builtin_amdgcn_readfirstlane(e);
      du_acc += du;
      na++;
    }
    if (W == 1) sem_wave_sync();
  }
  tid = sem_tid(wv);
  r.store(q, (typename Row::Z*)jb.ainv + ((int64_t)w * 2 + sp) * jb.mm * jb.mm, jb.mm, tid / Row::CG, tid % Row::CG);
  if (tid == 0) {
    jb.dlogpsi[w] += 0.5 * fma(pe, 0.6931471805599453, sem_log(pm)) - du_acc;
    jb.nacc[w] += na;
  }
}

// The rows of a spin by kind: rows a spin needs, and f(Row) for the spin's
// class of W wavefronts.  KIND: 0 real, 1 complex FP64, 2 complex FP32.
template <int KIND, int MR, int CG>
struct SemKind {
  typedef CplxRow<double2, MR, CG> Row;
};
template <int MR, int CG>
struct SemKind<0, MR, CG> {
  typedef RealRow<MR, CG> Row;
};
template <int MR, int CG>
struct SemKind<2, MR, CG> {
  typedef CplxRow<float2, MR, CG> Row;
};

// Wavefronts per SIMD the compiler has to fit: the most at which no vector
// register spills (an FP64 row of 32 complex entries takes 128 registers of its
// own, one of 16 half of that, the rest of a move some 60, 80 with u3).  Spills
// cost time (100 registers doubled the sweep's), and correctness: the compiler
// places a spill at the start of the block where diverged lanes join again,
// before it turns them on, so that lanes lose the value.  In the FP32 kernel of
// two wavefronts the sums kept over the call went that way.
template <int KIND, int W, bool U3>
struct SemBound {
  static constexpr int value = KIND == 1 ? (W == 2 ? 2 : U3 ? 3 : 4) : (W == 2 && U3 ? 3 : 4);
};

// The moves of walker w of a job by W wavefronts (wv), both spins in order.
template <int KIND, int W, bool U3, class Sh>
__device__ __forceinline__ void sem_walker(const SemJob& jb, Sh& sh, double* xs, int w, int wv) {
  int tid = sem_tid(wv);
  const DevSys& s = *jb.sys;
  const int N = __builtin_amdgcn_readfirstlane(s.nptot);
  double* xw = jb.x + (int64_t)w * 2 * N;
  SemWalk wk{0.0, 0.0, 0.0, 0.0};
  if (tid < N) {
    wk.px = xs[2 * tid] = xw[2 * tid];
    wk.py = xs[2 * tid + 1] = xw[2 * tid + 1];
  }
  if (tid == 0) sh.rng = (uint64_t)jb.rng[w];
  sem_sync<W>();
  if (U3 && s.has_u3 && tid < N) {
    // G_p = sum_b xi(r_pb) (x_b - x_p), minimum image: the per-particle
    // vector of the three-body factor
    const int tp = ptype(s, tid);
    // (a type at a time and without branches, so that the table loads of several
    // partners are in flight: with a test per partner the vectors took 7 of the
    // 116 us of a spin's call at N=58, 2048 walkers; sweeps 232 -> 206
    // us)
    for (int u = 0; u < s.ntypes; u++) {
      const TabRef a = tabref<TK_U3>(s, tpair(tp, u));
      if (a.row0 < 0) continue;
      const int q1 = pick2(s.ipf, u) + pick2(s.np, u);
#pragma unroll 4
      for (int q = pick2(s.ipf, u); q < q1; q++) {
        const PairGeo g = pair_geo(s, xs[2 * q], xs[2 * q + 1], wk.px, wk.py);
        // (a particle's own entry: the first row, and a distance of 0 turns into
        // no number, which is left out)
        const double4 c = tab_row(s.tab, a, q == tid ? 0 : g.ind);
        const double rm = g.rem * s.drti, f = fma(rm, fma(rm, fma(rm, c.w, c.z), c.y), c.x);
        wk.gx += q == tid ? 0.0 : f * g.ux;
        wk.gy += q == tid ? 0.0 : f * g.uy;
      }
    }
  }
  for (int sp = 0; sp < s.ntypes; sp++) {
    const int m = pick2(s.np, sp), a = max(jb.j0, pick2(s.ipf, sp)), e = min(jb.j1, pick2(s.ipf, sp) + m);
    if (a >= e) continue;
    auto run = [&](auto mr, auto cg) {
      typedef typename SemKind<KIND, decltype(mr)::value, decltype(cg)::value>::Row Row;
      sem_spin<Row, W, U3>(s, sh, xs, wk, w, wv, sp, a, e, jb);
    };
    typedef std::integral_constant<int, 2> C2;
    typedef std::integral_constant<int, 4> C4;
    typedef std::integral_constant<int, 16> R16;
    typedef std::integral_constant<int, 32> R32;
    typedef std::integral_constant<int, 64> R64;
    if constexpr (KIND == 0) {
      // particles and pairs (two rows of R each) must both fit
      const int rows = max(m, 2 * pick2(s.nslot, sp));
      if constexpr (W == 1) {
        if (rows <= 16) run(R16{}, C4{});
        else run(R32{}, C2{});
      } else {
        if (rows <= 32) run(R32{}, C4{});
        else run(R64{}, C2{});
      }
    } else {
      const int c = m <= 16 ? 0 : m <= 32 ? 1 : 2;
      if (c == 0) run(R16{}, C4{});
      else if (c == 1 && (W == 1 || jb.tile[1] == 2)) run(R32{}, C2{});
      else if (W > 1 && c == 1) run(R32{}, C4{});
      else if constexpr (W == 2) run(R64{}, C2{});
      else if constexpr (W == 4) run(R64{}, C4{});
    }
  }
  tid = sem_tid(wv);
  if (tid < N) {
    xw[2 * tid] = wk.px;
    xw[2 * tid + 1] = wk.py;
  }
  if (tid == 0) jb.rng[w] = (int64_t)sh.rng;
}

// One launch moves the walkers of several jobs (contexts of different N, decks
// and walker sets): job k owns the blocks from w0[k] on, one per walker, and
// reads its system description from device memory (uniform loads).  In a launch
// of two wavefronts per block a real-row job that needs one per walker
// (jb.narrow) takes two walkers per block, each wavefront on its own: 12 jobs of
// N=26..74 took 208 us for the wide ones and then 123 us for the others in two
// launches.
template <int KIND, int W, bool U3>
__global__ __launch_bounds__(64 * W, (SemBound<KIND, W, U3>::value)) void k_sem_moves(const SemJobs jobs) {
  typedef typename SemKind<KIND, 16, 4>::Row Any;
  constexpr bool PAIRS = KIND == 0 && W == 2;
  __shared__ union {
    SemShared<Any, W> one;
    SemShared<Any, 1> two[PAIRS ? 2 : 1];
  } sh;
  extern __shared__ __attribute__((aligned(16))) double sr_lds[];  // positions at the start of the call
  int k = 0;
  while (k + 1 < jobs.njobs && (int)blockIdx.x >= jobs.job[k + 1].w0) k++;
  const SemJob& jb = jobs.job[k];
  const int b = blockIdx.x - jb.w0, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if constexpr (PAIRS) {
    if (jb.narrow) {
      const int w = 2 * b + wv;
      if (w < jb.nw) sem_walker<KIND, 1, U3>(jb, sh.two[wv], sr_lds + 2 * wv * jb.sys->nptot, w, 0);
      return;
    }
  }
  sem_walker<KIND, W, U3>(jb, sh.one, sr_lds, b, wv);
}

int launch_sem_moves(const SemJobs& jobs, int nblocks, int kind, int waves, bool u3, int nmax, hipStream_t st) {
  const size_t lds = 2 * (size_t)nmax * sizeof(double);
  auto go = [&](auto k, auto w) {
    constexpr int K = decltype(k)::value, W = decltype(w)::value;
    if (u3) hipLaunchKernelGGL((k_sem_moves<K, W, true>), dim3(nblocks), dim3(64 * W), lds, st, jobs);
    else hipLaunchKernelGGL((k_sem_moves<K, W, false>), dim3(nblocks), dim3(64 * W), lds, st, jobs);
  };
  typedef std::integral_constant<int, 0> I0;
  typedef std::integral_constant<int, 1> I1;
  typedef std::integral_constant<int, 2> I2;
  typedef std::integral_constant<int, 4> I4;
  if (kind == 0) {
    if (waves == 1) go(I0{}, I1{});
    else go(I0{}, I2{});
  } else if (kind == 1) {
    if (waves == 1) go(I1{}, I1{});
    else if (waves == 2) go(I1{}, I2{});
    else go(I1{}, I4{});
  } else {
    if (waves == 1) go(I2{}, I1{});
    else if (waves == 2) go(I2{}, I2{});
    else go(I2{}, I4{});
  }
  HIPCHK(hipGetLastError());
  return QMC_OK;
}
