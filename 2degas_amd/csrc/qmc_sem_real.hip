// qmc_sem_real.hip -- FP64 single-electron moves for real orbitals (spins
// whose plane waves come with their opposites, no backflow): the moves of
// qmc_sem.hip with the inverse of the real matrix R (rows cos(g.r), sin(g.r);
// qmc_gjr.hip), X = R^-1, in place of the complex one.
//
// The ratio is R = sum_pairs X_c(j) cos(g.r') + X_s(j) sin(g.r'), and an
// accepted move updates X by the same rank-one formula: a quarter of the
// complex arithmetic in half of the registers.  A^-1(l, +-g) = (X_c(l) -+
// i X_s(l)) / 2, so the caller's complex inverse is read from the columns of g
// and written to both (exactly: the factors are powers of two).
//
// One block of W wavefronts per walker, for the whole call and both spins:
// thread (l, c) = (tid / CG, tid % CG) holds row l at pairs c, c + CG, ...  A
// walker whose spins have at most 32 rows takes one wavefront (16 x 4 or 32 x 2
// threads, no barrier at all), others two (32 x 4 or 64 x 2) and one barrier
// per move, what crosses it being double buffered; thread p takes the Jastrow
// terms of partner p, whose position and three-body vector stay in its
// registers.  The complex kernel's four wavefronts and two barriers per move
// left the vector units idle half of the time, waiting on its serial chain.
// One wavefront with whole rows (64 x 1 threads) needs 128 registers for the
// row, spilled inside the move loop and was slower than the complex kernel.
// Bound by instruction issue (some 300 per wavefront and move); the inverses'
// 0.98 GB in and out per sweep of 4096 walkers of N=122 take 0.2 ms of HBM time
// beside it.
#include "qmc_sem.h"

// Table row and grid size of a pair term of electrons of type pair tp.
struct SemTab {
  int row0, ng;
};

// Value of a table's cubic at the pair's grid index and remainder.
__device__ __forceinline__ double sem_spline(const DevSys& s, SemTab t, const PairGeo& p) {
  const int i = p.ind < t.ng ? (p.ind > 0 ? p.ind : 0) : t.ng;
  const double4 c = s.tab[t.row0 + i];
  const double rm = p.rem * s.drti;
  return c.x + rm * (c.y + rm * (c.z + rm * c.w));
}

__device__ __forceinline__ void sem_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Keeps the LDS and memory reads of an unrolled loop over the row from being
// issued all at once, which would need as many registers again as the row.
__device__ __forceinline__ void sem_chunk() { __asm__ volatile("" ::: "memory"); }

// LDS of a walker; the pairs of buffers alternate between moves.
template <int W>
struct SemShared {
  double2 ap[W][32];   // per wavefront: cos, sin of the pairs at the proposed position
  double2 row[2][32];  // row j' of X before the update
  double2 gj[2];       // three-body vector of electron j
  double red[2][W][3]; // the wavefronts' Jastrow sums
  double ratio[2];     // R
  double2 step[64];    // move i's displacement
  double uacc[64];     // move i's acceptance uniform
};

// The thread's partner electron (N <= 64 W): position, three-body vector.
struct SemWalk {
  double px, py, gx, gy;
  double dlog, nacc;
};

template <int W>
__device__ __forceinline__ void sem_sync() {
  if (W > 1) __syncthreads();
  else sem_wave_sync();
}

template <int W, int CG, bool U3>
__device__ __forceinline__ void sem_real_spin(const DevSys& s, SemShared<W>& sh, const double* __restrict__ xs,
                                              SemWalk& wk, int w, int sp, int j0, int j1, double sigma, uint64_t& st0,
                                              double2* __restrict__ ainv, int mm) {
  constexpr int MR = 64 * W / CG, EPT = MR / 2 / CG;  // rows, pairs per thread
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, N = s.nptot;
  const int m = pick2(s.np, sp), p0 = pick2(s.ipf, sp);
  const int nslot = pick2(s.nslot, sp), zero = pick2(s.zslot, sp);
  const double* gp = sp ? s.gpair[1] : s.gpair[0];
  const int2* kpm = sp ? s.kpm[1] : s.kpm[0];
  const int l = tid / CG, cg = tid % CG;
  const double gx = lane < nslot ? gp[2 * lane] : 0.0, gy = lane < nslot ? gp[2 * lane + 1] : 0.0;
  const int nmv = j1 - j0;
  sem_sync<W>();
  if (tid < nmv) {
    // the proposal of move tid: a Gaussian step of width sigma per dimension
    uint64_t st = (st0 * lcg_pow(3 * (uint64_t)tid)) & ((1ULL << 48) - 1ULL);
    const double u1 = rannyu(st), u2 = rannyu(st), ua = rannyu(st);
    double sv, cv;
    qsincos_sreg(6.283185307179586 * u2, &sv, &cv);
    const double rad = sigma * sqrt(-2.0 * sem_log(u1));
    sh.step[tid] = make_double2(rad * cv, rad * sv);
    sh.uacc[tid] = ua;
  }
  st0 = (st0 * lcg_pow(3 * (uint64_t)nmv)) & ((1ULL << 48) - 1ULL);
  // the row: X_c, X_s; rows and pairs beyond the spin's read a valid entry and
  // are zeroed
  double xc[EPT], xv[EPT];
  {
    const double2* in = ainv + ((int64_t)w * 2 + sp) * mm * mm + (int64_t)(l < m ? l : 0) * mm;
#pragma unroll
    for (int i = 0; i < EPT; i++) {
      const int sl = cg + CG * i;
      const double2 v = in[kpm[sl < nslot ? sl : 0].x];
      const double f = l < m && sl < nslot ? (zero && sl == 0 ? 1.0 : 2.0) : 0.0;
      xc[i] = f * v.x;
      xv[i] = zero && sl == 0 ? 0.0 : -f * v.y;
      if (i % 4 == 3) sem_chunk();
    }
  }
  // tables of the thread's partner
  const int tp = tpair(sp, ptype(s, tid));
  const TabRef r2 = tabref<TK_U2>(s, tp), r3 = tabref<TK_U3>(s, tp);
  const SemTab t2{r2.row0, r2.ng}, t3{r3.row0, r3.ng};
  double du_acc = 0.0, na = 0.0, pm = 1.0;
  int pe = 0;
  sem_sync<W>();
  for (int j = j0; j < j1; j++) {
    const int jj = j - p0, b = (j - j0) & 1;
    // (electron j has not moved before its own move: xs holds its position)
    const double2 dx = sh.step[j - j0], xo = ld2(xs, j);
    const double xn = xo.x + dx.x, yn = xo.y + dx.y;
    if (lane < 32) {
      double sv, cv;
      qsincos_sreg(gx * xn + gy * yn, &sv, &cv);
      sh.ap[wv][lane] = make_double2(cv, sv);
    }
    // the Jastrow change of partner tid: the u2 term and, with U3, the
    // three-body factor's pair term and its share of -1/2 sum_p |G_p|^2, as in
    // the complex kernel
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
    // t = X a', four accumulators
    double t[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int i = 0; i < EPT; i++) {
      const double2 a = sh.ap[wv][cg + CG * i];
      t[2 * (i & 1)] = fma(xc[i], a.x, t[2 * (i & 1)]);
      t[2 * (i & 1) + 1] = fma(xv[i], a.y, t[2 * (i & 1) + 1]);
      if (i % 4 == 3) sem_chunk();
    }
    double tl = (t[0] + t[1]) + (t[2] + t[3]);
    if (CG > 1) tl += dpp_f64<0xB1>(tl);
    if (CG > 2) tl += dpp_f64<0x4E>(tl);
    if (l == jj) {
#pragma unroll
      for (int i = 0; i < EPT; i++) sh.row[b][cg + CG * i] = make_double2(xc[i], xv[i]);
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
    if (W > 1) {
      du = sh.red[b][0][0] + sh.red[b][W - 1][0];
      if (U3) {
        gjx = sh.red[b][0][1] + sh.red[b][W - 1][1];
        gjy = sh.red[b][0][2] + sh.red[b][W - 1][2];
      }
    }
    if (U3) {
      const double2 g = sh.gj[b];
      du -= 0.5 * ((gjx * gjx + gjy * gjy) - (g.x * g.x + g.y * g.y));
    }
    const double rr = sh.ratio[b], mod2 = rr * rr;
    if (sh.uacc[j - j0] < mod2 * sem_exp(-2.0 * du)) {
      // X -= (t - e_j') (row j' of X) / R
      const double f = -(l == jj ? tl - 1.0 : tl) / rr;
#pragma unroll
      for (int i = 0; i < EPT; i++) {
        const double2 q = sh.row[b][cg + CG * i];
        xc[i] = fma(f, q.x, xc[i]);
        xv[i] = fma(f, q.y, xv[i]);
        if (i % 4 == 3) sem_chunk();
      }
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
      pe += e;
      du_acc += du;
      na += 1.0;
    }
    if (W == 1) sem_wave_sync();
  }
  if (l < m) {
    double2* out = ainv + ((int64_t)w * 2 + sp) * mm * mm + (int64_t)l * mm;
#pragma unroll
    for (int i = 0; i < EPT; i++) {
      const int sl = cg + CG * i;
      if (sl < nslot) {
        const int2 k = kpm[sl];
        const bool z = zero && sl == 0;
        const double c = z ? xc[i] : 0.5 * xc[i], v = 0.5 * xv[i];
        out[k.x] = make_double2(c, -v);
        if (!z) out[k.y] = make_double2(c, v);
      }
      if (i % 4 == 3) sem_chunk();
    }
  }
  wk.dlog += 0.5 * (sem_log(pm) + pe * 0.6931471805599453) - du_acc;
  wk.nacc += na;
}

template <int W, bool U3>
__global__ __launch_bounds__(64 * W, 4) void k_sem_real(const SemJobs jobs) {
  __shared__ SemShared<W> sh;
  extern __shared__ __attribute__((aligned(16))) double sr_lds[];
  int b = 0;
  while (b + 1 < jobs.njobs && (int)blockIdx.x >= jobs.job[b + 1].w0) b++;
  const SemJob& jb = jobs.job[b];
  const DevSys& s = *jb.sys;
  const int w = blockIdx.x - jb.w0, tid = threadIdx.x, N = s.nptot;
  double* xs = sr_lds;  // positions at the start of the call
  double* xw = jb.x + (int64_t)w * 2 * N;
  SemWalk wk{0.0, 0.0, 0.0, 0.0, jb.dlogpsi[w], jb.nacc[w]};
  if (tid < N) {
    wk.px = xs[2 * tid] = xw[2 * tid];
    wk.py = xs[2 * tid + 1] = xw[2 * tid + 1];
  }
  uint64_t st = (uint64_t)jb.rng[w];
  sem_sync<W>();
  if (U3 && s.has_u3 && tid < N) {
    // G_p = sum_b xi(r_pb) (x_b - x_p), minimum image: the per-particle
    // vector of the three-body factor
    const int tp = ptype(s, tid);
    for (int q = 0; q < N; q++) {
      const TabRef a = tabref<TK_U3>(s, tpair(tp, ptype(s, q)));
      if (q == tid || a.row0 < 0) continue;
      const PairGeo g = pair_geo(s, xs[2 * q], xs[2 * q + 1], wk.px, wk.py);
      const double f = sem_spline(s, SemTab{a.row0, a.ng}, g);
      wk.gx += f * g.ux;
      wk.gy += f * g.uy;
    }
  }
  for (int sp = 0; sp < s.ntypes; sp++) {
    const int m = pick2(s.np, sp), a = max(jb.j0, pick2(s.ipf, sp)), e = min(jb.j1, pick2(s.ipf, sp) + m);
    if (a >= e) continue;
    // particles and pairs (two rows of R each) must both fit
    const int rows = max(m, 2 * pick2(s.nslot, sp));
    if (rows <= 16 * W)
      sem_real_spin<W, 4, U3>(s, sh, xs, wk, w, sp, a, e, jb.sigma, st, (double2*)jb.ainv, jb.mm);
    else
      sem_real_spin<W, 2, U3>(s, sh, xs, wk, w, sp, a, e, jb.sigma, st, (double2*)jb.ainv, jb.mm);
  }
  if (tid < N) {
    xw[2 * tid] = wk.px;
    xw[2 * tid + 1] = wk.py;
  }
  if (tid == 0) {
    jb.rng[w] = (int64_t)st;
    jb.dlogpsi[w] = wk.dlog;
    jb.nacc[w] = wk.nacc;
  }
}

int launch_sem_real(const SemJobs& jobs, int nblocks, bool u3, bool wide, int nmax, hipStream_t st) {
  const size_t lds = 2 * (size_t)nmax * sizeof(double);
  auto go = [&](auto w) {
    constexpr int W = decltype(w)::value;
    if (u3) hipLaunchKernelGGL((k_sem_real<W, true>), dim3(nblocks), dim3(64 * W), lds, st, jobs);
    else hipLaunchKernelGGL((k_sem_real<W, false>), dim3(nblocks), dim3(64 * W), lds, st, jobs);
  };
  if (wide) go(std::integral_constant<int, 2>{});
  else go(std::integral_constant<int, 1>{});
  HIPCHK(hipGetLastError());
  return QMC_OK;
}
