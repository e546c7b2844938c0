// qmc_sem.hip -- single-electron VMC moves.  For trial functions without
// backflow (every backflow table zero, so quasi-coordinates are positions),
// with the two- and three-body Jastrow factors: Sherman-Morrison updates of
// the inverse Slater matrices.  With backflow: each move evaluates the
// proposal's log|psi| (further below).  The reference has no such move: its
// move displaces every electron and recomputes everything
// (reptation.f:4617-4680).  Checked against the full evaluation (the log|psi|
// change of every accepted move) and statistically against the all-electron
// walk.
//
// Moving electron j of spin s from r to r' changes column j' (its index in
// the spin) of A(k, j) = exp(i g_k . r_j) to a' and nothing else, so the
// determinant ratio is R = (A^-1 a')_j' and
// A'^-1 = A^-1 - (A^-1 a' - e_j') (row j' of A^-1) / R.  The Jastrow ratio is
// exp(-dU), dU = sum_p u(|r' - r_p|) - u(|r - r_p|) plus, with u3, the change
// of the three-body term sum_pairs (xi r)^2 - 1/2 sum_p |G_p|^2 of the full
// evaluation, G_p = sum_b xi(r_pb) (x_b - x_p), which needs only the O(N)
// changed pair terms and the stored G.  The move is accepted with
// probability |R|^2 exp(-2 dU) (a symmetric Gaussian proposal).
//
// The inverses live in HBM between calls ([nw][2][mm][mm] complex, row =
// particle, column = orbital), in FP64 or, with QMC_PREC_MIXED, in FP32 (the
// ratio and the update in FP32, the Jastrow and positions in FP64), and are
// recomputed in FP64 by qmc_sem_refresh (Gauss-Jordan with partial pivoting).
#include <algorithm>
#include <cstring>

#include "qmc_sem.h"

template <typename Z>
struct SemZ;
template <>
struct SemZ<double2> {
  typedef double R;
};
template <>
struct SemZ<float2> {
  typedef float R;
};

// The inverse of A for (walker, spin sp): one workgroup of MR x CG threads
// per walker, A(l, k) = exp(i g_l . r_k) built in registers with the layout
// of the move kernel (thread (l, c) keeps row l at columns c, c + CG, ...),
// inverted by Gauss-Jordan exchange steps with partial pivoting, in FP64.
// Step c pivots on the row p not yet used with the largest |re| + |im| in
// column c (ties: the lowest row) and exchanges row p's output with column
// c's input: T(p, c) <- 1 / piv, T(p, k) <- -T(p, k) / piv,
// T(r, c) <- T(r, c) / piv, T(r, k) <- T(r, k) - T(r, c) T(p, k) / piv.
// After the m steps, with p_c the pivot row of step c,
// A^-1(c, p_c') = T(p_c, c'), which the threads store as they hold it.
// Rows are never moved: the pivot search is a lane-shuffle argmax per
// wavefront and one over the wavefronts in LDS, the pivot row goes through
// LDS, and each thread updates its own entries; two barriers per step.
template <typename Z, int MR, int CG>
__global__ __launch_bounds__(MR* CG) void k_sem_inverse(DevSys s, int sp, const double* __restrict__ x,
                                                        Z* __restrict__ ainv, int mm) {
  typedef typename SemZ<Z>::R R;
  constexpr int T = MR * CG, EPT = MR / CG, NWV = T / 64 > 0 ? T / 64 : 1;
  __shared__ double2 prow[MR];  // pivot row of the step
  __shared__ double cbest[NWV];
  __shared__ int cidx[NWV];
  __shared__ int pr[MR], rk[MR];  // pivot row of step c, step of pivot row l
  const int w = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int m = pick2(s.np, sp), p0 = pick2(s.ipf, sp);
  const int l = tid / CG, cg = tid % CG;
  const double* xw = x + ((int64_t)w * s.nptot + p0) * 2;
  const double gx = l < m ? s.gvec[2 * l] : 0.0, gy = l < m ? s.gvec[2 * l + 1] : 0.0;
  double2 b[EPT];
#pragma unroll
  for (int i = 0; i < EPT; i++) {
    const int k = cg + CG * i;
    b[i] = make_double2(0.0, 0.0);
    if (l < m && k < m) {
      double sv, cv;
      qsincos(gx * xw[2 * k] + gy * xw[2 * k + 1], &sv, &cv);
      b[i] = make_double2(cv, sv);
    }
  }
  bool used = l >= m;
#pragma unroll
  for (int i = 0; i < EPT; i++) {
    for (int c4 = 0; c4 < CG; c4++) {
      const int c = CG * i + c4;
      if (c >= m) break;
      // T(l, c), held by the thread of row l with cg == c4
      const int src = (lane & ~(CG - 1)) | c4;
      const double2 f = make_double2(__shfl(b[i].x, src, 64), __shfl(b[i].y, src, 64));
      double mag = used ? -1.0 : fabs(f.x) + fabs(f.y);
      int idx = l;
#pragma unroll
      for (int o = CG; o < 64; o <<= 1) {
        const double om = __shfl_xor(mag, o, 64);
        const int oi = __shfl_xor(idx, o, 64);
        if (om > mag || (om == mag && oi < idx)) {
          mag = om;
          idx = oi;
        }
      }
      if (lane == 0) {
        cbest[wv] = mag;
        cidx[wv] = idx;
      }
      block_sync();
      double bm = cbest[0];
      int p = cidx[0];
#pragma unroll
      for (int k = 1; k < NWV; k++)
        if (cbest[k] > bm || (cbest[k] == bm && cidx[k] < p)) {
          bm = cbest[k];
          p = cidx[k];
        }
      // the pivot row's threads share u_k = T(p, k) / piv (k != c) and, in
      // column c, 1 / piv; every thread then updates its entries from them
      if (l == p) {
        const double dd = 1.0 / (f.x * f.x + f.y * f.y);
        const double2 ip = make_double2(f.x * dd, -f.y * dd);
#pragma unroll
        for (int ii = 0; ii < EPT; ii++) {
          const int k = cg + CG * ii;
          const double2 q = b[ii];
          prow[k] = k == c ? ip : make_double2(q.x * ip.x - q.y * ip.y, q.x * ip.y + q.y * ip.x);
        }
        used = true;
        if (cg == 0) rk[p] = c;
      }
      if (tid == 0) pr[c] = p;
      block_sync();
#pragma unroll
      for (int ii = 0; ii < EPT; ii++) {
        const int k = cg + CG * ii;
        const double2 u = prow[k];
        if (l == p) b[ii] = k == c ? u : make_double2(-u.x, -u.y);
        else if (k == c) b[ii] = make_double2(f.x * u.x - f.y * u.y, f.x * u.y + f.y * u.x);
        else b[ii] = make_double2(fma(-f.x, u.x, fma(f.y, u.y, b[ii].x)), fma(-f.x, u.y, fma(-f.y, u.x, b[ii].y)));
      }
    }
  }
  block_sync();
  if (l < m) {
    Z* out = ainv + ((int64_t)w * 2 + sp) * mm * mm + (int64_t)rk[l] * mm;
#pragma unroll
    for (int i = 0; i < EPT; i++) {
      const int k = cg + CG * i;
      if (k < m) out[pr[k]] = Z{(R)b[i].x, (R)b[i].y};
    }
  }
}

template <typename Z, int MR>
static int launch_sem_inverse(qmc_ctx* c, const qmc_walkers* w, const qmc_sem_state* d, int sp, int mm,
                              hipStream_t st) {
  hipLaunchKernelGGL((k_sem_inverse<Z, MR, 4>), dim3(w->nw), dim3(MR * 4), 0, st, c->s, sp, w->x, (Z*)d->ainv, mm);
  HIPCHK(hipGetLastError());
  return QMC_OK;
}

template <typename Z>
static int sem_inverse_spin(qmc_ctx* c, const qmc_walkers* w, const qmc_sem_state* d, int sp, int mm,
                            hipStream_t st) {
  const int m = c->s.np[sp];
  if (m <= 16) return launch_sem_inverse<Z, 16>(c, w, d, sp, mm, st);
  if (m <= 32) return launch_sem_inverse<Z, 32>(c, w, d, sp, mm, st);
  return launch_sem_inverse<Z, 64>(c, w, d, sp, mm, st);
}

static int sem_mm(const qmc_ctx* c) { return std::max(c->s.np[0], c->s.ntypes > 1 ? c->s.np[1] : 0); }

// The context's system description in device memory, sent again before a
// launch that reads it only when it has changed since it was last sent (new
// g-vectors, time step or tuning): a blocking copy, after the work already
// queued on the stream that may still read the old one.
static int upload_sys(qmc_ctx* c, hipStream_t st) {
  if (c->sys_valid && memcmp(&c->sys_sent, &c->s, sizeof(DevSys)) == 0) return QMC_OK;
  HIPCHK(hipStreamSynchronize(st));
  HIPCHK(hipMemcpy(c->d_sys, &c->s, sizeof(DevSys), hipMemcpyHostToDevice));
  c->sys_sent = c->s;
  c->sys_valid = true;
  return QMC_OK;
}

static int sem_class(int m) { return m <= 16 ? 0 : m <= 32 ? 1 : 2; }

extern "C" int qmc_sem_set_tile(qmc_ctx* c, int precision, int rows, int threads_per_row) {
  if (!c) return arg_fail("null context");
  if (precision != QMC_PREC_FP64 && precision != QMC_PREC_MIXED) return arg_fail("unknown precision mode");
  const int cls = rows == 16 ? 0 : rows == 32 ? 1 : rows == 64 ? 2 : -1;
  if (cls < 0) return arg_fail("row class must be 16, 32 or 64");
  if (threads_per_row != 4 && (threads_per_row != 2 || cls == 0))
    return arg_fail("threads per row must be 4, or 2 for the 32- and 64-row classes");
  c->sem_cg[precision == QMC_PREC_MIXED ? 1 : 0][cls] = threads_per_row;
  return QMC_OK;
}

static int sem_check(qmc_ctx* c, const qmc_walkers* w, const qmc_sem_state* d, int precision) {
  if (!c || !w || !d || w->nw < 0) return arg_fail("null argument");
  if (w->nw > 0 && (!w->x || !w->rng || !d->dlogpsi || !d->nacc))
    return arg_fail("null buffer for single-electron moves");
  if (precision != QMC_PREC_FP64 && precision != QMC_PREC_MIXED) return arg_fail("unknown precision mode");
  if (!c->s.has_det) return arg_fail("single-electron moves need the Slater determinants");
  if (c->b_zero) {
    if (w->nw > 0 && !d->ainv) return arg_fail("null inverse buffer for single-electron moves");
    if (std::max(c->s.np[0], c->s.ntypes > 1 ? c->s.np[1] : 0) > QMC_MAX_ORB)
      return arg_fail("single-electron moves support at most 64 particles per spin", QMC_ERR_LIMIT);
  } else if (w->nw > 0 && !w->props) {
    return arg_fail("null walker buffer: moves with backflow keep ltf in the walkers' properties");
  } else if (!c->use_gj) {
    return arg_fail("moves with backflow need the matrix-core determinant path (QMC_NO_GJ is set)");
  }
  return QMC_OK;
}

// With backflow every quasi-coordinate depends on every electron, so one
// electron's move changes every column of both orbital matrices and no
// low-rank update applies: each move takes the determinants of the proposed
// configuration anew (the pivots: no F, drift, Laplacian or potential) and is
// accepted with probability |psi'/psi|^2 = exp(-2 (ltf' - ltf)).  What is a
// sum over pairs changes by the pairs of the moved electron alone: the
// quasi-coordinates q_p = x_p + sum_b eta(r_pb) (x_p - x_b), the three-body
// vectors G_p and the Jastrow factor are formed at the start of a call
// (k_semf_init) and then follow the moves.  The pair terms are those of the
// evaluation in the call's precision (FP32 u2 and u3 tables in mixed
// precision); their sums are FP64.
//
// So a move is two launches: k_semf_step takes the decision on the move before
// and proposes the next, one block per walker with thread p taking partner p,
// and the determinant kernel follows.  All pairs evaluated for each proposal,
// with a copy of the walker, the evaluation's sum and the decision in kernels
// of their own, made 41 us per move for 512 walkers of N = 58 (now 20).
//
// Per walker: the current q in qc, G in gc; the proposal's in the evaluation's
// workspace, q where the determinants read it, G in the drift's place, and in
// the scalars' place:
enum { SF_U = 0, SF_UNEW = 1, SF_X = 2, SF_Y = 3, SF_UA = 4 };

template <bool MIX>
__device__ __forceinline__ double semf_spline(const DevSys& s, TabRef t, const PairGeo& p) {
  if (MIX) {
    const float4 c = tab_row(s.tab32, t, p.ind);
    const float rm = (float)(p.rem * s.drti);
    return (double)fmaf(rm, fmaf(rm, fmaf(rm, c.w, c.z), c.y), c.x);
  }
  const double4 c = tab_row(s.tab, t, p.ind);
  const double rm = p.rem * s.drti;
  return fma(rm, fma(rm, fma(rm, c.w, c.z), c.y), c.x);
}

// The terms of the pair (a, b) at separation p (u = x_a - x_b): u2 + (xi r)^2,
// xi u and eta u.
struct SemfPair {
  double u, gx, gy, qx, qy;
};
template <bool MIX>
__device__ __forceinline__ SemfPair semf_pair(const DevSys& s, TabRef t2, TabRef t3, TabRef tb, const PairGeo& p) {
  SemfPair o{0.0, 0.0, 0.0, 0.0, 0.0};
  if (t2.row0 >= 0) o.u = semf_spline<MIX>(s, t2, p);
  if (t3.row0 >= 0) {
    const double f = semf_spline<MIX>(s, t3, p), fr = f * p.r;
    o.u += fr * fr;
    o.gx = f * p.ux;
    o.gy = f * p.uy;
  }
  if (tb.row0 >= 0) {
    const double f = semf_spline<false>(s, tb, p);
    o.qx = f * p.ux;
    o.qy = f * p.uy;
  }
  return o;
}

// Sums over a block of up to two wavefronts of five values, on every thread.
__device__ __forceinline__ void semf_sum(double (&v)[5], double (*red)[5], int tid) {
#pragma unroll
  for (int q = 0; q < 5; q++) v[q] = wave_sum(v[q]);
  if ((tid & 63) == 0) {
#pragma unroll
    for (int q = 0; q < 5; q++) red[tid >> 6][q] = v[q];
  }
  block_sync();
  if (blockDim.x > 64) {
#pragma unroll
    for (int q = 0; q < 5; q++) v[q] = red[0][q] + red[1][q];
  }
}

// q, G and U of the walker's configuration.  One block per walker, eight lanes
// per particle, each summing over every eighth partner.
template <bool MIX>
__global__ __launch_bounds__(8 * QMC_MAX_PARTICLES) void k_semf_init(DevSys s, WsLayout L, double* __restrict__ ws,
                                                                     const double* __restrict__ x,
                                                                     double* __restrict__ qc,
                                                                     double* __restrict__ gc) {
  __shared__ __attribute__((aligned(16))) double xs[2 * QMC_MAX_PARTICLES];
  __shared__ double red[8 * QMC_MAX_PARTICLES / 64];
  const int w = blockIdx.x, tid = threadIdx.x, N = s.nptot;
  const int64_t at = (int64_t)w * 2 * N;
  for (int k = tid; k < 2 * N; k += blockDim.x) xs[k] = x[at + k];
  block_sync();
  const int a = tid >> 3;
  const bool li = a < N;
  double2 xp = make_double2(0.0, 0.0);
  double v[5] = {0.0, 0.0, 0.0, 0.0, 0.0};  // U, G, q
  if (li) {
    const int ti = ptype(s, a);
    xp = ld2(xs, a);
    for (int b = tid & 7; b < N; b += 8) {
      if (b == a) continue;
      const int tp = tpair(ti, ptype(s, b));
      const double2 xb = ld2(xs, b);
      const SemfPair t = semf_pair<MIX>(s, tabref<TK_U2>(s, tp), tabref<TK_U3>(s, tp), tabref<TK_B>(s, tp),
                                        pair_geo(s, xp.x, xp.y, xb.x, xb.y));
      v[0] += t.u;
      v[1] -= t.gx;
      v[2] -= t.gy;
      v[3] += t.qx;
      v[4] += t.qy;
    }
  }
#pragma unroll
  for (int q = 0; q < 5; q++) {
    v[q] += dpp_f64<0xB1>(v[q]);
    v[q] += dpp_f64<0x4E>(v[q]);
    v[q] += dpp_f64<0x141>(v[q]);  // the quads of a group of eight, mirrored
  }
  double u = 0.0;
  if (li && (tid & 7) == 0) {
    *reinterpret_cast<double2*>(qc + at + 2 * a) = make_double2(xp.x + v[3], xp.y + v[4]);
    *reinterpret_cast<double2*>(gc + at + 2 * a) = make_double2(v[1], v[2]);
    u = 0.5 * (v[0] - (v[1] * v[1] + v[2] * v[2]));
  }
  u = wave_sum(u);
  if ((tid & 63) == 0) red[tid >> 6] = u;
  block_sync();
  if (tid == 0) {
    double t = 0.0;
    for (int k = 0; k < (int)blockDim.x / 64; k++) t += red[k];
    ws[(int64_t)w * L.per_walker + L.off_sc + SF_U] = t;
  }
}

// Decision on the move of electron j - 1 (unless j is the call's first), then
// the proposal of electron j's (unless j is the end): the same three draws per
// move as the update path.
template <bool MIX>
__global__ __launch_bounds__(QMC_MAX_PARTICLES) void k_semf_step(
    DevSys s, WsLayout L, double* __restrict__ ws, int j, int j0, int j1, double sigma, int jltf,
    double* __restrict__ x, double* __restrict__ qc, double* __restrict__ gc, int64_t* __restrict__ rng,
    double* __restrict__ props, double* __restrict__ dlogpsi, double* __restrict__ nacc) {
  __shared__ double red[2][5];
  const int w = blockIdx.x, tid = threadIdx.x, N = s.nptot;
  const int64_t at = (int64_t)w * 2 * N;
  double* wsw = ws + (int64_t)w * L.per_walker;
  double* sc = wsw + L.off_sc;
  const bool li = tid < N;
  const int jp = j < j1 ? j : j - 1;  // the electron proposed (the last block only decides)
  uint64_t st = (uint64_t)rng[w];
  double2 xp = make_double2(0.0, 0.0), q = xp, g = xp, qn = xp, gn = xp;
  if (li) {
    xp = make_double2(x[at + 2 * tid], x[at + 2 * tid + 1]);
    q = *reinterpret_cast<const double2*>(qc + at + 2 * tid);
    g = *reinterpret_cast<const double2*>(gc + at + 2 * tid);
    qn = make_double2(wsw[L.off_q + 2 * tid], wsw[L.off_q + 2 * tid + 1]);
    gn = make_double2(wsw[L.off_gj + 2 * tid], wsw[L.off_gj + 2 * tid + 1]);
  }
  const double2 xj = make_double2(x[at + 2 * jp], x[at + 2 * jp + 1]);
  double U = sc[SF_U];
  if (j > j0) {
    const double Un = sc[SF_UNEW], ua = sc[SF_UA], xn = sc[SF_X], yn = sc[SF_Y];
    double* pl = props + (int64_t)w * s.n_props + jltf;
    const double lo = *pl, dl = dlogpsi[w], na = nacc[w];
    double ln = Un;
    bool sing = false;  // a singular proposal has psi' = 0
#pragma unroll
    for (int sp = 0; sp < 2; sp++) {
      if (sp >= s.ntypes || s.np[sp] == 0) continue;
      const double* dsc = wsw + L.off_det[sp];
      ln -= dsc[DS_LOGDET];
      sing = sing || dsc[DS_SING] != 0.0;
    }
    const bool acc = !sing && ua < exp(-2.0 * (ln - lo));
    block_sync();  // both wavefronts have read what is written below
    if (acc) {
      U = Un;
      q = qn;
      g = gn;
      if (tid == j - 1) {
        xp = make_double2(xn, yn);
        x[at + 2 * tid] = xn;
        x[at + 2 * tid + 1] = yn;
      }
      if (li) {
        *reinterpret_cast<double2*>(qc + at + 2 * tid) = q;
        *reinterpret_cast<double2*>(gc + at + 2 * tid) = g;
      }
      if (tid == 0) {
        sc[SF_U] = U;
        *pl = ln;
        dlogpsi[w] = dl + (lo - ln);
        nacc[w] = na + 1.0;
      }
    }
  }
  if (j >= j1) return;
  const double u1 = rannyu(st), u2 = rannyu(st), ua = rannyu(st);
  double sv, cv;
  qsincos(6.283185307179586 * u2, &sv, &cv);
  const double rad = sigma * sqrt(-2.0 * log(u1));
  const double xn = xj.x + rad * cv, yn = xj.y + rad * sv;
  // partner tid's terms at the new and the old position of j
  double v[5] = {0.0, 0.0, 0.0, 0.0, 0.0};  // dU, then G and q of j at its new position
  double2 dg = make_double2(0.0, 0.0), dq = dg;
  if (li && tid != j) {
    const int tp = tpair(ptype(s, j), ptype(s, tid));
    const TabRef t2 = tabref<TK_U2>(s, tp), t3 = tabref<TK_U3>(s, tp), tb = tabref<TK_B>(s, tp);
    const SemfPair a = semf_pair<MIX>(s, t2, t3, tb, pair_geo(s, xn, yn, xp.x, xp.y));
    const SemfPair o = semf_pair<MIX>(s, t2, t3, tb, pair_geo(s, xj.x, xj.y, xp.x, xp.y));
    dg = make_double2(a.gx - o.gx, a.gy - o.gy);
    dq = make_double2(o.qx - a.qx, o.qy - a.qy);
    // -1/2 (|G + dG|^2 - |G|^2) = -dG.G - 1/2 |dG|^2
    v[0] = (a.u - o.u) - (g.x * dg.x + g.y * dg.y) - 0.5 * (dg.x * dg.x + dg.y * dg.y);
    v[1] = -a.gx;
    v[2] = -a.gy;
    v[3] = a.qx;
    v[4] = a.qy;
  } else if (tid == j) {
    v[0] = 0.5 * (g.x * g.x + g.y * g.y);
  }
  semf_sum(v, red, tid);
  if (li) {
    const bool me = tid == j;
    wsw[L.off_q + 2 * tid] = me ? xn + v[3] : q.x + dq.x;
    wsw[L.off_q + 2 * tid + 1] = me ? yn + v[4] : q.y + dq.y;
    wsw[L.off_gj + 2 * tid] = me ? v[1] : g.x + dg.x;
    wsw[L.off_gj + 2 * tid + 1] = me ? v[2] : g.y + dg.y;
  }
  if (tid == 0) {
    sc[SF_UNEW] = U + v[0] - 0.5 * (v[1] * v[1] + v[2] * v[2]);
    sc[SF_X] = xn;
    sc[SF_Y] = yn;
    sc[SF_UA] = ua;
    rng[w] = (int64_t)st;
  }
}

static int sem_moves_full(qmc_ctx* c, const qmc_walkers* w, const qmc_sem_state* d, int j0, int j1, double sigma,
                          int precision, hipStream_t st) {
  if (j0 >= j1) return QMC_OK;
  const int nw = w->nw;
  const bool mix = precision == QMC_PREC_MIXED;
  int rc = ensure_vmc_scratch(c, nw);
  if (rc) return rc;
  rc = ensure_ws(c, nw);
  if (rc) return rc;
  const dim3 block(c->s.nptot <= 64 ? 64 : QMC_MAX_PARTICLES);
  hipLaunchKernelGGL(mix ? k_semf_init<true> : k_semf_init<false>, dim3(nw),
                     dim3((8 * c->s.nptot + 63) / 64 * 64), 0, st, c->s, c->L, c->d_ws, w->x, c->d_gn, c->d_xn);
  for (int j = j0; j <= j1; j++) {
    hipLaunchKernelGGL(mix ? k_semf_step<true> : k_semf_step<false>, dim3(nw), block, 0, st, c->s, c->L, c->d_ws, j,
                       j0, j1, sigma, c->info.jltf - 1, w->x, c->d_gn, c->d_xn, w->rng, w->props, d->dlogpsi,
                       d->nacc);
    if (j == j1) break;
    rc = launch_logdet(c, nw, st);
    if (rc) return rc;
  }
  HIPCHK(hipGetLastError());
  return QMC_OK;
}

// Kind of row and wavefronts per walker of a job's moves: real rows in FP64
// where the orbitals are real (one wavefront up to 32 rows per spin, two above),
// else complex ones with the context's threads per row for each class (16 rows:
// 4 threads; 32 and 64 rows: 2 or 4), as many wavefronts as the larger spin
// needs.
static void sem_shape(const qmc_ctx* c, int precision, int& kind, int& waves) {
  kind = precision == QMC_PREC_MIXED ? 2 : c->s.real_orb ? 0 : 1;
  waves = 1;
  for (int sp = 0; sp < c->s.ntypes; sp++) {
    const int m = c->s.np[sp];
    if (m == 0) continue;
    if (kind == 0) {
      waves = std::max(waves, std::max(m, 2 * c->s.nslot[sp]) <= 32 ? 1 : 2);
    } else {
      const int cls = sem_class(m);
      waves = std::max(waves, (16 << cls) * (cls == 0 ? 4 : c->sem_cg[precision == QMC_PREC_MIXED ? 1 : 0][cls]) / 64);
    }
  }
}

// Moves of jobs, each taking the spins of its range in order: one launch per
// kind of row and wavefronts per walker.  Jobs with the most electrons come
// first, so that the longest walkers start first.  A job's results do not
// depend on the others: its kind, wavefronts and tiles are its context's (the
// three-body variant also serves jobs without u3, whose u3 terms are skipped
// and add nothing).
static int sem_moves_jobs(const qmc_sem_job* jobs, int njobs, int precision, hipStream_t st) {
  std::vector<const qmc_sem_job*> order;
  for (int k = 0; k < njobs; k++)
    if (jobs[k].w->nw > 0 && jobs[k].j0 < jobs[k].j1) order.push_back(jobs + k);
  std::stable_sort(order.begin(), order.end(), [](const qmc_sem_job* a, const qmc_sem_job* b) {
    return a->ctx->s.nptot > b->ctx->s.nptot;
  });
  // real-row jobs of one wavefront per walker join a launch of two
  bool wide = false;
  for (const qmc_sem_job* j : order) {
    int k, w;
    sem_shape(j->ctx, precision, k, w);
    wide = wide || (k == 0 && w == 2);
  }
  for (int kind = 0; kind < 3; kind++)
    for (int waves = 4; waves >= 1; waves >>= 1) {
      SemJobs jb{};
      int nblocks = 0, nmax = 0;
      bool u3 = false;
      for (const qmc_sem_job* j : order) {
        qmc_ctx* c = j->ctx;
        int k, w;
        sem_shape(c, precision, k, w);
        const bool narrow = k == 0 && w == 1 && wide;
        if (narrow) w = 2;
        if (k != kind || w != waves) continue;
        const int rc = upload_sys(c, st);
        if (rc) return rc;
        SemJob& e = jb.job[jb.njobs++];
        e.sys = c->d_sys;
        e.x = j->w->x;
        e.rng = j->w->rng;
        e.ainv = j->d->ainv;
        e.dlogpsi = j->d->dlogpsi;
        e.nacc = j->d->nacc;
        e.sigma = j->sigma;
        e.w0 = nblocks;
        e.nw = j->w->nw;
        e.j0 = j->j0;
        e.j1 = j->j1;
        e.mm = sem_mm(c);
        for (int t = 0; t < 3; t++) e.tile[t] = c->sem_cg[precision == QMC_PREC_MIXED ? 1 : 0][t];
        e.narrow = narrow;
        nblocks += narrow ? (e.nw + 1) / 2 : e.nw;
        u3 = u3 || c->s.has_u3;
        nmax = std::max(nmax, narrow ? 2 * c->s.nptot : c->s.nptot);
      }
      if (jb.njobs == 0) continue;
      const int rc = launch_sem_moves(jb, nblocks, kind, waves, u3, nmax, st);
      if (rc) return rc;
    }
  return QMC_OK;
}

// The orbitals that a call's kernels read are there.
static int sem_orbitals(const qmc_ctx* c) {
  for (int sp = 0; sp < c->s.ntypes; sp++)
    if (c->s.np[sp] > c->s.ng) return arg_fail("fewer g-vectors than particles of a spin", QMC_ERR_NOTWIST);
  return QMC_OK;
}

extern "C" int qmc_sem_refresh(qmc_ctx* c, const qmc_walkers* w, const qmc_sem_state* d, int precision,
                               void* stream) {
  int rc = sem_check(c, w, d, precision);
  if (rc) return rc;
  if (w->nw == 0 || !c->b_zero) return QMC_OK;  // backflow: no inverse is carried
  rc = sem_orbitals(c);
  if (rc) return rc;
  HIPCHK(hipSetDevice(c->device));
  const int mm = sem_mm(c);
  if (c->s.real_orb && precision == QMC_PREC_FP64) {
    launch_gjr_inverse(c->s, w->nw, w->x, d->ainv, mm, (hipStream_t)stream);
    HIPCHK(hipGetLastError());
    return QMC_OK;
  }
  for (int sp = 0; sp < c->s.ntypes; sp++) {
    if (c->s.np[sp] == 0) continue;
    rc = precision == QMC_PREC_MIXED ? sem_inverse_spin<float2>(c, w, d, sp, mm, (hipStream_t)stream)
                                     : sem_inverse_spin<double2>(c, w, d, sp, mm, (hipStream_t)stream);
    if (rc) return rc;
  }
  return QMC_OK;
}

extern "C" int qmc_sem_moves(qmc_ctx* c, const qmc_walkers* w, const qmc_sem_state* d, int j0, int j1,
                             double sigma, int precision, void* stream) {
  int rc = sem_check(c, w, d, precision);
  if (rc) return rc;
  if (j0 < 0 || j1 > c->s.nptot || j0 > j1) return arg_fail("electron range out of bounds");
  if (!(sigma > 0.0)) return arg_fail("sigma must be positive");
  if (w->nw == 0 || j0 == j1) return QMC_OK;
  rc = sem_orbitals(c);
  if (rc) return rc;
  HIPCHK(hipSetDevice(c->device));
  if (!c->b_zero) return sem_moves_full(c, w, d, j0, j1, sigma, precision, (hipStream_t)stream);
  const qmc_sem_job one = {c, w, d, j0, j1, sigma};
  return sem_moves_jobs(&one, 1, precision, (hipStream_t)stream);
}

extern "C" int qmc_sem_moves_packed(const qmc_sem_job* jobs, int njobs, int precision, void* stream) {
  if (!jobs || njobs < 0 || njobs > SEM_MAX_PACK) return arg_fail("between 0 and 16 jobs per packed call");
  if (njobs == 0) return QMC_OK;
  hipStream_t st = (hipStream_t)stream;
  for (int k = 0; k < njobs; k++) {
    const qmc_sem_job& jb = jobs[k];
    int rc = sem_check(jb.ctx, jb.w, jb.d, precision);
    if (rc) return rc;
    if (!jb.ctx->b_zero) return arg_fail("jobs with backflow cannot be packed (each move is a full evaluation)");
    if (jb.ctx->device != jobs[0].ctx->device) return arg_fail("packed jobs must share one device");
    if (jb.j0 < 0 || jb.j1 > jb.ctx->s.nptot || jb.j0 > jb.j1) return arg_fail("electron range out of bounds");
    if (!(jb.sigma > 0.0)) return arg_fail("sigma must be positive");
    rc = jb.w->nw > 0 && jb.j0 < jb.j1 ? sem_orbitals(jb.ctx) : QMC_OK;
    if (rc) return rc;
  }
  HIPCHK(hipSetDevice(jobs[0].ctx->device));
  return sem_moves_jobs(jobs, njobs, precision, st);
}
