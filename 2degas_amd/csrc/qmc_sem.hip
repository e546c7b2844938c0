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
      __syncthreads();
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
      __syncthreads();
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
  __syncthreads();
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
// low-rank update applies: each move evaluates the proposed configuration's
// log|psi| (the pair kernel's Jastrow pass and quasi-coordinates, the
// determinants' pivots: no F, drift, Laplacian or potential), accepted with
// probability |psi'/psi|^2 = exp(-2 (ltf' - ltf)).  One wavefront per walker
// copies the walker with electron j displaced (the same three draws per move
// as the update path); after the evaluation one thread per walker takes the
// decision and, when accepted, moves the electron and keeps the new ltf in
// the walker's ltf slot.
__global__ __launch_bounds__(256) void k_semf_propose(DevSys s, int nw, int j, double sigma,
                                                      const double* __restrict__ x, double* __restrict__ xn,
                                                      int64_t* __restrict__ rng, double* __restrict__ ua) {
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int w = blockIdx.x * 4 + wv;
  if (w >= nw) return;
  const int N = s.nptot;
  const double* xw = x + (int64_t)w * 2 * N;
  double* xo = xn + (int64_t)w * 2 * N;
  for (int e = lane; e < 2 * N; e += 64)
    if (e != 2 * j && e != 2 * j + 1) xo[e] = xw[e];
  if (lane == 0) {
    uint64_t st = (uint64_t)rng[w];
    const double u1 = rannyu(st), u2 = rannyu(st), a = rannyu(st);
    double sv, cv;
    qsincos(6.283185307179586 * u2, &sv, &cv);
    const double rad = sigma * sqrt(-2.0 * log(u1));
    xo[2 * j] = xw[2 * j] + rad * cv;
    xo[2 * j + 1] = xw[2 * j + 1] + rad * sv;
    rng[w] = (int64_t)st;
    ua[w] = a;
  }
}

__global__ __launch_bounds__(256) void k_semf_accept(DevSys s, int nw, int j, int jltf, const double* __restrict__ xn,
                                                     const double* __restrict__ ltfn, const int32_t* __restrict__ stn,
                                                     const double* __restrict__ ua, double* __restrict__ x,
                                                     double* __restrict__ props, double* __restrict__ dlogpsi,
                                                     double* __restrict__ nacc) {
  const int w = blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= nw) return;
  const int N = s.nptot, NP = s.n_props;
  const double lo = props[(int64_t)w * NP + jltf], ln = ltfn[w];
  // a singular proposal (status bit 2) has psi' = 0
  if ((stn[w] & 2) != 0 || !(ua[w] < exp(-2.0 * (ln - lo)))) return;
  x[(int64_t)w * 2 * N + 2 * j] = xn[(int64_t)w * 2 * N + 2 * j];
  x[(int64_t)w * 2 * N + 2 * j + 1] = xn[(int64_t)w * 2 * N + 2 * j + 1];
  props[(int64_t)w * NP + jltf] = ln;
  dlogpsi[w] += lo - ln;
  nacc[w] += 1.0;
}

static int sem_moves_full(qmc_ctx* c, const qmc_walkers* w, const qmc_sem_state* d, int j0, int j1, double sigma,
                          int precision, hipStream_t st) {
  const int nw = w->nw;
  int rc = ensure_vmc_scratch(c, nw);
  if (rc) return rc;
  for (int j = j0; j < j1; j++) {
    hipLaunchKernelGGL(k_semf_propose, dim3((nw + 3) / 4), dim3(256), 0, st, c->s, nw, j, sigma, w->x, c->d_xn,
                       w->rng, c->d_wold);
    // the proposal's ltf in d_hn (nw doubles of the proposal buffers)
    rc = launch_value(c, nw, c->d_xn, c->d_hn, c->d_stn, c->d_pn, st, precision);
    if (rc) return rc;
    hipLaunchKernelGGL(k_semf_accept, dim3((nw + 255) / 256), dim3(256), 0, st, c->s, nw, j, c->info.jltf - 1,
                       c->d_xn, c->d_hn, c->d_stn, c->d_wold, w->x, w->props, d->dlogpsi, d->nacc);
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

extern "C" int qmc_sem_refresh(qmc_ctx* c, const qmc_walkers* w, const qmc_sem_state* d, int precision,
                               void* stream) {
  int rc = sem_check(c, w, d, precision);
  if (rc) return rc;
  if (w->nw == 0 || !c->b_zero) return QMC_OK;  // backflow: no inverse is carried
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
  }
  HIPCHK(hipSetDevice(jobs[0].ctx->device));
  return sem_moves_jobs(jobs, njobs, precision, st);
}
