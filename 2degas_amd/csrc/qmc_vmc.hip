// qmc_vmc.hip -- batched VMC step on the device: drift-diffusion proposal,
// evaluation, Metropolis test and block accumulation for every walker.
//
// Each walker owns a stream of the reference's 48-bit LCG (rannyu,
// reptation.f:5247-5291), so a batch of nw walkers draws exactly what nw MPI
// ranks of the reference draw (rank r is seeded with seed(4) = 2*(seed(4)+r)+1,
// reptation.f:37-39).
#include "qmc_internal.h"

#include <cstring>

// move, proposal half (reptation.f:4630-4646): for every moving type,
// particle and dimension chi = cos(pi u1) sqrt(-2 var log u2),
// x_new = chi - var g_old + x_old, w = -sum chi^2 / var.
// One block per walker, a thread per coordinate.  The reference draws two
// uniforms per moved coordinate in coordinate order, so the coordinate with
// ordinal o among the moved ones takes draws 2o+1 and 2o+2 of the walker's
// stream: each thread jumps there with a^(2o+1).  Bound by latency (a cosine, a
// logarithm and the sum): with a wavefront per walker that walked over its
// coordinates and one lane adding the chi^2 4.9 us at N = 26 and 7.9 us at
// N = 74 (256 walkers), now 3.6 and 4.7.
__global__ __launch_bounds__(QMC_BLOCK) void k_vmc_propose(
    DevSys s, const double* __restrict__ x_old, const double* __restrict__ g_old,
    double* __restrict__ x_new, int64_t* __restrict__ rng, double* __restrict__ wold,
    double var0, double var1, int bm_order) {
  __shared__ double red[2][QMC_BLOCK / 64];
  const int e = threadIdx.x, w = blockIdx.x;
  const int n2 = 2 * s.nptot;
  const uint64_t st0 = (uint64_t)rng[w];
  const double pi = 3.141592653589793;
  const uint64_t msk = (1ULL << 48) - 1ULL, a = 34522712143931ULL;
  const bool two = s.ntypes > 1;
  const bool mov0 = s.hbs2m[0] != 0.0, mov1 = two && s.hbs2m[1] != 0.0;
  const int m0 = mov0 ? 2 * s.np[0] : 0;  // moved coordinates of type 0
  const int nmov = m0 + (mov1 ? 2 * s.np[1] : 0);
  double c2 = 0.0;
  const int t = two && e >= 2 * s.ipf[1] ? 1 : 0;
  if (e < n2) {
    const double xo = x_old[(int64_t)w * n2 + e], go = g_old[(int64_t)w * n2 + e];
    double xe = xo;
    if (t ? mov1 : mov0) {
      const int o = t ? m0 + e - 2 * s.ipf[1] : e - 2 * s.ipf[0];
      const double var = t ? var1 : var0;
      const uint64_t x1 = (lcg_pow10(2 * o + 1) * st0) & msk, x2 = (a * x1) & msk;
      const double u1 = (double)x1 * 0x1p-48, u2 = (double)x2 * 0x1p-48;
      const double ua = bm_order == 0 ? u1 : u2, ub = bm_order == 0 ? u2 : u1;
      const double chi = cos(pi * ua) * sqrt(-2.0 * var * log(ub));
      c2 = chi * chi;
      xe = chi + (-var * go) + xo;
    }
    x_new[(int64_t)w * n2 + e] = xe;
  }
  const double s0 = wave_sum(t ? 0.0 : c2), s1 = wave_sum(t ? c2 : 0.0);
  if ((e & 63) == 0) {
    red[0][e >> 6] = s0;
    red[1][e >> 6] = s1;
  }
  block_sync();
  if (e == 0) {
    double w0 = 0.0, w1 = 0.0;
    for (int v = 0; v < QMC_BLOCK / 64; v++) {
      w0 -= red[0][v];
      w1 -= red[1][v];
    }
    double wo = 0.0;
    if (mov0) wo = wo + w0 * (1.0 / var0);
    if (mov1) wo = wo + w1 * (1.0 / var1);
    wold[w] = wo;
    rng[w] = (int64_t)((lcg_pow10(2 * nmov) * st0) & msk);
  }
}

// move, acceptance half (reptation.f:4648-4678) + metropolis_test
// (reptation.f:2622-2659) + averages(2) (reptation.f:4300-4305), and with DMC
// the walker's weight: the local energy metropolis_test leaves
// (reptation.f:2630-2632, 2652-2653: the mean of the new and old energies
// when accepted, the old one otherwise), the factor
// peso = exp(-npnorm (elocal - etrial) delta) bounded at mmult
// (reptation.f:897-903), wate *= peso, and averages(2) with weight wate
// (reptation.f:4300-4305: blk += p_old wate, blk_norm += wate).
//
// One block per walker.  The kernel is bound by latency: a few dependent
// loads, the exponential, and the pass over the properties.  So every
// wavefront forms the decision for itself from the same loads in the same
// order, the properties, the block sums and the new configuration are fetched
// before it, and one barrier stands between the last read and the first
// write.  A wavefront per walker, walking over the properties 64 at a time
// after the decision, took 11.0 us at N = 26 and 12.3 us at N = 74 (256 walkers;
// now 4.8 and 4.6).  For 4096 walkers of N = 122 in DMC the bytes count, some
// 0.4 GB of properties and sums: 86 us, where the weight's own kernel and pass
// took 91 us after the acceptance.
constexpr int VA_SLOTS = 4;  // properties per thread fetched ahead
template <bool DMC>
__global__ __launch_bounds__(QMC_BLOCK) void k_vmc_accept(
    DevSys s, double var0, double var1, double mage, double* __restrict__ x_old,
    double* __restrict__ g_old, double* __restrict__ h_old, double* __restrict__ p_old,
    double* __restrict__ age, const double* __restrict__ x_new, const double* __restrict__ g_new,
    const double* __restrict__ h_new, const double* __restrict__ p_new, int64_t* __restrict__ rng,
    const double* __restrict__ wold, const int32_t* __restrict__ status,
    int32_t* __restrict__ sticky, double* __restrict__ blk, double* __restrict__ trace_p,
    double* __restrict__ trace_age, int jacc, int jltf, DmcWeight dm) {
  const int w = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const int N = s.nptot, NP = s.n_props;
  double* xo = x_old + (int64_t)w * 2 * N;
  const double* xn = x_new + (int64_t)w * 2 * N;
  const double* gn = g_new + (int64_t)w * 2 * N;
  double* po = p_old + (int64_t)w * NP;
  const double* pn = p_new + (int64_t)w * NP;
  double* b = blk ? blk + (int64_t)w * NP : nullptr;
  double vn[VA_SLOTS], vo[VA_SLOTS], vb[VA_SLOTS];
#pragma unroll
  for (int u = 0; u < VA_SLOTS; u++) {
    const int k = tid + u * QMC_BLOCK;
    vn[u] = vo[u] = vb[u] = 0.0;
    if (k < NP) {
      vn[u] = pn[k];
      vo[u] = po[k];
      if (b) vb[u] = b[k];
    }
  }
  double xk = 0.0, gk = 0.0, hk = 0.0;
  if (tid < 2 * N) {
    xk = xn[tid];
    gk = gn[tid];
  }
  if (tid < 2) hk = h_new[(int64_t)w * 2 + tid];
  const double age0 = age[w], ltf0 = po[jltf], ltf1 = pn[jltf], wo = wold[w];
  uint64_t rs = (uint64_t)rng[w];
  double wt[2] = {0.0, 0.0};
  for (int ip = lane; ip < N; ip += 64) {
    const int t = ptype(s, ip);
    const double var = t == 0 ? var0 : var1;
    for (int d = 0; d < 2; d++) {
      const double drift = -var * gn[2 * ip + d];
      const double chi = xo[2 * ip + d] - xn[2 * ip + d] - drift;
      if (t == 0) wt[0] = wt[0] - chi * chi;
      else wt[1] = wt[1] - chi * chi;
    }
  }
  wt[0] = wave_sum(wt[0]);
  wt[1] = wave_sum(wt[1]);
  double p;
  if (age0 == mage) {
    p = 1.0;
  } else {
    double wnew = 0.0;
    if (s.hbs2m[0] != 0.0) wnew = wnew + wt[0] * (1.0 / var0);
    if (s.ntypes > 1 && s.hbs2m[1] != 0.0) wnew = wnew + wt[1] * (1.0 / var1);
    p = (ltf0 - ltf1) * 2.0 + 0.5 * (wnew - wo);
    p = fmin(0.0, fmax(-50.0, p));
    p = exp(p);
  }
  double u = 1.0;
  if (p < 1.0) u = rannyu(rs);
  const bool acc = p >= u;
  const double a = acc ? 0.0 : age0 + 1.0;
  double wgt = 1.0, wsum0 = 0.0;
  bool bounded = false;
  if (DMC) {
    const double eold = po[dm.jetot], enew = acc ? pn[dm.jetot] : eold;
    const double elocal = a == 0.0 ? 0.5 * (enew + eold) : eold;
    double peso = exp(-(double)s.npnorm * (elocal - dm.etrial) * dm.delta);
    bounded = peso > dm.mmult;
    if (bounded) peso = dm.mmult;
    wgt = dm.wate[w] * peso;
    wsum0 = dm.wsum[w];
  }
  block_sync();  // every wavefront has read what the stores below change
  // copy new into old where accepted, set p_old(jacc) = p and add p_old to
  // the block sums
#pragma unroll
  for (int q = 0; q < VA_SLOTS; q++) {
    const int k = tid + q * QMC_BLOCK;
    if (k < NP) {
      const double v = (k == jacc) ? p : (acc ? vn[q] : vo[q]);
      if (acc || k == jacc) po[k] = v;
      if (b) b[k] = DMC ? vb[q] + v * wgt : vb[q] + v;
    }
  }
  for (int k0 = VA_SLOTS * QMC_BLOCK + tid; k0 < NP; k0 += VA_SLOTS * QMC_BLOCK) {
    const double* ps = acc ? pn : po;
#pragma unroll
    for (int q = 0; q < VA_SLOTS; q++) {
      const int k = k0 + q * QMC_BLOCK;
      if (k < NP) {
        vn[q] = k == jacc ? p : ps[k];
        if (b) vb[q] = b[k];
      }
    }
#pragma unroll
    for (int q = 0; q < VA_SLOTS; q++) {
      const int k = k0 + q * QMC_BLOCK;
      if (k < NP) {
        if (acc || k == jacc) po[k] = vn[q];
        if (b) b[k] = DMC ? vb[q] + vn[q] * wgt : vb[q] + vn[q];
      }
    }
  }
  if (acc) {
    if (tid < 2 * N) {
      xo[tid] = xk;
      g_old[(int64_t)w * 2 * N + tid] = gk;
    }
    if (tid < 2) h_old[(int64_t)w * 2 + tid] = hk;
  }
  if (tid == 0) {
    rng[w] = (int64_t)rs;
    sticky[w] |= status[w];
    age[w] = a;
    if (trace_p) trace_p[w] = p;
    if (trace_age) trace_age[w] = a;
    if (DMC) {
      dm.wate[w] = wgt;
      dm.wsum[w] = wsum0 + wgt;
      if (bounded) atomicAdd(&dm.counts[0], 1);
      // move counts a forced move when the age reached mage (reptation.f:4650-4653)
      if (w == 0 && age0 == mage) atomicAdd(&dm.counts[3], 1);
    }
  }
}
static_assert(2 * QMC_MAX_PARTICLES <= QMC_BLOCK, "one coordinate per thread");

// read_conf's start: age 0 and p_old(jacc) = 1 after the evaluation.
__global__ void k_vmc_start(int nw, int np_, int jacc, double* __restrict__ props,
                            double* __restrict__ age, int32_t* __restrict__ sticky) {
  const int w = blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= nw) return;
  props[(int64_t)w * np_ + jacc] = 1.0;
  age[w] = 0.0;
  sticky[w] = 0;
}

void free_vmc(qmc_ctx* c) {
  free_vmc_graph(c);
  (void)hipFree(c->d_xn);
  (void)hipFree(c->d_gn);
  (void)hipFree(c->d_hn);
  (void)hipFree(c->d_pn);
  (void)hipFree(c->d_wold);
  (void)hipFree(c->d_stn);
  (void)hipFree(c->d_sticky);
  c->d_xn = c->d_gn = c->d_hn = c->d_pn = c->d_wold = nullptr;
  c->d_stn = c->d_sticky = nullptr;
  c->vmc_nw = 0;
}

// Proposal and status buffers for nw walkers (or reptiles).
int ensure_vmc_scratch(qmc_ctx* c, int nw) {
  if (nw <= c->vmc_nw) return QMC_OK;
  free_vmc(c);
  const size_t N = c->s.nptot, NP = c->info.n_props;
  HIPCHK(hipMalloc(&c->d_xn, sizeof(double) * 2 * N * nw));
  HIPCHK(hipMalloc(&c->d_gn, sizeof(double) * 2 * N * nw));
  HIPCHK(hipMalloc(&c->d_hn, sizeof(double) * 2 * nw));
  HIPCHK(hipMalloc(&c->d_pn, sizeof(double) * NP * nw));
  HIPCHK(hipMalloc(&c->d_wold, sizeof(double) * nw));
  HIPCHK(hipMalloc(&c->d_stn, sizeof(int32_t) * nw));
  HIPCHK(hipMalloc(&c->d_sticky, sizeof(int32_t) * nw));
  HIPCHK(hipMemset(c->d_pn, 0, sizeof(double) * NP * nw));
  // a sweep may run without a start call (state loaded by the caller)
  HIPCHK(hipMemset(c->d_sticky, 0, sizeof(int32_t) * nw));
  c->vmc_nw = nw;
  return QMC_OK;
}

static int check_walkers(qmc_ctx* c, const qmc_walkers* w) {
  if (!c || !w || w->nw < 0) return arg_fail("bad walker set");
  if (w->nw > 0 && (!w->x || !w->g || !w->h || !w->props || !w->grad2_ph || !w->age || !w->rng))
    return arg_fail("null walker buffer");
  return QMC_OK;
}

extern "C" int qmc_vmc_start(qmc_ctx* c, const qmc_walkers* w, void* stream) {
  int rc = check_walkers(c, w);
  if (rc) return rc;
  if (w->nw == 0) return QMC_OK;
  HIPCHK(hipSetDevice(c->device));
  hipStream_t st = (hipStream_t)stream;
  rc = ensure_vmc_scratch(c, w->nw);
  if (rc) return rc;
  rc = launch_eval(c, w->nw, w->x, w->props, w->g, w->h, w->grad2_ph, c->d_stn, st, c->delta);
  if (rc) return rc;
  hipLaunchKernelGGL(k_vmc_start, dim3((w->nw + 255) / 256), dim3(256), 0, st, w->nw,
                     c->info.n_props, c->info.jacc - 1, w->props, w->age, c->d_sticky);
  HIPCHK(hipGetLastError());
  return QMC_OK;
}

// One VMC step for every walker: proposal, evaluation, acceptance.
int vmc_step(qmc_ctx* c, const qmc_walkers* w, hipStream_t st, double delta, double var0, double var1,
             double mage, int bm_order, double* tp, double* ta, const DmcWeight* dm) {
  const DevSys& s = c->s;
  const int nw = w->nw;
  hipLaunchKernelGGL(k_vmc_propose, dim3(nw), dim3(QMC_BLOCK), 0, st, s, w->x, w->g, c->d_xn,
                     w->rng, c->d_wold, var0, var1, bm_order);
  // the fixed-phase scratch is shared by proposals, as the COMMON is
  int rc = launch_eval(c, nw, c->d_xn, c->d_pn, c->d_gn, c->d_hn, w->grad2_ph, c->d_stn, st, delta);
  if (rc) return rc;
  hipLaunchKernelGGL(dm ? k_vmc_accept<true> : k_vmc_accept<false>, dim3(nw), dim3(QMC_BLOCK), 0, st, s,
                     var0, var1, mage, w->x, w->g, w->h, w->props, w->age, c->d_xn, c->d_gn,
                     c->d_hn, c->d_pn, w->rng, c->d_wold, c->d_stn, c->d_sticky, w->blk, tp, ta,
                     c->info.jacc - 1, c->info.jltf - 1, dm ? *dm : DmcWeight{});
  return QMC_OK;
}

void free_vmc_graph(qmc_ctx* c) {
  if (c->vmc_exec) (void)hipGraphExecDestroy(c->vmc_exec);
  c->vmc_exec = nullptr;
  c->vmc_key.clear();
  if (c->rmc_exec) (void)hipGraphExecDestroy(c->rmc_exec);
  c->rmc_exec = nullptr;
  c->rmc_key.clear();
}

extern "C" int qmc_vmc_sweep(qmc_ctx* c, const qmc_walkers* w, int nsteps, double delta,
                             double mage, int bm_order, double* trace_p, double* trace_age,
                             void* stream) {
  int rc = check_walkers(c, w);
  if (rc) return rc;
  if (w->nw == 0 || nsteps <= 0) return QMC_OK;
  if (!(delta > 0.0)) return arg_fail("delta must be positive");
  HIPCHK(hipSetDevice(c->device));
  hipStream_t st = (hipStream_t)stream;
  rc = ensure_vmc_scratch(c, w->nw);
  if (rc) return rc;
  rc = ensure_ws(c, w->nw);
  if (rc) return rc;
  const DevSys& s = c->s;
  // the vmc record sets the COMMON delta before sigma (reptation.f:740-746)
  c->delta = delta;
  // sigma (reptation.f:855-870)
  const double var0 = 2.0 * s.hbs2m[0] * delta;
  const double var1 = s.ntypes > 1 ? 2.0 * s.hbs2m[1] * delta : 1.0;
  const int nw = w->nw;
  const bool graph = c->use_graph && !trace_p && !trace_age && !c->timing && nsteps > 1;
  if (!graph) {
    for (int k = 0; k < nsteps; k++) {
      rc = vmc_step(c, w, st, delta, var0, var1, mage, bm_order,
                    trace_p ? trace_p + (int64_t)k * nw : nullptr,
                    trace_age ? trace_age + (int64_t)k * nw : nullptr, nullptr);
      if (rc) return rc;
    }
    HIPCHK(hipGetLastError());
    return QMC_OK;
  }
  // The step as a captured graph, replayed nsteps times: rebuilt whenever
  // anything its kernels were given changes (buffers, step parameters, the
  // g-vectors).  Captured on the context's own stream, launched on st.
  double dk[4] = {var0, var1, mage, delta};
  std::vector<uint64_t> key = {(uint64_t)nw, (uint64_t)(uintptr_t)w->x, (uint64_t)(uintptr_t)w->g,
                               (uint64_t)(uintptr_t)w->h, (uint64_t)(uintptr_t)w->props,
                               (uint64_t)(uintptr_t)w->age, (uint64_t)(uintptr_t)w->rng,
                               (uint64_t)(uintptr_t)w->blk, (uint64_t)(uintptr_t)w->grad2_ph,
                               (uint64_t)(uintptr_t)c->d_xn, (uint64_t)(uintptr_t)c->d_ws,
                               (uint64_t)(uintptr_t)c->d_F, (uint64_t)(uintptr_t)c->d_A,
                               (uint64_t)(uintptr_t)s.gvec, (uint64_t)s.ng, (uint64_t)bm_order};
  for (double v : dk) {
    uint64_t b;
    memcpy(&b, &v, sizeof b);
    key.push_back(b);
  }
  if (!c->vmc_exec || key != c->vmc_key) {
    free_vmc_graph(c);
    HIPCHK(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
    rc = vmc_step(c, w, c->stream, delta, var0, var1, mage, bm_order, nullptr, nullptr, nullptr);
    hipGraph_t g = nullptr;
    const hipError_t e = hipStreamEndCapture(c->stream, &g);
    if (rc) {
      if (g) (void)hipGraphDestroy(g);
      return rc;
    }
    if (e != hipSuccess) return hip_fail(e, "hipStreamEndCapture");
    const hipError_t e2 = hipGraphInstantiate(&c->vmc_exec, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (e2 != hipSuccess) {
      c->vmc_exec = nullptr;
      return hip_fail(e2, "hipGraphInstantiate");
    }
    c->vmc_key = key;
  }
  for (int k = 0; k < nsteps; k++) HIPCHK(hipGraphLaunch(c->vmc_exec, st));
  return QMC_OK;
}

extern "C" int qmc_vmc_status(qmc_ctx* c, int nw, int32_t* sticky_host) {
  if (!c || nw < 0 || nw > c->vmc_nw || (nw > 0 && !sticky_host)) return arg_fail("bad status query");
  if (nw == 0) return QMC_OK;
  HIPCHK(hipSetDevice(c->device));
  HIPCHK(hipDeviceSynchronize());
  HIPCHK(hipMemcpy(sticky_host, c->d_sticky, sizeof(int32_t) * nw, hipMemcpyDeviceToHost));
  for (int k = 0; k < nw; k++)
    if (sticky_host[k] & 2) return arg_fail("slater_bckflw_orbitals: singular orbital matrix", QMC_ERR_SINGULAR);
  return QMC_OK;
}
