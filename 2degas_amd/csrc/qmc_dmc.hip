// qmc_dmc.hip -- diffusion Monte Carlo with fixed-population branching on
// the device: the reference's dmc driver (reptation.f:872-921) with branch2
// (reptation.f:2162-2271), each walker playing one MPI rank that holds one
// configuration.
//
// A step is mmstep moves of every walker (the VMC step of qmc_vmc.hip: the
// rank's own random stream), each followed by the walker's weight factor and
// the weighted averages(2), then branch2: the weights of all ranks, gathered
// in rank order, are normalized to the population and combed with the second
// generator, which every rank draws alike; each rank left with no copy then
// receives one from the lowest rank with copies to spare (the send/receive
// loop of branch2).  As in the reference's send/receive, the receiving rank
// takes the configuration, drift, Laplacian and properties, and keeps its own
// walker age and fixed-phase term (reptation.f:2279-2317 send x, g, h and
// the properties; the age and sign live in separate arrays).
#include "qmc_internal.h"

#include <type_traits>

#define DMC_WMULT 10.0  // branch2's bound of a weight (reptation.f:2167-2168)

// Start of a step: every weight 1 (dmc, reptation.f:886-890).
__global__ void k_dmc_begin(int nw, double* __restrict__ wate) {
  const int w = blockIdx.x * blockDim.x + threadIdx.x;
  if (w < nw) wate[w] = 1.0;
}

// branch2 (reptation.f:2162-2271) over the nw ranks.  What the reference forms
// in rank order, one operation after the other, stays in that order on one
// thread: the sum of the weights, the sum of their fractional parts and the
// comb's running sum k.  Everything else is spread over the workgroup: the
// bound, the normalization, the integer parts, the comb's draws and marks, the
// transfers.  LDS: nw doubles (the weights, then their fractional parts,
// then the prefix sums of the extra copies) and nw ints (the
// multiplicities).  On return src[j] is the walker j takes its configuration
// from.
//
// The comb (reptation.f:2196-2210) makes nint(k0) draws of rannyu2, one in each
// unit of k.  The reference moves its walker pointer while k < r (then marks
// the walker), then while k < 1, and subtracts 1 from k before each draw.  A
// draw r is below 1, so that whether k has reached 1 does not depend on r:
// walker j adds its fractional part, and 1 is taken off when k is then 1 or
// more, which is what the fraction of k leaves (k < 2, the subtraction is
// exact).  That chain, two operations per walker, is all that thread does; k0
// is summed by a second wavefront meanwhile.  Thread c takes the walkers from
// S c on: it gets k there, repeats their additions, counts the units that end
// before them, jumps the stream to their draw and marks in parallel.  With the
// draws, the comparisons with r and the marks on the one thread too, 4096
// walkers took 242 us (now 72).
#define DMC_BRANCH_THREADS 1024
#define DMC_CHUNK 16

// f(j, v[j]) for j = 0..nw-1 in order, two register chunks read in turn, each a
// chunk's walk ahead of its use (the barriers keep the compiler from moving the
// reads down to it).
template <class F>
__device__ __forceinline__ void dmc_in_order(const double* v, int nw, F&& f) {
  constexpr int C = DMC_CHUNK;
  const int n = nw / (2 * C) * (2 * C);
  double a[C], b[C];
  if (n > 0) {
#pragma unroll
    for (int u = 0; u < C; u++) a[u] = v[u];
  }
  for (int j = 0; j < n; j += 2 * C) {
#pragma unroll
    for (int u = 0; u < C; u++) b[u] = v[j + C + u];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < C; u++) f(j + u, a[u]);
    const int jn = j + 2 * C < n ? j + 2 * C : j;
#pragma unroll
    for (int u = 0; u < C; u++) a[u] = v[jn + u];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < C; u++) f(j + C + u, b[u]);
  }
  for (int j = n; j < nw; j++) f(j, v[j]);
}

// Exclusive prefix sums over the workgroup of each thread's a and b; ta: the
// total of a.
__device__ __forceinline__ void dmc_scan(int tid, int* pa, int* pb, int& a, int& b, int& ta) {
  const int a0 = a, b0 = b;
  block_sync();
  pa[tid] = a;
  pb[tid] = b;
  block_sync();
  for (int o = 1; o < DMC_BRANCH_THREADS; o <<= 1) {
    const int aa = tid >= o ? pa[tid - o] : 0, ab = tid >= o ? pb[tid - o] : 0;
    block_sync();
    pa[tid] += aa;
    pb[tid] += ab;
    block_sync();
  }
  a = pa[tid] - a0;
  b = pb[tid] - b0;
  ta = pa[DMC_BRANCH_THREADS - 1];
}

struct DmcBranchShared {
  // places used one after the other
  union {
    struct {
      double somma;
      int odd;
    };
    double start[DMC_BRANCH_THREADS];
    int scan[2][DMC_BRANCH_THREADS];
  };
  long draws;
};

__global__ __launch_bounds__(DMC_BRANCH_THREADS) void k_dmc_branch(int nw, double* __restrict__ wate,
                                                                   int64_t* __restrict__ rng2,
                                                                   int32_t* __restrict__ src,
                                                                   int32_t* __restrict__ counts) {
  extern __shared__ __attribute__((aligned(16))) unsigned char dmc_lds[];
  double* sw = reinterpret_cast<double*>(dmc_lds);
  int* sm = reinterpret_cast<int*>(sw + nw);
  __shared__ DmcBranchShared sh;
  const int tid = threadIdx.x;
  const uint64_t st0 = (uint64_t)rng2[0];
  if (tid == 0) sh.odd = 0;
  // weights above wmult are bounded (reptation.f:2176-2182)
  for (int i = tid; i < nw; i += DMC_BRANCH_THREADS) {
    double v = wate[i];
    if (v > DMC_WMULT) {
      v = DMC_WMULT;
      atomicAdd(&counts[1], 1);
      if (i == 0) atomicAdd(&counts[2], 1);
    }
    sw[i] = v;
  }
  block_sync();
  if (tid == 0) {
    double somma = 0.0;
    dmc_in_order(sw, nw, [&](int, double v) { somma = somma + v; });
    sh.somma = somma;
  }
  block_sync();
  // multiplicities: integer parts, and the fractional parts to comb
  // (reptation.f:2189-2195)
  const double somma = sh.somma;
  bool odd = false;
  for (int i = tid; i < nw; i += DMC_BRANCH_THREADS) {
    const double ww = ((double)nw * sw[i]) / somma;
    const int tm = (int)ww;
    const double v = ww - (double)tm;
    sm[i] = tm;
    sw[i] = v;
    odd |= !(v >= 0.0 && v < 1.0);
  }
  if (odd) sh.odd = 1;
  block_sync();
  // threads' walkers, in order
  const int S = nw <= 4 * DMC_BRANCH_THREADS ? 4 : nw <= 8 * DMC_BRANCH_THREADS ? 8 : 16;
  const int i0 = min(nw, tid * S), i1 = min(nw, i0 + S);
  const bool any_odd = sh.odd;
  block_sync();
  if (any_odd) {
    // fractional parts outside [0, 1) (weights below 0 or that are no
    // numbers): the reference's walk as it is, on one thread
    if (tid == 0) {
      double k0 = 0.0, k = 0.0;
      for (int i = 0; i < nw; i++) k0 = k0 + sw[i];
      const long ndraw = lround(k0);
      uint64_t st = st0;
      long d = ndraw > 0 ? 1 : 0;
      double r = d ? rannyu(st) : 0.0;
      bool seek_r = true;  // k = 1 - 1 before the first draw
      for (int j = 0; j < nw && d > 0; j++) {
        k = k + sw[j];
        for (;;) {
          if (seek_r) {
            if (k < r) break;
            sm[j] += 1;
            seek_r = false;
          }
          if (k < 1.0) break;
          if (d >= ndraw) {
            d = 0;
            break;
          }
          k = k - 1.0;
          r = rannyu(st);
          d++;
          seek_r = true;
        }
      }
      rng2[0] = (int64_t)st;
    }
  } else {
    // k at walker S c, c = 0, 1, ..: with its fractional part, before 1 is
    // taken off
    auto chain = [&](auto stride) {
      constexpr int S = decltype(stride)::value;
      double k = 0.0;
      dmc_in_order(sw, nw, [&](int j, double v) {
        const double t = k + v;
        if (j % S == 0) sh.start[j / S] = t;
        k = __builtin_amdgcn_fract(t);
      });
    };
    if (tid == 0) {
      if (S == 4) chain(std::integral_constant<int, 4>{});
      else if (S == 8) chain(std::integral_constant<int, 8>{});
      else chain(std::integral_constant<int, 16>{});
    }
    if (tid == 64) {
      double k0 = 0.0;
      dmc_in_order(sw, nw, [&](int, double v) { k0 = k0 + v; });
      sh.draws = lround(k0);
    }
    block_sync();
    const long ndraw = sh.draws;
    // k after walker i0 - 1, and before 1 is taken off at walker i0
    double kb = 0.0, t0 = 0.0;
    if (i0 < i1) {
      t0 = sh.start[tid];
      if (i0 > 0) {
        kb = __builtin_amdgcn_fract(sh.start[tid - 1]);
        for (int i = i0 - S + 1; i < i0; i++) kb = __builtin_amdgcn_fract(kb + sw[i]);
      }
    }
    int ends = 0, none = 0, units;
    double t = t0;
    for (int i = i0; i < i1; i++) {
      if (i > i0) t = __builtin_amdgcn_fract(t) + sw[i];
      ends += t >= 1.0 ? 1 : 0;
    }
    dmc_scan(tid, sh.scan[0], sh.scan[1], ends, none, units);
    long d = 1 + ends;  // the draw walker i0 is combed with, if it is made
    if (i0 < i1 && d <= ndraw) {
      uint64_t st = (lcg_pow((uint32_t)d) * st0) & ((1ULL << 48) - 1ULL);
      double r = (double)st * 0x1p-48;
      // not marked by a walker before: k is still below it (the first draw's
      // first walker has none before)
      bool seek_r = i0 == 0 || kb < r;
      t = t0;
      for (int i = i0; i < i1; i++) {
        if (i > i0) t = __builtin_amdgcn_fract(t) + sw[i];
        int mk = 0;
        if (seek_r && t >= r) {
          mk = 1;
          seek_r = false;
        }
        if (t >= 1.0) {
          if (d < ndraw) {
            r = rannyu(st);
            seek_r = t - 1.0 < r;
            if (!seek_r) mk++;
          }
          d++;
        }
        if (mk) sm[i] += mk;
        if (d > ndraw) break;
      }
    }
    if (tid == 0 && ndraw > 0) {
      const long made = 1 + (units < ndraw - 1 ? (long)units : ndraw - 1);
      rng2[0] = (int64_t)((lcg_pow((uint32_t)made) * st0) & ((1ULL << 48) - 1ULL));
    }
  }
  block_sync();
  // The ranks left with no copy take the extra copies of the others: each
  // transfer from the lowest rank with more than one to the lowest rank with
  // none (reptation.f:2220-2258).  So receiver q (in walker order) takes
  // from the walker s whose extra copies, counted in walker order, cover q:
  // E(s) <= q < E(s+1), E the exclusive prefix sum of max(mult - 1, 0).
  int e = 0, q = 0, etot;
  for (int i = i0; i < i1; i++) {
    e += max(sm[i] - 1, 0);
    q += sm[i] == 0 ? 1 : 0;
  }
  dmc_scan(tid, sh.scan[0], sh.scan[1], e, q, etot);
  // exclusive prefix sums of the extras per walker, in the fractional parts'
  // place (no longer read); E(nw) is the total
  double* E = sw;
  for (int i = i0; i < i1; i++) {
    E[i] = (double)e;
    e += max(sm[i] - 1, 0);
  }
  block_sync();
  for (int i = i0; i < i1; i++) {
    if (sm[i] >= 1) {
      src[i] = i;
      continue;
    }
    int sidx = i;
    if (q < etot) {
      // the last walker with E <= q
      int lo = 0, hi = nw - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if ((int)E[mid] <= q) lo = mid;
        else hi = mid - 1;
      }
      sidx = lo;
    }
    src[i] = sidx;
    q++;
  }
}

static size_t dmc_branch_lds(int nw) { return (size_t)nw * (sizeof(double) + sizeof(int)); }

// The copies the branching asks for: walker j takes the configuration, drift,
// Laplacian and properties of walker src[j].  The walkers copied from keep
// their own (a multiplicity of at least 1), so no walker is both read and
// written.  One wavefront per walker.
__global__ __launch_bounds__(QMC_BLOCK) void k_dmc_copy(int nw, int N, int np_, const int32_t* __restrict__ src,
                                                        double* __restrict__ x, double* __restrict__ g,
                                                        double* __restrict__ h, double* __restrict__ props) {
  const int w = blockIdx.x * (QMC_BLOCK / 64) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (w >= nw) return;
  const int from = src[w];
  if (from == w || from < 0 || from >= nw) return;
  for (int k = lane; k < 2 * N; k += 64) {
    x[(int64_t)w * 2 * N + k] = x[(int64_t)from * 2 * N + k];
    g[(int64_t)w * 2 * N + k] = g[(int64_t)from * 2 * N + k];
  }
  if (lane < 2) h[(int64_t)w * 2 + lane] = h[(int64_t)from * 2 + lane];
  for (int k = lane; k < np_; k += 64) props[(int64_t)w * np_ + k] = props[(int64_t)from * np_ + k];
}

static int check_dmc(qmc_ctx* c, int nw, const qmc_dmc_state* d) {
  if (!c || !d || nw < 0) return arg_fail("bad DMC state");
  if (nw > 0 && (!d->wate || !d->wsum || !d->src || !d->rng2 || !d->counts))
    return arg_fail("null DMC buffer");
  return QMC_OK;
}

// The branching's LDS holds 12 bytes per walker beside the kernel's own 8.2 KB
// (16-byte steps): the populations that the LDS of a workgroup can take, 12969
// walkers at 160 KB.
static int dmc_branch_check(qmc_ctx* c, int nw) {
  int lds_max = 0;
  HIPCHK(hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, c->device));
  const size_t need = ((sizeof(DmcBranchShared) + 15) & ~(size_t)15) + dmc_branch_lds(nw);
  if (need > (size_t)lds_max) return arg_fail("DMC population above what the branching's LDS holds", QMC_ERR_LIMIT);
  if (need > 65536)
    HIPCHK(hipFuncSetAttribute((const void*)k_dmc_branch, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)dmc_branch_lds(nw)));
  return QMC_OK;
}

extern "C" int qmc_dmc_branch(qmc_ctx* c, int nw, double* d_wate, int64_t* d_rng2, int32_t* d_src,
                              int32_t* d_counts, void* stream) {
  if (!c || nw < 0 || (nw > 0 && (!d_wate || !d_rng2 || !d_src || !d_counts)))
    return arg_fail("bad branching arguments");
  if (nw == 0) return QMC_OK;
  HIPCHK(hipSetDevice(c->device));
  int rc;
  rc = dmc_branch_check(c, nw);
  if (rc) return rc;
  hipLaunchKernelGGL(k_dmc_branch, dim3(1), dim3(DMC_BRANCH_THREADS), dmc_branch_lds(nw), (hipStream_t)stream,
                     nw, d_wate, d_rng2, d_src, d_counts);
  HIPCHK(hipGetLastError());
  return QMC_OK;
}

extern "C" int qmc_dmc_sweep(qmc_ctx* c, const qmc_walkers* w, const qmc_dmc_state* d, int nsteps,
                             const qmc_dmc_params* prm, void* stream) {
  if (!c || !w || !prm) return arg_fail("null argument");
  int rc = check_dmc(c, w->nw, d);
  if (rc) return rc;
  if (w->nw > 0 && (!w->x || !w->g || !w->h || !w->props || !w->grad2_ph || !w->age || !w->rng))
    return arg_fail("null walker buffer");
  if (w->nw > 0 && !w->blk) return arg_fail("DMC needs the block sums (w->blk)");
  if (w->nw == 0 || nsteps <= 0) return QMC_OK;
  if (!(prm->delta > 0.0)) return arg_fail("delta must be positive");
  if (prm->mmstep < 1) return arg_fail("mmstep must be at least 1");
  HIPCHK(hipSetDevice(c->device));
  hipStream_t st = (hipStream_t)stream;
  rc = dmc_branch_check(c, w->nw);
  if (rc) return rc;
  rc = ensure_vmc_scratch(c, w->nw);
  if (rc) return rc;
  rc = ensure_ws(c, w->nw);
  if (rc) return rc;
  const DevSys& s = c->s;
  c->delta = prm->delta;
  // sigma (reptation.f:855-870)
  const double var0 = 2.0 * s.hbs2m[0] * prm->delta;
  const double var1 = s.ntypes > 1 ? 2.0 * s.hbs2m[1] * prm->delta : 1.0;
  const int nw = w->nw, NP = c->info.n_props, jetot = c->info.jetot - 1;
  const DmcWeight dm{d->wate, d->wsum, d->counts, prm->etrial, prm->delta, (double)prm->mmult, jetot};
  const int wpb = QMC_BLOCK / 64;
  for (int k = 0; k < nsteps; k++) {
    hipLaunchKernelGGL(k_dmc_begin, dim3((nw + 255) / 256), dim3(256), 0, st, nw, d->wate);
    for (int m = 0; m < prm->mmstep; m++) {
      rc = vmc_step(c, w, st, prm->delta, var0, var1, prm->mage, prm->bm_order, nullptr, nullptr, &dm);
      if (rc) return rc;
    }
    hipLaunchKernelGGL(k_dmc_branch, dim3(1), dim3(DMC_BRANCH_THREADS), dmc_branch_lds(nw), st, nw, d->wate,
                       d->rng2, d->src, d->counts);
    // without this branching's sources no walker is copied
    HIPCHK(hipGetLastError());
    hipLaunchKernelGGL(k_dmc_copy, dim3((nw + wpb - 1) / wpb), dim3(QMC_BLOCK), 0, st, nw, s.nptot, NP, d->src,
                       w->x, w->g, w->h, w->props);
  }
  HIPCHK(hipGetLastError());
  return QMC_OK;
}
