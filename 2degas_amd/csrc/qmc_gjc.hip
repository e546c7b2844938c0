// qmc_gjc.hip -- determinant path for complex orbitals (twisted boundary
// conditions, open shells) on the FP64 matrix cores, up to 64 particles per spin.
//
// F_b = A^-1 (G_b A) (zv of reptation.f:10182-10194, with A(i,j) = exp(i g_i .
// q_j), G_b = diag(i g^b)) and log|det A| (zgedi's det, reptation.f:9412-9430)
// by the elimination of qmc_gjr.hip on the complex augmented matrix
// [A | G_x A | G_y A]: one workgroup of NT wavefronts per (walker, spin), NT the
// 16-row tiles, wavefront c holding column tile c of each part as real and
// imaginary accumulators (a complex product is four real MFMAs); blocks of 4
// columns, one barrier each; row p_k of the two right parts ends as piv_k
// F_b(k, .).  Pivot choice is zgefa's (largest |re|+|im| among the rows not yet
// used, reptation.f:9286-9298; rows whose magnitudes agree to 14 bits may be
// taken in another order, which changes rounding only).
//
// What bounds it: at 64 particles the matrix cores (2700 products per walker) and
// the pivot chain, which two workgroups per CU hide from each other (192 of 256
// registers are accumulators); at small sizes the chain alone.  An in-place
// inverse with two barriers and a copy of the matrix in LDS per block, then two
// complex products, always on 64 rows, took 250 us for 4096 walkers of N=26 (now
// 63), 267 us for 2048 of N=58 (now 130), 218 us for 1024 of N=74 (now 193), 191
// us for 1024 of 61 polarized particles (now 180) and 16 us for one of N=26 (now
// 10).  Wavefronts per SIMD: what the accumulators allow without spills (48
// registers per row tile); one part's operands are in registers at a time.
#include "qmc_gj.h"

template <int NT>
constexpr bool gc_copies = NT == 1;  // as gr_copies

template <int NT, int NP>
struct GcShared {
  static constexpr bool COPY = gc_copies<NT>;
  static constexpr int LDC = 17, PART = COPY ? 16 * NT * LDC : 8 * 16;
  double q[2 * 16 * NT], g[2 * 16 * NT];
  double2 panel[COPY ? 1 : 16 * NT * 4];  // the block's columns, row r at 4 r (else read from the copy)
  double2 Fl[2][16 * NT * 4];             // F' of the block, row r at 4 r
  // per wavefront: its column tiles, or the block's pivot rows in them and spare
  // places
  double2 u[NT][NP * PART];
  double2 pinv[16 * NT];  // by pivot row
  double pmod[16 * NT];
  int prow[2][4];
  int rank[16 * NT];  // step of pivot row r, -1: none
  int used[16 * NT];
  int sing;
};

// The pivot steps of columns k0..k0+nb-1 by one wavefront, lane = row, as
// gr_pivots.
template <int NT, int NP>
__device__ __forceinline__ void gc_pivots(GcShared<NT, NP>& sh, const double2* panel, int buf, int k0, int nb,
                                          int lane) {
  const bool in = NT == 4 || lane < 16 * NT;
  zd P[4], Fp[4];
  bool used = true;
#pragma unroll
  for (int j = 0; j < 4; j++) P[j] = Fp[j] = zmk(0.0, 0.0);
  if (in) {
#pragma unroll
    for (int j = 0; j < 4; j++) P[j] = zmk(panel[j].x, panel[j].y);
    used = sh.used[lane] != 0;
  }
#pragma unroll
  for (int j = 0; j < 4; j++) {
    if (j < nb) {
      const double dl = fma(P[j].x, P[j].x, P[j].y * P[j].y), rl = gr_rcp(dl);
      const unsigned top = (unsigned)(__double_as_longlong(cabs1(P[j])) >> 32);
      const unsigned key = used ? 0u : ((((top >> 6) + 1u) << 6) | (unsigned)(63 - lane));
      const int p = 63 - (int)(gj_wave_max(key) & 63u);
      const zd pi = zmk(gj_readlane(P[j].x * rl, p), gj_readlane(-P[j].y * rl, p));
      const bool me = lane == p;
      const zd f = zmul(P[j], pi), nf = me ? zmk(0.0, 0.0) : zmk(-f.x, -f.y);
#pragma unroll
      for (int jj = j + 1; jj < 4; jj++)
        P[jj] = zfma(nf, zmk(gj_readlane(P[jj].x, p), gj_readlane(P[jj].y, p)), P[jj]);
#pragma unroll
      for (int i = 0; i < j; i++)
        Fp[i] = zfma(nf, zmk(gj_readlane(Fp[i].x, p), gj_readlane(Fp[i].y, p)), Fp[i]);
      Fp[j] = nf;
      if (me) {
        used = true;
        sh.prow[buf][j] = p;
        sh.rank[p] = k0 + j;
        sh.pinv[p] = make_double2(pi.x, pi.y);
        sh.pmod[p] = dl;
        sh.used[p] = 1;
        if (!(dl > 0.0)) sh.sing = 1;
      }
    } else if (lane == 0) {
      sh.prow[buf][j] = 0;
    }
  }
  if (in) {
#pragma unroll
    for (int j = 0; j < 4; j++) sh.Fl[buf][4 * lane + j] = make_double2(Fp[j].x, Fp[j].y);
  }
}

template <int NT, bool VAL>
__global__ __launch_bounds__(64 * NT, VAL || NT == 1 ? 4 : 2) void k_gjc(DevSys s, WsLayout L, double* __restrict__ ws,
                                                              double* __restrict__ Fbuf, int sp0) {
  constexpr int NP = VAL ? 1 : 3;  // parts of the augmented matrix
  typedef GcShared<NT, NP> S;
  __shared__ __attribute__((aligned(16))) S sh;
  const int w = blockIdx.x, sp = sp0 + blockIdx.y;
  if (s.nact && w >= *s.nact) return;
  const int m = pick2(s.np, sp);
  if (m == 0) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // MFMA lane roles: accumulator rows lr + 4v, column lc; operand k index lr
  const int lr = lane >> 4, lc = lane & 15, ct = wave, col = 16 * wave + lc;
  const double* qw = ws + (int64_t)w * L.per_walker + L.off_q + 2 * pick2(s.ipf, sp);
  for (int e = tid; e < 2 * m; e += 64 * NT) {
    sh.q[e] = qw[e];
    sh.g[e] = s.gvec[e];
  }
  for (int r = tid; r < 16 * NT; r += 64 * NT) {
    sh.used[r] = r >= m;
    sh.rank[r] = -1;
  }
  if (tid == 0) sh.sing = 0;
  block_sync();
  gr_d4 re[NP][NT], im[NP][NT];
  {
    const bool jn = col < m;
    const double qx = jn ? sh.q[2 * col] : 0.0, qy = jn ? sh.q[2 * col + 1] : 0.0;
#pragma unroll
    for (int T = 0; T < NT; T++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int r = 16 * T + lr + 4 * v;
        double sv = 0.0, cv = 0.0, gx = 0.0, gy = 0.0;
        if (jn && r < m) {
          gx = sh.g[2 * r];
          gy = sh.g[2 * r + 1];
          qsincos_sreg(fma(gx, qx, gy * qy), &sv, &cv);
        }
        re[0][T][v] = cv;
        im[0][T][v] = sv;
        if constexpr (NP == 3) {
          re[1][T][v] = -gx * sv;
          im[1][T][v] = gx * cv;
          re[2][T][v] = -gy * sv;
          im[2][T][v] = gy * cv;
        }
      }
  }
  double2* ub = sh.u[wave];
  constexpr int LDC = S::LDC, PART = S::PART;
  auto copy = [&](auto t0, auto t1) {
#pragma unroll
    for (int t = decltype(t0)::value; t < decltype(t1)::value; t++)
#pragma unroll
      for (int T = 0; T < NT; T++)
#pragma unroll
        for (int v = 0; v < 4; v++)
          ub[t * PART + (16 * T + lr + 4 * v) * LDC + lc] = make_double2(re[t][T][v], im[t][T][v]);
  };
  typedef std::integral_constant<int, 0> C0;
  typedef std::integral_constant<int, 1> C1;
  typedef std::integral_constant<int, NP> CN;
  auto panel = [&](int k0, int buf) {
    const double2* src;
    if constexpr (S::COPY) {
      copy(C0{}, C1{});
      src = ub + lane * LDC + (k0 & 15);
    } else {
      const int j = lc - (k0 & 15);
      if (j >= 0 && j < 4) {
#pragma unroll
        for (int T = 0; T < NT; T++)
#pragma unroll
          for (int v = 0; v < 4; v++)
            sh.panel[4 * (16 * T + lr + 4 * v) + j] = make_double2(re[0][T][v], im[0][T][v]);
      }
      src = sh.panel + 4 * lane;
    }
    gr_wave_sync();
    // every other wavefront waits for these steps: they issue first
    __builtin_amdgcn_s_setprio(1);
    gc_pivots(sh, src, buf, k0, min(4, m - k0), lane);
    __builtin_amdgcn_s_setprio(0);
    if constexpr (S::COPY) copy(C1{}, CN{});
  };
  if (ct == 0) panel(0, 0);
  else if constexpr (S::COPY) copy(C0{}, CN{});
  for (int k0 = 0; k0 < m; k0 += 4) {
    const int buf = (k0 >> 2) & 1, nb = min(4, m - k0);
    block_sync();
    int p = 0;
    if constexpr (S::COPY) {
      p = sh.prow[buf][lr];
    } else {
      int pb[4];
#pragma unroll
      for (int k = 0; k < 4; k++) pb[k] = __builtin_amdgcn_readfirstlane(sh.prow[buf][k]);
#pragma unroll
      for (int k = 0; k < 4; k++) {
        // the lanes that hold row p; the others' values go to their own places
        // behind the block's rows.  (Between the scheduling barriers the picks
        // share one index mode instead of a switch for each.)
        double2* to = ub + (lr == (pb[k] & 3) ? k * 16 : (4 + lr) * 16) + lc;
        double2 row[NP];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < NP; t++) {
          row[t].x = gr_pick<NT>(re[t], pb[k] >> 2);
          row[t].y = gr_pick<NT>(im[t], pb[k] >> 2);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < NP; t++) to[t * PART] = row[t];
      }
      gr_wave_sync();
    }
    double2 fo[NT];
#pragma unroll
    for (int T = 0; T < NT; T++) fo[T] = sh.Fl[buf][4 * (16 * T + lc) + lr];
#pragma unroll
    for (int t = 0; t < NP; t++) {
      // one part's operands at a time: the accumulators leave few registers
      __asm__ volatile("" ::: "memory");
      if (t == 0 && (k0 >> 4) > ct) continue;  // A's columns here are all eliminated
      double2 uo = ub[t * PART + (S::COPY ? p * LDC + lc : lane)];
      uo.x = lr < nb ? uo.x : 0.0;
      uo.y = lr < nb ? uo.y : 0.0;
      const double ny = -uo.y;
#pragma unroll
      for (int T = 0; T < NT; T++) {
        re[t][T] = gr_mfma(fo[T].x, uo.x, re[t][T]);
        im[t][T] = gr_mfma(fo[T].x, uo.y, im[t][T]);
      }
#pragma unroll
      for (int T = 0; T < NT; T++) {
        re[t][T] = gr_mfma(fo[T].y, ny, re[t][T]);
        im[t][T] = gr_mfma(fo[T].y, uo.x, im[t][T]);
      }
    }
    if (k0 + 4 < m) {
      if (((k0 + 4) >> 4) == ct) panel(k0 + 4, buf ^ 1);
      else if constexpr (S::COPY) copy(C0{}, CN{});
    }
  }
  block_sync();
  double* dsc = ws + (int64_t)w * L.per_walker + pick2(L.off_det, sp);
  if constexpr (!VAL) {
    // F_b(k, j): row p_k of part b over piv_k; the diagonal also goes to the
    // per-orbital terms (real and imaginary parts)
    double* Fd = dsc + DS_N + 2 * s.nptot + 3 * m;
    zd* Fg = (zd*)(Fbuf + (int64_t)w * L.f_per_walker + pick2(L.f_off, sp));
    const int j = col;
    if (j < m) {
#pragma unroll
      for (int T = 0; T < NT; T++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
          __asm__ volatile("" ::: "memory");
          const int r = 16 * T + lr + 4 * v;
          const int k = sh.rank[r];
          if (k >= 0) {
            const zd pi = zmk(sh.pinv[r].x, sh.pinv[r].y);
#pragma unroll
            for (int b = 0; b < 2; b++) {
              const zd f = zmul(zmk(re[1 + b][T][v], im[1 + b][T][v]), pi);
              if (!s.plain) Fg[(b * m + k) * m + j] = f;
              if (k == j) {
                Fd[4 * j + 2 * b] = f.x;
                Fd[4 * j + 2 * b + 1] = f.y;
              }
            }
          }
        }
    }
  }
  if (wave == 0) {
    const bool piv = lane < 16 * NT && sh.rank[lane < 16 * NT ? lane : 0] >= 0;
    const double t = wave_sum(piv ? 0.5 * log(sh.pmod[lane]) : 0.0);
    if (lane == 0) {
      dsc[DS_LOGDET] = t;
      dsc[DS_SING] = sh.sing ? 1.0 : 0.0;
    }
  }
}

template <bool VAL>
static void gjc_spins(const DevSys& s, const WsLayout& L, int nw, int sp0, int nsp, int nt, double* ws, double* F,
                      hipStream_t st) {
  const dim3 grid(nw, nsp);
  switch (nt) {
    case 1: hipLaunchKernelGGL((k_gjc<1, VAL>), grid, dim3(64), 0, st, s, L, ws, F, sp0); break;
    case 2: hipLaunchKernelGGL((k_gjc<2, VAL>), grid, dim3(128), 0, st, s, L, ws, F, sp0); break;
    case 3: hipLaunchKernelGGL((k_gjc<3, VAL>), grid, dim3(192), 0, st, s, L, ws, F, sp0); break;
    default: hipLaunchKernelGGL((k_gjc<4, VAL>), grid, dim3(256), 0, st, s, L, ws, F, sp0); break;
  }
}

// One launch when the spins have the same tile count, else one per spin.
void launch_gjc(const DevSys& s, const WsLayout& L, int nw, bool value, double* ws, double* F, hipStream_t st) {
  auto go = [&](int sp0, int nsp, int nt) {
    if (value) gjc_spins<true>(s, L, nw, sp0, nsp, nt, ws, F, st);
    else gjc_spins<false>(s, L, nw, sp0, nsp, nt, ws, F, st);
  };
  int nt[2] = {0, 0};
  for (int sp = 0; sp < s.ntypes; sp++) nt[sp] = (s.np[sp] + 15) / 16;
  if (s.ntypes == 2 && nt[0] == nt[1]) {
    if (nt[0]) go(0, 2, nt[0]);
    return;
  }
  for (int sp = 0; sp < s.ntypes; sp++)
    if (nt[sp]) go(sp, 1, nt[sp]);
}
