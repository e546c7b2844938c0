// qmc_gjr.hip -- determinant path for real orbitals: spins whose plane waves
// come with their opposites (every untwisted closed shell), up to 64
// particles per spin.
//
// With g and -g both occupied the two rows e^{+-i g.q} of A are a constant
// combination of cos(g.q) and sin(g.q) (a 2 x 2 block of determinant -2i), so
// with R the real matrix of those rows F_b = A^-1 (i g^b A) equals
// R^-1 D_b R, D_b R being the derivative rows (-g^b sin, g^b cos), and
// log|det A| = log|det R| + (pairs) log 2.  Everything is real: a quarter of
// the arithmetic of the complex matrices of qmc_gjc.hip and half of their
// registers.
//
// One workgroup of NT wavefronts per (walker, spin), NT the 16-row tiles of R.
// The augmented matrix [R | D_x R | D_y R] is held in v_mfma_f64_16x16x4f64
// accumulators, wavefront c holding column tile c of each of the three parts
// (3 NT tiles), and R is eliminated by Gauss-Jordan steps with partial
// pivoting, so that row p_k of the two right parts ends as piv_k F_b(k, .):
// there is no inverse and no second product.  Columns are eliminated in
// blocks of 4.  The wavefront that holds the block's columns passes them
// through LDS (lane = row), takes the 4 pivot steps and posts the block's row
// operations as a rank-4 update M += F' U, U the block's 4 pivot rows as they
// were before it.  Every wavefront takes U for its own columns from its own
// accumulators, so one barrier per block suffices, the posted operands being
// double buffered.  Column tiles of R whose columns are all eliminated are
// left out.
//
// The chain from block to block bounds the kernel (panel, pivot search, posted
// rows, update), so U must not lengthen it: rows are taken from the registers
// in index mode or, where the LDS allows, from a copy of the tiles stored while
// the pivot steps run, which then also is the panel.  By a switch over the
// registers, a dozen branches per row: N=122, 4096 walkers 471 us (now 436);
// log|det| alone, N=58, 512 walkers 17.7 us (now 13.5); N=26, 256 walkers 9.9 us
// (now 7.9), but 4096 walkers of N=26 33 us (now 34: the copy's LDS).
//
// Rows: the two rows of plane-wave pair n sit in one lane of a tile (rows
// r and r + 4), so that one sin/cos gives R and both derivatives of both
// rows.  A zero plane wave is the cos row of a pair of its own, whose sin row
// does not take part.
#include "qmc_gj.h"

// Whether a wavefront keeps a copy of its column tiles in LDS for the pivot
// rows to be read from (as many stores as picking the four rows out of the
// registers for one row tile, and none of them between a block's barrier and its
// update); beyond, the LDS would bound the walkers per CU.
template <int NT, int NP>
constexpr bool gr_copies = NT == 1 || (NT == 2 && NP == 1);

template <int NT, int NP>
struct GrShared {
  static constexpr bool COPY = gr_copies<NT, NP>;
  // a copied row's stride: rows 16 lanes read together fall on different banks
  static constexpr int LDC = 18, PART = COPY ? 16 * NT * LDC : 8 * 16;
  double q[2 * 16 * NT], g[2 * 8 * NT];
  double panel[COPY ? 1 : 16 * NT * 4];  // the block's columns, row r at 4 r (else read from the copy)
  double Fl[2][16 * NT * 4];      // F' of the block, row r at 4 r
  // per wavefront: its column tiles, or the block's pivot rows in them and spare
  // places
  __attribute__((aligned(16))) double u[NT][NP * PART];
  double pinv[16 * NT], pabs[16 * NT];  // by pivot row
  int prow[2][4];
  int rank[16 * NT];              // step of pivot row r, -1: none
  int used[16 * NT];
  int sing;
};

// The pivot steps of columns k0..k0+nb-1 (panel in LDS) by one wavefront,
// lane = row.  Pivot: the largest magnitude among the unused rows, rows whose
// top 14 bits agree in the order of their index.  Every lane forms the
// reciprocal of its own entry while the maximum is searched, so that the
// chain waits for the longer of the two only.
template <int NT, int NP>
__device__ __forceinline__ void gr_pivots(GrShared<NT, NP>& sh, const double* panel, int buf, int k0, int nb,
                                          int lane) {
  const bool in = NT == 4 || lane < 16 * NT;
  double P[4] = {0, 0, 0, 0}, Fp[4] = {0, 0, 0, 0};
  bool used = true;
  if (in) {
#pragma unroll
    for (int j = 0; j < 4; j++) P[j] = panel[j];
    used = sh.used[lane] != 0;
  }
#pragma unroll
  for (int j = 0; j < 4; j++) {
    if (j < nb) {
      const unsigned top = (unsigned)(__double_as_longlong(P[j]) >> 32) & 0x7fffffffu;
      const unsigned key = used ? 0u : ((((top >> 6) + 1u) << 6) | (unsigned)(63 - lane));
      const double ri = gr_rcp(P[j]);
      const int p = 63 - (int)(gj_wave_max(key) & 63u);
      const double pi = gj_readlane(ri, p);
      const bool me = lane == p;
      const double nf = me ? 0.0 : -(P[j] * pi);
#pragma unroll
      for (int jj = j + 1; jj < 4; jj++) P[jj] = fma(nf, gj_readlane(P[jj], p), P[jj]);
#pragma unroll
      for (int i = 0; i < j; i++) Fp[i] = fma(nf, gj_readlane(Fp[i], p), Fp[i]);
      Fp[j] = nf;
      if (me) {
        used = true;
        const double a = fabs(P[j]);
        sh.prow[buf][j] = p;
        sh.rank[p] = k0 + j;
        sh.pinv[p] = pi;
        sh.pabs[p] = a;
        sh.used[p] = 1;
        if (!(a > 0.0)) sh.sing = 1;
      }
    } else if (lane == 0) {
      sh.prow[buf][j] = 0;
    }
  }
  if (in) {
#pragma unroll
    for (int j = 0; j < 4; j++) sh.Fl[buf][4 * lane + j] = Fp[j];
  }
}

// Tables of the spin into LDS: quasi-coordinates (or positions) and pairs;
// rows without an orbital are marked used.
template <int NT, int NP>
__device__ __forceinline__ void gr_setup(GrShared<NT, NP>& sh, const double* __restrict__ q, const double* __restrict__ gp,
                                         int m, int nslot, int zero, int tid) {
  for (int e = tid; e < 2 * m; e += 64 * NT) sh.q[e] = q[e];
  for (int e = tid; e < 2 * nslot; e += 64 * NT) sh.g[e] = gp[e];
  for (int r = tid; r < 16 * NT; r += 64 * NT) {
    // row r = 16 T + lr + 4 v: pair T * 8 + (v >> 1) * 4 + lr, cos (v even) or sin
    const int v = (r >> 2) & 3, sl = (r >> 4) * 8 + (v >> 1) * 4 + (r & 3);
    sh.used[r] = sl >= nslot || (zero && sl == 0 && (v & 1));
    sh.rank[r] = -1;
  }
  if (tid == 0) sh.sing = 0;
  block_sync();
}

// The wavefront's column tile of R and, with NP = 3, of its two derivatives.
template <int NT, int NP>
__device__ __forceinline__ void gr_build(const GrShared<NT, NP>& sh, gr_d4 (&acc)[NP][NT], int m, int nslot, int col,
                                         int lr) {
  const bool jn = col < m;
  const double qx = jn ? sh.q[2 * col] : 0.0, qy = jn ? sh.q[2 * col + 1] : 0.0;
#pragma unroll
  for (int T = 0; T < NT; T++)
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int sl = T * 8 + h * 4 + lr;
      double sv = 0.0, cv = 0.0, gx = 0.0, gy = 0.0;
      if (jn && sl < nslot) {
        gx = sh.g[2 * sl];
        gy = sh.g[2 * sl + 1];
        qsincos_sreg(gx * qx + gy * qy, &sv, &cv);
      }
      acc[0][T][2 * h] = cv;
      acc[0][T][2 * h + 1] = sv;
      if constexpr (NP == 3) {
        acc[1][T][2 * h] = -gx * sv;
        acc[1][T][2 * h + 1] = gx * cv;
        acc[2][T][2 * h] = -gy * sv;
        acc[2][T][2 * h + 1] = gy * cv;
      }
    }
}

// The elimination, in blocks of 4 columns.  INPLACE (NP = 1): the columns of
// an eliminated block take the columns e_{p_j} of the identity, so that after
// the last block column k holds column p_k of the accumulated transform S,
// S R having row p_k equal to piv_k e_k; else R's eliminated column tiles are
// left out.  Ends with a barrier.
template <int NT, int NP, bool INPLACE>
__device__ __forceinline__ void gr_eliminate(GrShared<NT, NP>& sh, gr_d4 (&acc)[NP][NT], int m, int wave, int lane) {
  // MFMA lane roles: accumulator rows lr + 4v, column lc; operand k index lr
  const int lr = lane >> 4, lc = lane & 15, ct = wave;
  // the block's columns from the accumulators of the wavefront that holds
  // them to LDS, and its pivot steps
  double* ub = sh.u[wave];
  constexpr bool COPY = GrShared<NT, NP>::COPY;
  constexpr int LDC = GrShared<NT, NP>::LDC, PART = GrShared<NT, NP>::PART;
  // the wavefront's tiles of parts t0..t1-1 to its copy
  auto copy = [&](auto t0, auto t1) {
#pragma unroll
    for (int t = decltype(t0)::value; t < decltype(t1)::value; t++)
#pragma unroll
      for (int T = 0; T < NT; T++)
#pragma unroll
        for (int v = 0; v < 4; v++) ub[t * PART + (16 * T + lr + 4 * v) * LDC + lc] = acc[t][T][v];
  };
  typedef std::integral_constant<int, 0> C0;
  typedef std::integral_constant<int, 1> C1;
  typedef std::integral_constant<int, NP> CN;
  auto panel = [&](int k0, int buf) {
    const double* src;
    if constexpr (COPY) {
      copy(C0{}, C1{});
      src = ub + lane * LDC + (k0 & 15);
    } else {
      const int j = lc - (k0 & 15);
      if (j >= 0 && j < 4) {
#pragma unroll
        for (int T = 0; T < NT; T++)
#pragma unroll
          for (int v = 0; v < 4; v++) sh.panel[4 * (16 * T + lr + 4 * v) + j] = acc[0][T][v];
      }
      src = sh.panel + 4 * lane;
    }
    gr_wave_sync();
    // every other wavefront waits for these steps: they issue first
    __builtin_amdgcn_s_setprio(1);
    gr_pivots(sh, src, buf, k0, min(4, m - k0), lane);
    __builtin_amdgcn_s_setprio(0);
    if constexpr (COPY) copy(C1{}, CN{});
  };
  if (ct == 0) panel(0, 0);
  else if constexpr (COPY) copy(C0{}, CN{});
  for (int k0 = 0; k0 < m; k0 += 4) {
    const int buf = (k0 >> 2) & 1, nb = min(4, m - k0);
    block_sync();
    const bool left = INPLACE || (k0 >> 4) <= ct;  // R's columns here are not all eliminated
    int pb[4];
    double uo[NP], fo[NT];
    if constexpr (COPY) {
      const int p = sh.prow[buf][lr];
#pragma unroll
      for (int t = 0; t < NP; t++) {
        const double v = ub[t * PART + p * LDC + lc];
        uo[t] = lr < nb ? v : 0.0;
      }
    }
    if constexpr (!COPY || INPLACE) {
#pragma unroll
      for (int k = 0; k < 4; k++) pb[k] = __builtin_amdgcn_readfirstlane(sh.prow[buf][k]);
    }
    if constexpr (!COPY) {
#pragma unroll
      for (int k = 0; k < 4; k++) {
        // the lanes that hold row p; the others' values go to their own places
        // behind the block's rows.  (Between the scheduling barriers the picks
        // share one index mode instead of a switch for each.)
        double* to = ub + (lr == (pb[k] & 3) ? k * 16 : (4 + lr) * 16) + lc;
        double row[NP];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < NP; t++) row[t] = gr_pick<NT>(acc[t], pb[k] >> 2);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < NP; t++) to[t * PART] = row[t];
      }
      gr_wave_sync();
#pragma unroll
      for (int t = 0; t < NP; t++) uo[t] = lr < nb ? ub[t * PART + lane] : 0.0;
    }
#pragma unroll
    for (int T = 0; T < NT; T++) fo[T] = sh.Fl[buf][4 * (16 * T + lc) + lr];
    if constexpr (INPLACE) {
      const int jj = lc - (k0 & 15);
      if ((k0 >> 4) == ct && jj >= 0 && jj < nb) {
        const int pr = jj == 0 ? pb[0] : (jj == 1 ? pb[1] : (jj == 2 ? pb[2] : pb[3]));
#pragma unroll
        for (int T = 0; T < NT; T++)
#pragma unroll
          for (int v = 0; v < 4; v++) acc[0][T][v] = 16 * T + lr + 4 * v == pr ? 1.0 : 0.0;
        uo[0] = lr == jj ? 1.0 : 0.0;
      }
    }
    if (left) {
#pragma unroll
      for (int T = 0; T < NT; T++) acc[0][T] = gr_mfma(fo[T], uo[0], acc[0][T]);
    }
#pragma unroll
    for (int t = 1; t < NP; t++)
#pragma unroll
      for (int T = 0; T < NT; T++) acc[t][T] = gr_mfma(fo[T], uo[t], acc[t][T]);
    if (k0 + 4 < m) {
      if (((k0 + 4) >> 4) == ct) panel(k0 + 4, buf ^ 1);
      else if constexpr (COPY) copy(C0{}, CN{});
    }
  }
  block_sync();
}

template <int NT, bool VAL>
__global__ __launch_bounds__(64 * NT, NT == 4 ? 3 : 4) void k_gjr(DevSys s, WsLayout L, double* __restrict__ ws,
                                                                  double* __restrict__ Fbuf, int sp0) {
  constexpr int NP = VAL ? 1 : 3;  // parts of the augmented matrix
  __shared__ __attribute__((aligned(16))) GrShared<NT, NP> sh;
  const int w = blockIdx.x, sp = sp0 + blockIdx.y;
  if (s.nact && w >= *s.nact) return;
  const int m = pick2(s.np, sp);
  if (m == 0) return;
  const int nslot = pick2(s.nslot, sp), zero = pick2(s.zslot, sp);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane >> 4, col = 16 * wave + (lane & 15);
  gr_setup(sh, ws + (int64_t)w * L.per_walker + L.off_q + 2 * pick2(s.ipf, sp), sp ? s.gpair[1] : s.gpair[0], m,
           nslot, zero, tid);
  gr_d4 acc[NP][NT];
  gr_build<NT, NP>(sh, acc, m, nslot, col, lr);
  gr_eliminate<NT, NP, false>(sh, acc, m, wave, lane);
  double* dsc = ws + (int64_t)w * L.per_walker + pick2(L.off_det, sp);
  if constexpr (!VAL) {
    // F_b(k, j): row p_k of part b over piv_k; the diagonal also goes to the
    // per-orbital terms (real and imaginary parts)
    double* Fd = dsc + DS_N + 2 * s.nptot + 3 * m;
    double* Fg = Fbuf + (int64_t)w * L.f_per_walker + pick2(L.f_off, sp);
    const int j = col;
    if (j < m) {
#pragma unroll
      for (int T = 0; T < NT; T++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const int r = 16 * T + lr + 4 * v;
          const int k = sh.rank[r];
          if (k >= 0) {
            const double pi = sh.pinv[r];
#pragma unroll
            for (int b = 0; b < 2; b++) {
              const double f = acc[1 + b][T][v] * pi;
              if (!s.plain) Fg[(b * m + k) * m + j] = f;
              if (k == j) {
                Fd[4 * j + 2 * b] = f;
                Fd[4 * j + 2 * b + 1] = 0.0;
              }
            }
          }
        }
    }
  }
  if (wave == 0) {
    const bool piv = lane < 16 * NT && sh.rank[lane < 16 * NT ? lane : 0] >= 0;
    const double t = wave_sum(piv ? log(sh.pabs[lane]) : 0.0);
    if (lane == 0) {
      dsc[DS_LOGDET] = t + (nslot - zero) * 0.6931471805599453;
      dsc[DS_SING] = sh.sing ? 1.0 : 0.0;
    }
  }
}

// A^-1 of single-electron moves (row = particle, column = orbital, complex)
// for real orbitals: R^-1 by the in-place elimination, R^-1(k, p_c) = M(p_k, c)
// / piv_k, brought into row order in LDS, where the two rows of a pair meet:
// A^-1(k, +-g) = (X_cos -+ i X_sin) / 2.  Bound by the pivot chains and the
// complex store (0.98 GB for 4096 walkers of N=122).
template <int NT>
struct GrInverse {
  static constexpr int LD = 16 * NT + 1;
  GrShared<NT, 1> sh;
  double X[16 * NT * LD];  // X(k, r) at k LD + r
  int pcol[16 * NT];       // pivot row of column c
};

template <int NT>
__global__ __launch_bounds__(64 * NT, 4) void k_gjr_inverse(DevSys s, int sp0, const double* __restrict__ x,
                                                            double2* __restrict__ ainv, int mm) {
  extern __shared__ __attribute__((aligned(16))) unsigned char gi_lds[];
  GrInverse<NT>& gi = *reinterpret_cast<GrInverse<NT>*>(gi_lds);
  GrShared<NT, 1>& sh = gi.sh;
  const int w = blockIdx.x, sp = sp0 + blockIdx.y;
  const int m = pick2(s.np, sp);
  if (m == 0) return;
  const int nslot = pick2(s.nslot, sp), zero = pick2(s.zslot, sp);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane >> 4, col = 16 * wave + (lane & 15);
  gr_setup(sh, x + ((int64_t)w * s.nptot + pick2(s.ipf, sp)) * 2, sp ? s.gpair[1] : s.gpair[0], m, nslot, zero, tid);
  gr_d4 acc[1][NT];
  gr_build<NT, 1>(sh, acc, m, nslot, col, lr);
  gr_eliminate<NT, 1, true>(sh, acc, m, wave, lane);
  for (int r = tid; r < 16 * NT; r += 64 * NT)
    if (sh.rank[r] >= 0) gi.pcol[sh.rank[r]] = r;
  block_sync();
  if (col < m) {
    const int pc = gi.pcol[col];
#pragma unroll
    for (int T = 0; T < NT; T++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int r = 16 * T + lr + 4 * v;
        const int k = sh.rank[r];
        if (k >= 0) gi.X[k * GrInverse<NT>::LD + pc] = acc[0][T][v] * sh.pinv[r];
      }
  }
  block_sync();
  double2* out = ainv + ((int64_t)w * 2 + sp) * mm * mm;
  const int2* kpm = sp ? s.kpm[1] : s.kpm[0];
  for (int e = tid; e < m * nslot; e += 64 * NT) {
    const int k = e / nslot, sl = e - k * nslot;
    const int r = (sl >> 3) * 16 + ((sl >> 2) & 1) * 8 + (sl & 3);
    const double xc = gi.X[k * GrInverse<NT>::LD + r];
    const int2 o = kpm[sl];
    if (zero && sl == 0) {
      out[k * mm + o.x] = make_double2(xc, 0.0);
    } else {
      const double hc = 0.5 * xc, hs = 0.5 * gi.X[k * GrInverse<NT>::LD + r + 4];
      out[k * mm + o.x] = make_double2(hc, -hs);
      out[k * mm + o.y] = make_double2(hc, hs);
    }
  }
}

template <bool VAL>
static void gjr_spins(const DevSys& s, const WsLayout& L, int nw, int sp0, int nsp, int nt, double* ws, double* F,
                      hipStream_t st) {
  const dim3 grid(nw, nsp);
  switch (nt) {
    case 1: hipLaunchKernelGGL((k_gjr<1, VAL>), grid, dim3(64), 0, st, s, L, ws, F, sp0); break;
    case 2: hipLaunchKernelGGL((k_gjr<2, VAL>), grid, dim3(128), 0, st, s, L, ws, F, sp0); break;
    case 3: hipLaunchKernelGGL((k_gjr<3, VAL>), grid, dim3(192), 0, st, s, L, ws, F, sp0); break;
    default: hipLaunchKernelGGL((k_gjr<4, VAL>), grid, dim3(256), 0, st, s, L, ws, F, sp0); break;
  }
}

// go(first spin, spins, tile count) for every launch of a real-orbital kernel:
// one when the spins have the same tile count, else one per spin.  A spin of m
// particles has m or, with the zero plane wave (m odd), m + 1 rows.
template <class G>
static void gjr_launches(const DevSys& s, G&& go) {
  int nt[2] = {0, 0};
  for (int sp = 0; sp < s.ntypes; sp++) nt[sp] = s.np[sp] ? (2 * s.nslot[sp] + 15) / 16 : 0;
  if (s.ntypes == 2 && nt[0] == nt[1]) {
    if (nt[0]) go(0, 2, nt[0]);
    return;
  }
  for (int sp = 0; sp < s.ntypes; sp++)
    if (nt[sp]) go(sp, 1, nt[sp]);
}

void launch_gjr(const DevSys& s, const WsLayout& L, int nw, bool value, double* ws, double* F, hipStream_t st) {
  gjr_launches(s, [&](int sp0, int nsp, int nt) {
    if (value) gjr_spins<true>(s, L, nw, sp0, nsp, nt, ws, F, st);
    else gjr_spins<false>(s, L, nw, sp0, nsp, nt, ws, F, st);
  });
}

void launch_gjr_inverse(const DevSys& s, int nw, const double* x, void* ainv, int mm, hipStream_t st) {
  double2* a = (double2*)ainv;
  gjr_launches(s, [&](int sp0, int nsp, int nt) {
    const dim3 grid(nw, nsp);
    switch (nt) {
      case 1: hipLaunchKernelGGL(k_gjr_inverse<1>, grid, dim3(64), sizeof(GrInverse<1>), st, s, sp0, x, a, mm); break;
      case 2: hipLaunchKernelGGL(k_gjr_inverse<2>, grid, dim3(128), sizeof(GrInverse<2>), st, s, sp0, x, a, mm); break;
      case 3: hipLaunchKernelGGL(k_gjr_inverse<3>, grid, dim3(192), sizeof(GrInverse<3>), st, s, sp0, x, a, mm); break;
      default: hipLaunchKernelGGL(k_gjr_inverse<4>, grid, dim3(256), sizeof(GrInverse<4>), st, s, sp0, x, a, mm); break;
    }
  });
}
