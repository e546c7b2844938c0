// qmc_fgrad.hip -- drift and first-derivative Laplacian terms of the backflow
// determinants for up to 64 particles per spin (reptation.f:10195-10240; the
// second-derivative terms are k_cross's).
//
// The per-orbital factors d_j = F_b(j,j) come from the determinant kernel
// (stored beside the determinant scalars); this kernel adds the backflow
// Jacobian, regenerated from the eta table, over the pairs.
//
// One workgroup per walker, every pair once on the schedule of qmc_pairs.h.
// With mb the pair's Jacobian block (even in the pair), u = x_i - x_j and
// cc = eta'' + 3 eta'/r, a pair adds
//   mb to the backflow blocks Q of i and of j,
//   -d_i mb to the drift terms z of j and -d_j mb to those of i,
//   cc (d_i - d_j).u to the Laplacian terms of i's and of j's type: both ends
//   take their own determinant's second Jacobian derivative and the partner's,
// and each particle d (1 + Q) to its own drift terms.  A determinant couples to
// the types it has backflow with (iub_flag).  Real orbitals have real d; with
// complex ones the imaginary parts of z, whose squares are the fixed-phase term,
// are kept per determinant.  A lane keeps its own particle's sums in registers
// while the wavefront's run stays in its block; the partner's go to the lane
// group's partial sums in LDS, added in a fixed order at the end.
//
// What bounds it: the chain of a step, as k_pairs.  One block per (walker,
// spin) on blocks of 64 lanes, with the pairs across the types twice and
// Laplacian sums per particle, took 185 us at N=122, 4096 walkers (now 124), 24
// us at N=58, 512 walkers (now 10), 14 us for one walker of N=26 twisted (now
// 7).
#include "qmc_internal.h"
#include "qmc_pairs.h"

// Per-particle sums: Q11, Q12, Q22, Re z; with complex orbitals Im z of the two
// determinants too.  ONE: particles of one type alone (half the sums' rows, one
// determinant: 21 us for 1024 walkers of 61 twisted polarized particles, 24 in
// the general form, whose LDS holds two blocks per CU).
template <bool REAL, bool ONE, int P>
struct FgShape {
  using S = PairShape<false, P>;
  static constexpr int NS = ONE ? P : 2 * P;
  static constexpr int NQ = REAL ? 5 : ONE ? 7 : 9, PART = NQ * NS;
  static size_t lds(int N) { return sizeof(double) * ((REAL ? 4 : 6) * (size_t)N + (size_t)S::NA * PART); }
};

// Whether determinant sp has backflow with type t.
__device__ __forceinline__ bool fg_on(const DevSys& s, int sp, int t) {
  return (sp ? pick2(s.iub_flag[1], t) : pick2(s.iub_flag[0], t)) != 0;
}

// LDS: xs[2N], Re d[2N] (x, y per particle), Im d[2N] (complex), the partial sums.
template <bool REAL, bool ONE, int P>
__global__ __launch_bounds__((PairShape<false, P>::T), 4) void k_fgrad(DevSys s, WsLayout L,
                                                                       const double* __restrict__ x,
                                                                       double* __restrict__ ws) {
  using S = PairShape<false, P>;
  using G = FgShape<REAL, ONE, P>;
  constexpr int NQ = G::NQ, NS = G::NS;
  extern __shared__ __attribute__((aligned(16))) double sm[];
  __shared__ double red[S::NW][3];
  const int w = blockIdx.x;
  if (s.nact && w >= *s.nact) return;
  const int N = s.nptot, tid = threadIdx.x, l = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  double* wsw = ws + (int64_t)w * L.per_walker;
  double* ds[2];
  bool sing = false;
#pragma unroll
  for (int sp = 0; sp < 2; sp++) {
    ds[sp] = wsw + L.off_det[sp];
    if (sp < s.ntypes && s.np[sp] > 0) sing = sing || ds[sp][DS_SING] != 0.0;
  }
  if (sing) return;
  double* xs = sm;
  double* dr = sm + 2 * N;
  double* di = REAL ? nullptr : sm + 4 * N;
  double* parts = sm + (REAL ? 4 : 6) * N;
  const int lp = l & (P - 1);
  double* part = parts + (wv * S::SUB + l / P) * G::PART;
  const double* xw = x + (int64_t)w * 2 * N;
  for (int k = tid; k < 2 * N; k += S::T) xs[k] = xw[k];
  for (int p = tid; p < N; p += S::T) {
    const int t = ptype(s, p);
    const double* Fd = (t ? ds[1] : ds[0]) + DS_N + 2 * N + 3 * pick2(s.np, t) + 4 * (p - pick2(s.ipf, t));
    dr[2 * p] = Fd[0];
    dr[2 * p + 1] = Fd[2];
    if (!REAL) {
      di[2 * p] = Fd[1];
      di[2 * p + 1] = Fd[3];
    }
  }
  for (int k = tid; k < S::NA * G::PART; k += S::T) parts[k] = 0.0;
  block_sync();
  bool all = true;
#pragma unroll
  for (int e = 0; e < 4; e++)
    if ((e >> 1) < s.ntypes && (e & 1) < s.ntypes && s.np[e >> 1] > 0 && s.np[e & 1] > 0)
      all = all && s.iub_flag[e >> 1][e & 1] != 0;
  double ia[NQ] = {}, hi = 0.0, hj = 0.0, h0 = 0.0, h1 = 0.0;
  // ALL: every determinant couples to every type
  auto run = [&](auto allc) {
    constexpr bool ALL = decltype(allc)::value;
    pair_run<S, P>(
        s, wv, l,
        [&](TpPtr T, int tp, int i, int j) {
          const TabRef tb{T->row[TK_B], T->ng[TK_B]};
          if (tb.row0 < 0) return;
          const int ti = tp == 2, tj = tp >= 1;
          const double2 xi2 = ld2(xs, i), xj2 = ld2(xs, j);
          const PairGeo p = pair_geo(s, xi2.x, xi2.y, xj2.x, xj2.y);
          double eta, deta, ddeta;
          spline3(s, tb, p.ind, p.rem, eta, deta, ddeta);
          const double cb = deta * p.byr;
          const double m11 = eta + cb * p.ux * p.ux, m12 = cb * p.ux * p.uy, m22 = eta + cb * p.uy * p.uy;
          const double cc = ddeta + 3.0 * cb;
          const double2 a = ld2(dr, i), b = ld2(dr, j);
          const double ca = cc * (a.x * p.ux + a.y * p.uy), cd = cc * (b.x * p.ux + b.y * p.uy);
          const bool aj = ALL || fg_on(s, ti, tj), bi = ALL || fg_on(s, tj, ti);
          hi -= ALL ? ca - cd : (fg_on(s, ti, ti) ? ca : 0.0) - (bi ? cd : 0.0);
          hj -= ALL ? ca - cd : (aj ? ca : 0.0) - (fg_on(s, tj, tj) ? cd : 0.0);
          ia[0] += m11;
          ia[1] += m12;
          ia[2] += m22;
          double* pj = part + j;
          pj[0] += m11;
          pj[NS] += m12;
          pj[2 * NS] += m22;
          if (bi) {
            ia[3] -= b.x * m11 + b.y * m12;
            ia[4] -= b.x * m12 + b.y * m22;
          }
          if (aj) {
            pj[3 * NS] -= a.x * m11 + a.y * m12;
            pj[4 * NS] -= a.x * m12 + a.y * m22;
          }
          if constexpr (!REAL) {
            const double2 ai = ld2(di, i), bj = ld2(di, j);
            if (bi) {
              const double zx = bj.x * m11 + bj.y * m12, zy = bj.x * m12 + bj.y * m22;
              ia[5] -= ONE || tj == 0 ? zx : 0.0;
              ia[6] -= ONE || tj == 0 ? zy : 0.0;
              if constexpr (!ONE) {
                ia[7] -= tj == 0 ? 0.0 : zx;
                ia[8] -= tj == 0 ? 0.0 : zy;
              }
            }
            if (aj) {
              double* pz = pj + (ONE || ti == 0 ? 5 : 7) * NS;
              pz[0] -= ai.x * m11 + ai.y * m12;
              pz[NS] -= ai.x * m12 + ai.y * m22;
            }
          }
        },
        [&](int ti, int tj) {
          h0 += (ti == 0 ? hi : 0.0) + (tj == 0 ? hj : 0.0);
          h1 += (ti == 0 ? 0.0 : hi) + (tj == 0 ? 0.0 : hj);
          hi = hj = 0.0;
        },
        [&](int ti) {
          if (lp < pick2(s.np, ti)) {
            double* pi = part + pick2(s.ipf, ti) + lp;
#pragma unroll
            for (int q = 0; q < NQ; q++) pi[q * NS] += ia[q];
          }
#pragma unroll
          for (int q = 0; q < NQ; q++) ia[q] = 0.0;
        });
  };
  if (all) run(std::true_type{});
  else run(std::false_type{});
  block_sync();
  // the groups' partial sums in order, then each particle's own block
  double g2 = 0.0;
  for (int e = tid; e < NQ * NS; e += S::T) {
    double v = parts[e];
#pragma unroll
    for (int a = 1; a < S::NA; a++) v += parts[a * G::PART + e];
    parts[e] = v;
  }
  block_sync();
  if (tid < N) {
    const int p = tid, t = ptype(s, p);
    double v[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) v[q] = parts[q * NS + p];
    const double a11 = 1.0 + v[0], a12 = v[1], a22 = 1.0 + v[2];
    if (fg_on(s, t, t)) {
      const double2 a = ld2(dr, p);
      v[3] += a.x * a11 + a.y * a12;
      v[4] += a.x * a12 + a.y * a22;
      if constexpr (!REAL) {
        const double2 b = ld2(di, p);
        const double zx = b.x * a11 + b.y * a12, zy = b.x * a12 + b.y * a22;
        v[5] += ONE || t == 0 ? zx : 0.0;
        v[6] += ONE || t == 0 ? zy : 0.0;
        if constexpr (!ONE) {
          v[7] += t == 0 ? 0.0 : zx;
          v[8] += t == 0 ? 0.0 : zy;
        }
      }
    }
    double* own = t ? ds[1] : ds[0];
    double* Qd = own + DS_N + 2 * N + 3 * (p - pick2(s.ipf, t));
    Qd[0] = v[0];
    Qd[1] = v[1];
    Qd[2] = v[2];
    // both determinants' drift in the place of the particle's own spin's
    own[DS_N + 2 * p] = -v[3];
    own[DS_N + 2 * p + 1] = -v[4];
    if (s.ntypes > 1) {
      double* oth = t ? ds[0] : ds[1];
      oth[DS_N + 2 * p] = 0.0;
      oth[DS_N + 2 * p + 1] = 0.0;
    }
    if constexpr (!REAL) {
#pragma unroll
      for (int q = 5; q < NQ; q++) g2 += v[q] * v[q];
      g2 *= pick2(s.hbs2m, t);
    }
  }
  {
    const double v[3] = {wave_sum(h0), wave_sum(h1), REAL ? 0.0 : wave_sum(g2)};
    if (l == 0) {
#pragma unroll
      for (int q = 0; q < 3; q++) red[wv][q] = v[q];
    }
  }
  block_sync();
  if (tid == 0) {
    double v[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int a = 0; a < S::NW; a++)
#pragma unroll
      for (int q = 0; q < 3; q++) v[q] += red[a][q];
    // the walker's sums with the first spin that has particles
    const int sp = s.np[0] > 0 ? 0 : 1;
#pragma unroll
    for (int t = 0; t < 2; t++) {
      if (t >= s.ntypes || s.np[t] == 0) continue;
      ds[t][DS_H0] = t == sp ? v[0] : 0.0;
      ds[t][DS_H1] = t == sp ? v[1] : 0.0;
      ds[t][DS_G2] = t == sp ? v[2] : 0.0;
    }
  }
}

void launch_fgrad(const DevSys& s, const WsLayout& L, int nw, const double* x, double* ws, hipStream_t st) {
  with_lanes(s, [&](auto p) {
    constexpr int P = decltype(p)::value, T = PairShape<false, P>::T;
    auto go = [&](auto real, auto one) {
      constexpr bool R = decltype(real)::value, O = decltype(one)::value;
      hipLaunchKernelGGL((k_fgrad<R, O, P>), dim3(nw), dim3(T), (FgShape<R, O, P>::lds(s.nptot)), st, s, L, x, ws);
    };
    const bool one = pair_one(s);
    if (s.real_orb && one) go(std::true_type{}, std::true_type{});
    else if (s.real_orb) go(std::true_type{}, std::false_type{});
    else if (one) go(std::false_type{}, std::true_type{});
    else go(std::false_type{}, std::false_type{});
  });
}
