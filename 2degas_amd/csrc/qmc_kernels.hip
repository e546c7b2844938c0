// qmc_kernels.hip -- FP64 walker-evaluation kernels for gfx950.
//
// One local-energy evaluation (compute_properties(1), reptation.f:2661-2727)
// of a batch of walkers is five launches: k_pairs, k_gjr or k_gjc (qmc_gjr.hip,
// qmc_gjc.hip: the determinant on the matrix cores, of real or complex
// orbitals), k_fgrad (qmc_fgrad.hip), k_cross and k_final; without backflow the
// two before k_final are left out; with QMC_NO_GJ set, k_det takes the part of
// the determinant kernel and k_fgrad:
//   k_pairs   one workgroup per walker: pair geometry, u2 and u3 Jastrow
//             (two_body/three_body/dotg, reptation.f:2777-3046), backflow
//             quasi-coordinates (reptation.f:10023-10058), real-space Ewald
//             (reptation.f:3994-4033), rho_k and k-space Ewald
//             (reptation.f:4224-4243, 4034-4052).
//   k_det     one workgroup per (walker, spin): plane-wave orbital matrix of
//             the quasi-coordinates, LU with LINPACK pivoting and inverse in
//             LDS (zgefa/zgedi, reptation.f:9227-9472), F = A^-1 dA, drift
//             and the diagonal Laplacian terms (reptation.f:10159-10240).
//   k_cross   (qmc_cross.hip) one workgroup per (walker, spin): the backflow
//             Laplacian cross term sum_ip tr(C_ip^2) (reptation.f:10241-10259)
//             as a symmetric contraction of S = V V^T against M = Re(F o F^T).
//   k_final   kinetic and potential energies and the property slots
//             (kinetic, reptation.f:2729-2775; potential tail, 4088-4096).
#include <algorithm>
#include <type_traits>
#include <utility>

#include "qmc_internal.h"
#include "qmc_pairs.h"

// k-vectors per thread and pass in k_pairs
#define KMAXPT 4
#define KRUN 9  // phases of one particle built from one sin/cos pair (odd: lanes' runs start in different LDS banks)

// ---------------------------------------------------------------------------
// k_pairs
// LDS: xs[2N], Gs[2N], red[8 NW], then a region shared by the partial sums of
// the pair passes (NA x 6 x NS doubles) and, afterwards, the phase steps (4N) and
// phases of rho_k.
//
// The pair passes run on the schedule of qmc_pairs.h.
//
// What bounds it: a step is a chain of some 1500 cycles (geometry, table
// loads, spline, LDS sums), so short runs count where few walkers are in
// flight, and occupancy where many are.  8 wavefronts against 4 (200 shells of
// k-vectors): N=58, 1 walker 26 against 38 us, 256 walkers 30 against 40, 1024
// walkers 70 against 66, 8192 walkers 428 against 391; N=122, 4096 walkers 500
// against 528 (16 wavefronts: 701).  The count depends on the deck alone, not on
// the batch, so that a walker's result does not depend on the batch it is in;
// between the two ends it favours the small batch, which a served job's steps
// and a reptation move evaluate and where the kernel is the longest of the call
// (10 of 73 us at N=58, 256 walkers, against 37 of 876 at 8192).  The mixed
// kernel's FP32 phases need more registers, and 4 wavefronts are the better count
// at both ends (N=122 413 against 554 us, N=58 at 8192 walkers 276 against 445).
#define PP_NQ 6  // per-particle sums of a pass

// part[q * NS + p] += v for the lane group's partial sums
template <int NS>
__device__ __forceinline__ void pp_add(double* part, int p, const double (&v)[PP_NQ], int nq) {
#pragma unroll
  for (int q = 0; q < PP_NQ; q++)
    if (q < nq) part[q * NS + p] += v[q];
}

// The NA partial sums of each of the nq per-particle sums, added in order
// into the first one.
template <class S>
__device__ __forceinline__ void pp_reduce(double* parts, int nq, int tid) {
  block_sync();
  for (int e = tid; e < nq * S::NS; e += S::T) {
    double v = parts[e];
#pragma unroll
    for (int a = 1; a < S::NA; a++) v += parts[a * S::PART + e];
    parts[e] = v;
  }
  block_sync();
}

// Ewald sums over the k-vectors that carry coefficients, from the rho_k of a
// k-vector: ordered type pairs (0,0), (0,1), (1,0), (1,1) (reptation.f:4034-4052).
__device__ __forceinline__ void kspace_terms(const DevSys& s, int k, double c0, double s0, double c1, double s1,
                                             double& pk0, double& pk1, double& pkt) {
  if (k < s.nke[0]) {
    const double aux = s.vk[0][k] * (c0 * c0 + s0 * s0);
    pk0 += aux;
    pkt += aux;
  }
  if (s.ntypes > 1) {
    if (k < s.nke[1]) {
      const double aux = s.vk[1][k] * (c0 * c1 + s0 * s1);
      pk0 += aux;
      pk1 += aux;
      pkt += 2.0 * aux;
    }
    if (k < s.nke[2]) {
      const double aux = s.vk[2][k] * (c1 * c1 + s1 * s1);
      pk1 += aux;
      pkt += aux;
    }
  }
}

// rho_k in FP64 on the matrix cores, for k-vectors over few distinct |kx| and
// |ky|: with C_a, S_a = cos, sin(|kx|_a x_i) and likewise in y, the four
// products CC, CS, SC, SS over a type's particles hold every sign combination
// of (kx, ky) at once:
//   rho = sum_i e^{i k.r_i} = (CC - sx sy SS) + i (sx SC + sy CS).
// A task is one 16 x 16 tile of (a, b) of one type, 4 accumulators on one
// wavefront; the phases of kchunk particles of each type at a time go to LDS
// (row = particle: C_a, S_a, C_b, S_b), an operand being one 8-byte read a
// lane.  A type without particles has no rows and no tasks (it had: k_pairs of 61
// polarized particles, 4096 walkers, 225 us, now 200).  On vector units, one product per k-vector, the same sums read three
// 16-byte phases from LDS for each pair of k-vectors and particle and took
// twice as many operations (both signs of ky separately).
#define KRUN2 5  // phases of one particle from one sin/cos and the step's products
typedef double pk_d4 __attribute__((ext_vector_type(4)));

template <class S>
__device__ __forceinline__ void rho_tiles(const DevSys& s, const double* __restrict__ xs, double* __restrict__ ks,
                                          double* __restrict__ ph, double* __restrict__ pw, int tid) {
  const int N = s.nptot, lane = tid & 63, lr = lane >> 4, lc = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int na = s.nkax, nb = s.nkby, ta = (na + 15) >> 4, tb = (nb + 15) >> 4;
  const int ox = 16 * ta, oy = 32 * ta, ld = 32 * (ta + tb) + 16;
  // the types that have particles: both, or t1 alone
  constexpr int nt = S::ONE ? 1 : 2;
  const int t1 = S::ONE && s.ntypes > 1 && s.np[0] == 0 ? 1 : 0, ntask = ta * tb * nt;
  const int kc = (s.kchunk + 3) & ~3;  // rows per type and chunk
  const int nmax = S::ONE ? pick2(s.np, t1) : max(s.np[0], s.np[1]);
  // items of a phase row: runs of KRUN2 phases; the thread's first item
  const int gx = (na + KRUN2 - 1) / KRUN2, ng = gx + (nb + KRUN2 - 1) / KRUN2;
  const int row_0 = tid / ng, g_0 = tid - row_0 * ng, row_d = S::T / ng, g_d = S::T - row_d * ng;
  // e^{i dk x}, e^{i dk y} of every particle
  if (s.kaprog)
    for (int e = tid; e < 2 * N; e += S::T) {
      double sv, cv;
      qsincos_sreg(((e & 1) ? s.dkby : s.dkax) * xs[e], &sv, &cv);
      ks[2 * e] = cv;
      ks[2 * e + 1] = sv;
    }
  for (int t0 = 0; t0 < ntask; t0 += S::NW) {
    const int task = t0 + wv;
    const bool on = task < ntask;
    const int row_t = on && nt > 1 ? task / (ta * tb) : 0, tile = on ? task - row_t * ta * tb : 0;
    const int type = S::ONE ? t1 : row_t;
    const int ra = 16 * (tile / tb), rb = 16 * (tile % tb);
    pk_d4 cc{0, 0, 0, 0}, cs{0, 0, 0, 0}, sc{0, 0, 0, 0}, ss{0, 0, 0, 0};
    for (int c0 = 0; c0 < nmax; c0 += kc) {
      block_sync();
      // rows: type t's particles c0..c0+kc-1 (zero beyond its count, up to a
      // multiple of 4)
      for (int row = row_0, g = g_0; row < nt * kc; row += row_d, g += g_d) {
        if (g >= ng) {
          g -= ng;
          row++;
          if (row >= nt * kc) break;
        }
        const int r1 = nt > 1 && row >= kc ? 1 : 0, t = S::ONE ? t1 : r1, c = c0 + row - r1 * kc;
        const int np_t = pick2(s.np, t);
        if (c >= ((np_t + 3) & ~3)) continue;
        const bool isx = g < gx, live = c < np_t;
        const int v0 = (isx ? g : g - gx) * KRUN2, n = isx ? na : nb, nrun = min(KRUN2, n - v0);
        double* dst = ph + row * ld + (isx ? 0 : oy) + v0;
        const int od = isx ? ox : 16 * tb;  // from the cosines to the sines
        const int i = pick2(s.ipf, t) + c;
        const double* kv = isx ? s.kax : s.kby;
        const double u = live ? xs[2 * i + (isx ? 0 : 1)] : 0.0;
        double sa = 0.0, ca = 0.0, sd = 0.0, cd = 0.0;
        if (live) {
          qsincos_sreg(kv[v0] * u, &sa, &ca);
          if (s.kaprog) {
            cd = ks[4 * i + (isx ? 0 : 2)];
            sd = ks[4 * i + (isx ? 1 : 3)];
          }
        }
        dst[0] = ca;
        dst[od] = sa;
#pragma unroll
        for (int r = 1; r < KRUN2; r++) {
          if (r < nrun) {
            if (s.kaprog) {
              const double c2 = fma(ca, cd, -sa * sd);
              sa = fma(ca, sd, sa * cd);
              ca = c2;
            } else if (live) {
              qsincos_sreg(kv[v0 + r] * u, &sa, &ca);
            }
            dst[r] = ca;
            dst[od + r] = sa;
          }
        }
      }
      block_sync();
      if (on) {
        const int cn = min(kc, pick2(s.np, type) - c0);
        const double* base = ph + (row_t * kc + lr) * ld + lc;
        for (int k = 0; k < cn; k += 4) {
          const double* row = base + k * ld;
          const double ca = row[ra], sa = row[ox + ra], cb = row[oy + rb], sb = row[oy + 16 * tb + rb];
          cc = __builtin_amdgcn_mfma_f64_16x16x4f64(ca, cb, cc, 0, 0, 0);
          cs = __builtin_amdgcn_mfma_f64_16x16x4f64(ca, sb, cs, 0, 0, 0);
          sc = __builtin_amdgcn_mfma_f64_16x16x4f64(sa, cb, sc, 0, 0, 0);
          ss = __builtin_amdgcn_mfma_f64_16x16x4f64(sa, sb, ss, 0, 0, 0);
        }
      }
    }
    // each (a, b) cell's k-vectors: k * 4 + (kx < 0) * 2 + (ky < 0), -1 none
    const int irk = on ? pick2(s.irhok, type) : 0;
    if (irk) {
      double* out = pw + s.jrhok + (irk - 1) * 2 * s.nk;
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int4 cell = s.kcell[(ra + lr + 4 * v) * 16 * tb + rb + lc];
        const int ent[4] = {cell.x, cell.y, cell.z, cell.w};
#pragma unroll
        for (int q = 0; q < 4; q++) {
          if (ent[q] < 0) continue;
          const bool nx = ent[q] & 2, ny = ent[q] & 1;
          const int k = ent[q] >> 2;
          out[2 * k] = nx != ny ? cc[v] + ss[v] : cc[v] - ss[v];
          out[2 * k + 1] = (nx ? -sc[v] : sc[v]) + (ny ? -cs[v] : cs[v]);
        }
      }
    }
  }
}

// MIX (the mixed-precision evaluation): the u2, u3 and pair-potential
// tables are read from their FP32 copy and evaluated in FP32 (spline3m), and
// the rho_k phases are stored in LDS as FP32 pairs and multiplied and summed
// over each chunk of particles in FP32, the chunk sums added in FP64; the
// pair geometry, the backflow coordinates, every accumulator and the k-space
// sum stay FP64.
template <bool MIX, int P, bool ONE>
__device__ __forceinline__ void k_pairs_body(const DevSys& s, const WsLayout& L,
                                             const double* __restrict__ x,
                                             double* __restrict__ ws,
                                             double* __restrict__ props) {
  using S = PairShape<MIX, P, ONE>;
  extern __shared__ __attribute__((aligned(16))) double sm[];
  const int w = blockIdx.x;
  if (s.nact && w >= *s.nact) return;
  const int N = s.nptot;
  double* xs = sm;
  double* Gs = sm + 2 * N;
  double* red = sm + 4 * N;
  double* parts = sm + 4 * N + 8 * S::NW;
  const double* xw = x + (int64_t)w * 2 * N;
  const int tid = threadIdx.x, l = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  double* part = parts + (wv * S::SUB + l / P) * S::PART;
  const int lp = l & (P - 1);
  for (int k = tid; k < 2 * N; k += S::T) xs[k] = xw[k];
  for (int k = tid; k < S::NA * S::PART; k += S::T) parts[k] = 0.0;
  block_sync();
  double* wsw = ws + (int64_t)w * L.per_walker;
  double acc_ltf = 0.0, acc_h0 = 0.0, acc_h1 = 0.0, acc_v0 = 0.0, acc_v1 = 0.0;

  // pass 1: u2, the pair term and G of u3, backflow q, pair potential
  {
    double ia[PP_NQ] = {0, 0, 0, 0, 0, 0};  // gx, gy, Gx, Gy, qx, qy of particle i
    double hb = 0.0, vb = 0.0;              // the block pair's Laplacian and potential
    pair_run<S, P>(
        s, wv, l,
        [&](TpPtr T, int, int i, int j) {
          const TabRef tu2{T->row[TK_U2], T->ng[TK_U2]}, tu3{T->row[TK_U3], T->ng[TK_U3]},
              tb{T->row[TK_B], T->ng[TK_B]}, tv{T->row[TK_V], T->ng[TK_V]};
          const double2 xi2 = ld2(xs, i), xj2 = ld2(xs, j);
          PairGeo p = pair_geo(s, xi2.x, xi2.y, xj2.x, xj2.y);
          double ja[PP_NQ] = {0, 0, 0, 0, 0, 0};
          double hh = 0.0;
          double f, df, ddf;
          if (tu2.row0 >= 0) {
            spline3m<MIX>(s, tu2, p.ind, p.rem, f, df, ddf);
            acc_ltf += f;
            const double dtr = df * p.byr;
            ja[0] -= dtr * p.ux;
            ja[1] -= dtr * p.uy;
            hh += ddf + dtr;
          }
          if (tu3.row0 >= 0) {
            spline3m<MIX>(s, tu3, p.ind, p.rem, f, df, ddf);
            ja[2] += f * p.ux;
            ja[3] += f * p.uy;
            // (xi r)^2 pair term of the three-body factor (reptation.f:2822-2832)
            const double r = p.r;
            const double tr = f * r;
            const double d3 = 2.0 * f * (f + r * df);
            const double dd3 = 2.0 * (f * f + 4.0 * r * f * df + r * r * (df * df + ddf * f));
            acc_ltf += tr * tr;
            ja[0] -= d3 * p.ux;
            ja[1] -= d3 * p.uy;
            hh += dd3 + d3;
          }
          if (tb.row0 >= 0) {
            spline3(s, tb, p.ind, p.rem, f, df, ddf);
            ja[4] -= f * p.ux;
            ja[5] -= f * p.uy;
          }
          // the pair gives i the opposite of j's vector terms (u -> -u)
#pragma unroll
          for (int q = 0; q < PP_NQ; q++) ia[q] -= ja[q];
          hb += hh;
          if (tv.row0 >= 0) vb += 0.5 * spline0<MIX>(s, tv, T->vexp, p.ind, p.rem, p.byr) * T->v2value;
          pp_add<S::NS>(part, j, ja, PP_NQ);
        },
        [&](int ti, int tj) {
          // (selected, not subtracted: what is infinite or no number in one
          // type's pairs stays out of the other's sums)
          acc_h0 += (ti == 0 ? hb : 0.0) + (tj == 0 ? hb : 0.0);
          acc_h1 += (ti == 0 ? 0.0 : hb) + (tj == 0 ? 0.0 : hb);
          acc_v0 += (ti == 0 ? vb : 0.0) + (tj == 0 ? vb : 0.0);
          acc_v1 += (ti == 0 ? 0.0 : vb) + (tj == 0 ? 0.0 : vb);
          hb = vb = 0.0;
        },
        [&](int ti) {
          if (lp < pick2(s.np, ti)) pp_add<S::NS>(part, pick2(s.ipf, ti) + lp, ia, PP_NQ);
#pragma unroll
          for (int q = 0; q < PP_NQ; q++) ia[q] = 0.0;
        });
  }
  pp_reduce<S>(parts, PP_NQ, tid);
  // Gs for pass 2, q out, g kept
  double gpx = 0.0, gpy = 0.0;  // gradient of particle tid (N <= 128)
  if (tid < N) {
    const int p = tid;
    double v[PP_NQ];
#pragma unroll
    for (int q = 0; q < PP_NQ; q++) v[q] = parts[q * S::NS + p];
    gpx = v[0];
    gpy = v[1];
    Gs[2 * p] = v[2];
    Gs[2 * p + 1] = v[3];
    wsw[L.off_q + 2 * p] = xs[2 * p] + v[4];
    wsw[L.off_q + 2 * p + 1] = xs[2 * p + 1] + v[5];
    acc_ltf -= 0.5 * (v[2] * v[2] + v[3] * v[3]);
  }
  block_sync();

  // pass 2: three-body contraction (dotg, reptation.f:2928-2979), written per
  // particle i as g_i += sum_k M_ik (G_i - G_k),
  // h_i += -|sum_k M_ik|^2 - sum_k |M_ik|^2 + sum_k a_ik u_ik.(G_i - G_k)
  // with M = xi I + (xi'/r) u u^T and a = xi'' + 3 xi'/r; M and a.(u dG) are
  // even in the pair, M dG is odd
  if (s.has_u3) {
    for (int k = tid; k < S::NA * S::PART; k += S::T) parts[k] = 0.0;
    block_sync();
    double ia[PP_NQ] = {0, 0, 0, 0, 0, 0};  // g3x, g3y, e11, e12, e22 of particle i
    double hb = 0.0;
    pair_run<S, P>(
        s, wv, l,
        [&](TpPtr T, int, int i, int j) {
          const TabRef tu3{T->row[TK_U3], T->ng[TK_U3]};
          if (tu3.row0 < 0) return;
          const double2 xi2 = ld2(xs, i), xj2 = ld2(xs, j);
          PairGeo p = pair_geo(s, xi2.x, xi2.y, xj2.x, xj2.y);
          double t, dt, ddt;
          spline3m<MIX>(s, tu3, p.ind, p.rem, t, dt, ddt);
          const double c = dt * p.byr;
          const double m11 = t + c * p.ux * p.ux, m12 = c * p.ux * p.uy, m22 = t + c * p.uy * p.uy;
          const double2 Gi = ld2(Gs, i), Gj = ld2(Gs, j);
          const double dGx = Gi.x - Gj.x, dGy = Gi.y - Gj.y;
          const double g3x = m11 * dGx + m12 * dGy, g3y = m12 * dGx + m22 * dGy;
          const double nm2 = m11 * m11 + 2.0 * m12 * m12 + m22 * m22;
          const double h3 = (ddt + 3.0 * c) * (p.ux * dGx + p.uy * dGy) - nm2;
          ia[0] += g3x;
          ia[1] += g3y;
          ia[2] += m11;
          ia[3] += m12;
          ia[4] += m22;
          const double ja[PP_NQ] = {-g3x, -g3y, m11, m12, m22, 0.0};
          pp_add<S::NS>(part, j, ja, 5);
          hb += h3;
        },
        [&](int ti, int tj) {
          acc_h0 += (ti == 0 ? hb : 0.0) + (tj == 0 ? hb : 0.0);
          acc_h1 += (ti == 0 ? 0.0 : hb) + (tj == 0 ? 0.0 : hb);
          hb = 0.0;
        },
        [&](int ti) {
          if (lp < pick2(s.np, ti)) pp_add<S::NS>(part, pick2(s.ipf, ti) + lp, ia, 5);
#pragma unroll
          for (int q = 0; q < PP_NQ; q++) ia[q] = 0.0;
        });
    pp_reduce<S>(parts, 5, tid);
    if (tid < N) {
      double v[5];
#pragma unroll
      for (int q = 0; q < 5; q++) v[q] = parts[q * S::NS + tid];
      gpx += v[0];
      gpy += v[1];
      const double e2 = v[2] * v[2] + 2.0 * v[3] * v[3] + v[4] * v[4];
      if (ptype(s, tid) == 0) acc_h0 -= e2; else acc_h1 -= e2;
    }
  }
  if (tid < N) {
    wsw[L.off_gj + 2 * tid] = gpx;
    wsw[L.off_gj + 2 * tid + 1] = gpy;
  }

  // the pair sums over each wavefront (lane 0 of each has a row of red)
  {
    const double v[5] = {wave_sum(acc_ltf), wave_sum(acc_h0), wave_sum(acc_h1), wave_sum(acc_v0), wave_sum(acc_v1)};
    if (l == 0) {
#pragma unroll
      for (int q = 0; q < 5; q++) red[8 * wv + q] = v[q];
    }
  }

  // rho_k per type and the k-space Ewald sum
  double pk0 = 0.0, pk1 = 0.0, pkt = 0.0;
  double* pw = props + (int64_t)w * s.n_props;
  if (!MIX && s.nrhok && s.nkax > 0) {
    block_sync();  // Gs and the partial sums have been read
    rho_tiles<S>(s, xs, parts, parts + 4 * N, pw, tid);
    block_sync();  // rho_k of this walker is in memory
    double* r0 = s.irhok[0] ? pw + s.jrhok + (s.irhok[0] - 1) * 2 * s.nk : nullptr;
    double* r1 = s.ntypes > 1 && s.irhok[1] ? pw + s.jrhok + (s.irhok[1] - 1) * 2 * s.nk : nullptr;
    if constexpr (S::ONE) {
      // rho_k of a type without particles
      double*& none = s.np[0] == 0 ? r0 : r1;
      if (none)
        for (int k = tid; k < 2 * s.nk; k += S::T) none[k] = 0.0;
      none = nullptr;
    }
    for (int k = tid; k < s.nk; k += S::T)
      kspace_terms(s, k, r0 ? r0[2 * k] : 0.0, r0 ? r0[2 * k + 1] : 0.0, r1 ? r1[2 * k] : 0.0,
                   r1 ? r1[2 * k + 1] : 0.0, pk0, pk1, pkt);
  } else if (!MIX && s.nrhok) {
    // k-vectors off the grid: each thread sums its own directly
    for (int k = tid; k < s.nk; k += S::T) {
      const double kx = s.kvec[2 * k], ky = s.kvec[2 * k + 1];
      double rc[2] = {0.0, 0.0}, rs[2] = {0.0, 0.0};
#pragma unroll
      for (int t = 0; t < 2; t++) {
        if (t >= s.ntypes || !s.irhok[t]) continue;
        for (int i = s.ipf[t]; i < s.ipf[t] + s.np[t]; i++) {
          double sv, cv;
          qsincos_sreg(kx * xs[2 * i] + ky * xs[2 * i + 1], &sv, &cv);
          rc[t] += cv;
          rs[t] += sv;
        }
        const int slot = s.jrhok + (s.irhok[t] - 1) * 2 * s.nk + 2 * k;
        pw[slot] = rc[t];
        pw[slot + 1] = rs[t];
      }
      kspace_terms(s, k, rc[0], rs[0], rc[1], rs[1], pk0, pk1, pkt);
    }
  } else if (s.nrhok) {
    // passes of KMAXPT slots per thread: slots q = 2h, 2h+1 of a thread are
    // the two k-vectors of one item, which share their ky component
    const bool items = MIX && s.nkxv > 0;  // else one slot per k-vector
    const int nslot = items ? s.nkslot : s.nk;
    for (int kb = 0; kb < nslot; kb += KMAXPT * S::T) {
      double rc0[KMAXPT], rc1[KMAXPT], rs0[KMAXPT], rs1[KMAXPT];
      int kq[KMAXPT];              // k-vector of slot q (-1: none)
      int ox[KMAXPT], oy[KMAXPT];  // kx and ky phase slots of slot q (0 when none)
#pragma unroll
      for (int q = 0; q < KMAXPT; q++) {
        rc0[q] = rc1[q] = rs0[q] = rs1[q] = 0.0;
        const int n = kb + 2 * (threadIdx.x + (q >> 1) * S::T) + (q & 1);
        const int code = items && n < nslot ? s.kxy[n] : 0;
        kq[q] = n >= nslot ? -1 : (items ? (code >> 16) - 1 : n);
        ox[q] = code & 0xff;
        oy[q] = ((code >> 8) & 0xff) + s.nkxv;
      }
      if (items) {
        // e^{i k.x} = e^{i kx x} e^{i ky y}: per particle chunk, the distinct
        // x and y phases go to LDS, then each thread multiplies its k's pairs
        float2* ph = (float2*)parts;
        const int nv = s.nkxv + s.nkyv;
        for (int c0 = 0; c0 < N; c0 += s.kchunk) {
          const int cn = min(s.kchunk, N - c0);
          block_sync();
          if (s.kprog) {
            // runs of KRUN phases: the first directly, the rest by products
            // with e^{i dk x} (at most KRUN - 1 roundings from a direct value)
            const int gx = (s.nkxv + KRUN - 1) / KRUN, ng = gx + (s.nkyv + KRUN - 1) / KRUN;
            for (int e = threadIdx.x; e < cn * ng; e += S::T) {
              const int pc = e / ng, g = e - pc * ng;
              const int i = c0 + pc;
              const bool isx = g < gx;
              const int v0 = (isx ? g : g - gx) * KRUN, nrun = min(KRUN, (isx ? s.nkxv : s.nkyv) - v0);
              const double u = isx ? xs[2 * i] : xs[2 * i + 1];
              double sa, ca, sd, cd;
              qsincos_sreg((isx ? s.kxv[v0] : s.kyv[v0]) * u, &sa, &ca);
              qsincos_sreg((isx ? s.dkx : s.dky) * u, &sd, &cd);
              float2* dst = ph + pc * nv + (isx ? 0 : s.nkxv) + v0;
              dst[0] = float2{(float)ca, (float)sa};
#pragma unroll
              for (int r = 1; r < KRUN; r++) {
                if (r < nrun) {
                  const double c2 = fma(ca, cd, -sa * sd);
                  sa = fma(ca, sd, sa * cd);
                  ca = c2;
                  dst[r] = float2{(float)ca, (float)sa};
                }
              }
            }
          } else {
            for (int e = threadIdx.x; e < cn * nv; e += S::T) {
              const int pc = e / nv, v = e - pc * nv;
              const int i = c0 + pc;
              const double arg = v < s.nkxv ? s.kxv[v] * xs[2 * i] : s.kyv[v - s.nkxv] * xs[2 * i + 1];
              double sv, cv;
              qsincos_sreg(arg, &sv, &cv);
              ph[e] = float2{(float)cv, (float)sv};
            }
          }
          block_sync();
          // particles of type 0 come first: [0, split) of the chunk, each
          // type a loop of its own
          const int split = s.ntypes > 1 ? min(max(s.ipf[1] - c0, 0), cn) : cn;
          auto accum = [&](int pa, int pb, double (&rc)[KMAXPT], double (&rs)[KMAXPT]) {
            // the chunk's products summed in FP32, the chunk sum added to
            // the FP64 accumulators
            float qc[KMAXPT], qs[KMAXPT];
#pragma unroll
            for (int h = 0; h < KMAXPT; h++) qc[h] = qs[h] = 0.0f;
            for (int pc = pa; pc < pb; pc++) {
              const float2* row = ph + pc * nv;
#pragma unroll
              for (int h = 0; h < KMAXPT; h += 2) {
                // one ky phase for the item's two kx phases
                const float2 b = row[oy[h]], a0 = row[ox[h]], a1 = row[ox[h + 1]];
                qc[h] = fmaf(a0.x, b.x, fmaf(-a0.y, b.y, qc[h]));
                qs[h] = fmaf(a0.x, b.y, fmaf(a0.y, b.x, qs[h]));
                qc[h + 1] = fmaf(a1.x, b.x, fmaf(-a1.y, b.y, qc[h + 1]));
                qs[h + 1] = fmaf(a1.x, b.y, fmaf(a1.y, b.x, qs[h + 1]));
              }
            }
#pragma unroll
            for (int h = 0; h < KMAXPT; h++) {
              rc[h] += (double)qc[h];
              rs[h] += (double)qs[h];
            }
          };
          accum(0, split, rc0, rs0);
          accum(split, cn, rc1, rs1);
        }
      } else {
#pragma unroll
        for (int q = 0; q < KMAXPT; q++) {
          const int k = kq[q];
          if (k < 0) continue;
          const double kx = s.kvec[2 * k], ky = s.kvec[2 * k + 1];
          const int split = s.ntypes > 1 ? s.ipf[1] : N;
          for (int i = 0; i < split; i++) {
            double sv, cv;
            qsincos_sreg(kx * xs[2 * i] + ky * xs[2 * i + 1], &sv, &cv);
            rc0[q] += cv;
            rs0[q] += sv;
          }
          for (int i = split; i < N; i++) {
            double sv, cv;
            qsincos_sreg(kx * xs[2 * i] + ky * xs[2 * i + 1], &sv, &cv);
            rc1[q] += cv;
            rs1[q] += sv;
          }
        }
      }
#pragma unroll
      for (int q = 0; q < KMAXPT; q++) {
        const int k = kq[q];
        if (k < 0) continue;
        if (!s.irhok[0]) rc0[q] = rs0[q] = 0.0;
        if (s.ntypes < 2 || !s.irhok[1]) rc1[q] = rs1[q] = 0.0;
        if (s.irhok[0]) {
          const int slot = s.jrhok + (s.irhok[0] - 1) * 2 * s.nk + 2 * k;
          pw[slot] = rc0[q];
          pw[slot + 1] = rs0[q];
        }
        if (s.ntypes > 1 && s.irhok[1]) {
          const int slot = s.jrhok + (s.irhok[1] - 1) * 2 * s.nk + 2 * k;
          pw[slot] = rc1[q];
          pw[slot + 1] = rs1[q];
        }
        kspace_terms(s, k, rc0[q], rs0[q], rc1[q], rs1[q], pk0, pk1, pkt);
      }
    }
  }

  // the walker's eight sums: over each wavefront, then over the wavefronts
  {
    const double v[3] = {wave_sum(pk0), wave_sum(pk1), wave_sum(pkt)};
    if (l == 0) {
#pragma unroll
      for (int q = 0; q < 3; q++) red[8 * wv + 5 + q] = v[q];
    }
  }
  block_sync();
  if (wv != 0) return;
  // lane q adds sum q of the wavefronts
  double mine = 0.0;
#pragma unroll
  for (int a = 0; a < S::NW; a++) mine += red[8 * a + (l & 7)];
  double v[8];
#pragma unroll
  for (int q = 0; q < 8; q++) v[q] = gj_readlane(mine, q);
  if (l == 0) {
    double c0 = 0.0, c1 = 0.0, ct = 0.0;
    for (int it = 0; it < s.ntypes; it++)
      for (int jt = 0; jt < s.ntypes; jt++) {
        const int tp = tpair(it, jt);
        if (pick3(s.nke, tp) != 0) {
          const double a = pick3(s.vk0, tp) * s.npnorm;
          if (it == 0) c0 += a;
          else c1 += a;
          ct += a;
        }
      }
    double* sc = wsw + L.off_sc;
    sc[SC_LTF] = v[0];
    sc[SC_H0] = v[1];
    sc[SC_H1] = v[2];
    // the pair-potential tail constants are added in k_final (held here
    // through the pair loops, they had taken scalar registers the loops need)
    sc[SC_P0] = v[3] + v[5] + c0;
    sc[SC_P1] = v[4] + v[6] + c1;
    sc[SC_PT] = v[3] + v[4] + v[7] + ct;
  }
}

// (6 and 5 wavefronts per SIMD fit without spilling vector registers: the pair
// sums leave for LDS before the phases, whose loops need the registers)
template <bool MIX, int P, bool ONE>
__global__ __launch_bounds__((PairShape<MIX, P, ONE>::T), MIX ? 5 : 6) void k_pairs(DevSys s, WsLayout L,
                                                                                   const double* __restrict__ x,
                                                                                   double* __restrict__ ws,
                                                                                   double* __restrict__ props) {
  k_pairs_body<MIX, P, ONE>(s, L, x, ws, props);
}

// f(integral_constant P, bool_constant ONE) for the system's pair kernel.
template <class F>
static auto with_pairs(const DevSys& s, F&& f) {
  return with_lanes(s, [&](auto p) { return pair_one(s) ? f(p, std::true_type{}) : f(p, std::false_type{}); });
}

// Doubles of the FP64 phase rows of kc particles of each type that has any.
static size_t rho_doubles(const DevSys& s, int kc) {
  const size_t ld = 32 * (size_t)((s.nkax + 15) / 16 + (s.nkby + 15) / 16) + 16;
  return (pair_one(s) ? 1 : 2) * (size_t)((kc + 3) & ~3) * ld;
}

// LDS bytes of the pair kernels with kc particles per phase chunk (0: no
// phases).
size_t pairs_lds(const DevSys& s, int kc, bool mix) {
  const size_t N = s.nptot;
  auto sums = [&](auto m) {
    return with_pairs(s, [&](auto p, auto one) {
      using S = PairShape<decltype(m)::value, decltype(p)::value, decltype(one)::value>;
      return std::pair<size_t, size_t>(8 * S::NW, (size_t)S::NA * S::PART);
    });
  };
  const auto [red, parts] = mix ? sums(std::true_type{}) : sums(std::false_type{});
  size_t region = sizeof(double) * parts;
  if (mix) {
    if (s.nkxv) region = std::max(region, sizeof(float) * 2 * (size_t)kc * (s.nkxv + s.nkyv));
  } else if (s.nkax) {
    region = std::max(region, sizeof(double) * (4 * N + rho_doubles(s, kc)));
  }
  return sizeof(double) * (4 * N + red) + region;
}

// Particles of each type per FP64 phase chunk: at most 32, and as many as fit
// where two types' partial sums do.  (A CU holds as many blocks with that LDS as
// the registers allow.  One type's sums are half of that: rows that fit there,
// 16 at N = 61 and 900 k-vectors, take 204 us for 4096 walkers, 32 rows 199 and
// all 64, with two blocks per CU, 235.)  As many chunks as that takes, of equal
// size.
int pairs_chunk(const DevSys& s) {
  const size_t room = with_lanes(s, [&](auto p) {
    using S = PairShape<false, decltype(p)::value>;
    return sizeof(double) * ((size_t)S::NA * S::PART - 4 * s.nptot);
  });
  int kc = 32;
  while (kc > 4 && sizeof(double) * rho_doubles(s, kc) > room) kc -= 4;
  const int most = std::max(s.np[0], s.np[1]), n = (most + kc - 1) / kc;
  return std::max(4, ((most + n - 1) / n + 3) & ~3);
}

// Queue the pair kernel of nw walkers on st.
void launch_pairs(const DevSys& s, const WsLayout& L, int nw, bool mix, size_t lds, const double* x, double* ws,
                  double* props, hipStream_t st) {
  with_pairs(s, [&](auto p, auto one) {
    constexpr int P = decltype(p)::value;
    constexpr bool O = decltype(one)::value;
    auto go = [&](auto m) {
      constexpr bool M = decltype(m)::value;
      hipLaunchKernelGGL((k_pairs<M, P, O>), dim3(nw), dim3(PairShape<M, P, O>::T), lds, st, s, L, x, ws, props);
    };
    if (mix) go(std::true_type{});
    else go(std::false_type{});
  });
}

// ---------------------------------------------------------------------------
// k_det
// LDS: A[m*m] complex (column-major, row = orbital, column = particle; the
// inverse overwrites it with row = particle, column = orbital), then a union
// region reused by the phases.
__global__ __launch_bounds__(QMC_BLOCK) void k_det(DevSys s, WsLayout L,
                                                   const double* __restrict__ x,
                                                   double* __restrict__ ws,
                                                   double* __restrict__ Fbuf,
                                                   double* __restrict__ Abuf, int kc,
                                                   int tpp_log2) {
  extern __shared__ __attribute__((aligned(16))) double sm[];
  __shared__ int s_piv[QMC_MAX_ORB];
  __shared__ int s_l, s_sing;
  __shared__ double s_pmax;
  __shared__ zd s_pv, s_akk;
  __shared__ double red[QMC_BLOCK / 64];
  const int w = blockIdx.x, sp = blockIdx.y;
  if (s.nact && w >= *s.nact) return;
  const int m = pick2(s.np, sp);
  if (m == 0) return;
  const int N = s.nptot, p0 = pick2(s.ipf, sp);
  const int tid = threadIdx.x;
  zd* A = (zd*)sm;
  double* U = sm + 2 * m * m;
  double* wsw = ws + (int64_t)w * L.per_walker;
  double* dsc = wsw + pick2(L.off_det, sp);
  zd* Ag = (zd*)(Abuf + (int64_t)w * L.a_per_walker + pick2(L.a_off, sp));  // row-major [k][j]
  zd* Fg = (zd*)(Fbuf + (int64_t)w * L.f_per_walker + pick2(L.f_off, sp));   // [beta][l][j]
  const double* qw = wsw + L.off_q;
  if (tid == 0) s_sing = 0;

  // 1. orbital matrix A(k,i) = exp(i g_k . q_i) (paho_orbitals, reptation.f:10298-10305)
  for (int e = tid; e < m * m; e += QMC_BLOCK) {
    const int k = e / m, i = e - k * m;
    const double kr = qw[2 * (p0 + i)] * s.gvec[2 * k] + qw[2 * (p0 + i) + 1] * s.gvec[2 * k + 1];
    double sv, cv;
    sincos(kr, &sv, &cv);
    const zd z = zmk(cv, sv);
    A[i * m + k] = z;
    Ag[k * m + i] = z;
  }
  block_sync();

  // 2. LU with partial pivoting, LINPACK zgefa semantics: pivot = first row
  // of maximal |re|+|im|; rows are swapped only right of the pivot column.
  for (int k = 0; k < m - 1; k++) {
    if (tid < 64) {
      const int r = k + tid;
      double v = -1.0;
      int idx = 0x7fffffff;
      if (r < m) { v = cabs1(A[k * m + r]); idx = r; }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        const double ov = __shfl_xor(v, o, 64);
        const int oi = __shfl_xor(idx, o, 64);
        if (ov > v || (ov == v && oi < idx)) { v = ov; idx = oi; }
      }
      if (tid == 0) {
        s_l = idx;
        s_pmax = v;
        s_pv = A[k * m + idx];
        s_akk = A[k * m + k];
        s_piv[k] = idx;
        if (v == 0.0) s_sing = 1;
      }
    }
    block_sync();
    if (s_pmax == 0.0) {  // column already triangular (zgefa info = k)
      block_sync();
      continue;
    }
    const int l = s_l;
    const zd pv = s_pv, akk = s_akk;
    const zd tneg = zrcp(pv);
    const zd t = zmk(-tneg.x, -tneg.y);
    const int nr = m - k - 1;
    for (int e = tid; e < nr + nr + 1; e += QMC_BLOCK) {
      if (e < nr) {
        const int j = k + 1 + e;
        if (l != k) {
          const zd a = A[j * m + k];
          A[j * m + k] = A[j * m + l];
          A[j * m + l] = a;
        }
      } else {
        const int i = k + (e - nr);
        if (i == k) A[k * m + k] = pv;
        else {
          const zd old = (i == l) ? akk : A[k * m + i];
          A[k * m + i] = zmul(t, old);
        }
      }
    }
    block_sync();
    for (int e = tid; e < nr * nr; e += QMC_BLOCK) {
      const int jj = e / nr, ii = e - jj * nr;
      const int i = k + 1 + ii, j = k + 1 + jj;
      A[j * m + i] = zfma(A[j * m + k], A[k * m + i], A[j * m + i]);
    }
    block_sync();
  }
  if (tid == 0) {
    s_piv[m - 1] = m - 1;
    if (cabs1(A[(m - 1) * m + (m - 1)]) == 0.0) s_sing = 1;
  }
  block_sync();
  // log|det| = sum log|U_kk| (zgedi det + log, reptation.f:10063, 9412-9430)
  {
    double v = 0.0;
    if (tid < m) v = log(hypot(A[tid * m + tid].x, A[tid * m + tid].y));
    v = block_sum(v, red);
    if (tid == 0) {
      dsc[DS_LOGDET] = v;
      dsc[DS_SING] = s_sing ? 1.0 : 0.0;
    }
  }
  if (s_sing) return;

  // 3. inverse (zgedi job=01 ordering, reptation.f:9437-9468)
  // 3a. inverse of U in place
  zd* rowk = (zd*)U;
  zd* colk = rowk + m;
  for (int k = 0; k < m; k++) {
    for (int e = tid; e < m; e += QMC_BLOCK) {
      if (e > k) rowk[e] = A[e * m + k];
      else if (e < k) colk[e] = A[k * m + e];
      else colk[e] = A[k * m + k];
    }
    block_sync();
    const zd tk = zrcp(colk[k]);
    const int ncol = m - k - 1;
    for (int e = tid; e < (k + 1) * (ncol + 1); e += QMC_BLOCK) {
      const int jj = e / (k + 1), i = e - jj * (k + 1);
      const zd ci = (i < k) ? zmul(zmk(-tk.x, -tk.y), colk[i]) : tk;
      if (jj == 0) {
        A[k * m + i] = ci;
      } else {
        const int j = k + jj;
        const zd base = (i < k) ? A[j * m + i] : zmk(0.0, 0.0);
        A[j * m + i] = zfma(rowk[j], ci, base);
      }
    }
    block_sync();
  }
  // 3b. inverse(U) * inverse(L), right to left, with the column swaps
  zd* work = (zd*)U;
  zd* part = work + m;  // [4][m]
  for (int k = m - 2; k >= 0; k--) {
    for (int i = tid; i < m; i += QMC_BLOCK)
      if (i > k) work[i] = A[k * m + i];
    block_sync();
    {
      const int g = tid >> 6, i = tid & 63;
      zd acc = zmk(0.0, 0.0);
      if (i < m)
        for (int j = k + 1 + g; j < m; j += 4) acc = zfma(work[j], A[j * m + i], acc);
      if (i < m) part[g * m + i] = acc;
    }
    block_sync();
    if (tid < m) {
      const int i = tid;
      zd v = (i <= k) ? A[k * m + i] : zmk(0.0, 0.0);
      for (int g = 0; g < 4; g++) v = zadd(v, part[g * m + i]);
      A[k * m + i] = v;
    }
    block_sync();
    const int l = s_piv[k];
    if (l != k) {
      for (int i = tid; i < m; i += QMC_BLOCK) {
        const zd a = A[k * m + i];
        A[k * m + i] = A[l * m + i];
        A[l * m + i] = a;
      }
    }
    block_sync();
  }

  // 4. F_b = A^-1 diag(i g^b) A (zv, reptation.f:10182-10194), 4x4 tiles;
  // A rows staged from the global copy kc at a time.
  {
    const int tl = tid & 15, tj = tid >> 4;
    const int l0 = 4 * tl, j0 = 4 * tj;
    zd Qx[4][4], Qy[4][4];
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int c = 0; c < 4; c++) { Qx[r][c] = zmk(0, 0); Qy[r][c] = zmk(0, 0); }
    zd* Ac = (zd*)U;
    for (int k0 = 0; k0 < m; k0 += kc) {
      const int kn = min(kc, m - k0);
      for (int e = tid; e < kn * m; e += QMC_BLOCK) Ac[e] = Ag[k0 * m + e];
      block_sync();
      if (l0 < m && j0 < m) {
        for (int kk = 0; kk < kn; kk++) {
          const int k = k0 + kk;
          const double gx = s.gvec[2 * k], gy = s.gvec[2 * k + 1];
          zd ai[4], aj[4];
#pragma unroll
          for (int r = 0; r < 4; r++) ai[r] = (l0 + r < m) ? A[k * m + l0 + r] : zmk(0, 0);
#pragma unroll
          for (int c = 0; c < 4; c++) aj[c] = (j0 + c < m) ? Ac[kk * m + j0 + c] : zmk(0, 0);
#pragma unroll
          for (int r = 0; r < 4; r++)
#pragma unroll
            for (int c = 0; c < 4; c++) {
              const zd P = zmul(ai[r], aj[c]);
              Qx[r][c].x = fma(gx, P.x, Qx[r][c].x);
              Qx[r][c].y = fma(gx, P.y, Qx[r][c].y);
              Qy[r][c].x = fma(gy, P.x, Qy[r][c].x);
              Qy[r][c].y = fma(gy, P.y, Qy[r][c].y);
            }
        }
      }
      block_sync();
    }
    // F = i Q; store and keep the diagonal
    double* dl = U;  // d[j][b] complex: 4 doubles per j
    if (l0 < m && j0 < m) {
#pragma unroll
      for (int r = 0; r < 4; r++)
#pragma unroll
        for (int c = 0; c < 4; c++) {
          const int l = l0 + r, j = j0 + c;
          if (l < m && j < m) {
            const zd fx = zmk(-Qx[r][c].y, Qx[r][c].x);
            const zd fy = zmk(-Qy[r][c].y, Qy[r][c].x);
            Fg[(0 * m + l) * m + j] = fx;
            Fg[(1 * m + l) * m + j] = fy;
            if (l == j) {
              dl[4 * j + 0] = fx.x;
              dl[4 * j + 1] = fx.y;
              dl[4 * j + 2] = fy.x;
              dl[4 * j + 3] = fy.y;
            }
          }
        }
    }
  }
  double* xs = U + 4 * m;
  const double* xw = x + (int64_t)w * 2 * N;
  for (int k = tid; k < 2 * N; k += QMC_BLOCK) xs[k] = xw[k];
  block_sync();

  // 5. drift and the first-derivative Laplacian terms for every particle
  // (reptation.f:10195-10240; the second-derivative ones are k_cross's), with the backflow Jacobian qa and the
  // quasi-coordinate Laplacian qb regenerated from the pair table.
  const double* dl = U;
  const int tpp = 1 << tpp_log2;
  const int lane = tid & (tpp - 1), grp = tid >> tpp_log2, ngrp = QMC_BLOCK >> tpp_log2;
  double acc_g2 = 0.0, acc_h0 = 0.0, acc_h1 = 0.0;
  double* gdet = dsc + DS_N;
  double* Qd = gdet + 2 * N;
  for (int i0 = 0; i0 < N; i0 += ngrp) {
    const int ip = i0 + grp;
    const bool act = ip < N;
    const int ti = act ? ptype(s, ip) : 0;
    const bool on = act && (sp ? pick2(s.iub_flag[1], ti) : pick2(s.iub_flag[0], ti));
    const bool insp = ip >= p0 && ip < p0 + m;
    double zxr = 0, zxi = 0, zyr = 0, zyi = 0, hq = 0;
    double q11 = 0, q12 = 0, q22 = 0, bx = 0, by = 0;
    if (on) {
      const double xi = xs[2 * ip], yi = xs[2 * ip + 1];
      for (int c = lane; c < N; c += tpp) {
        if (c == ip) continue;
        const TabRef tb = tabref<TK_B>(s, tpair(ti, ptype(s, c)));
        if (tb.row0 < 0) continue;
        PairGeo p = pair_geo(s, xi, yi, xs[2 * c], xs[2 * c + 1]);
        double eta, deta, ddeta;
        spline3(s, tb, p.ind, p.rem, eta, deta, ddeta);
        const double cb = deta * p.byr;
        const double mb11 = eta + cb * p.ux * p.ux, mb12 = cb * p.ux * p.uy,
                     mb22 = eta + cb * p.uy * p.uy;
        const double cc = ddeta + 3.0 * cb;
        if (insp) {
          q11 += mb11; q12 += mb12; q22 += mb22;
          bx += cc * p.ux; by += cc * p.uy;
        }
        if (c >= p0 && c < p0 + m) {
          const int jf = c - p0;
          const double dxr = dl[4 * jf], dxi = dl[4 * jf + 1], dyr = dl[4 * jf + 2],
                       dyi = dl[4 * jf + 3];
          // qa(.,.,c,ip) = -mb
          zxr -= dxr * mb11 + dyr * mb12;
          zxi -= dxi * mb11 + dyi * mb12;
          zyr -= dxr * mb12 + dyr * mb22;
          zyi -= dxi * mb12 + dyi * mb22;
          // qb(.,ip,c) = -cc u
          hq -= cc * (dxr * p.ux + dyr * p.uy);
        }
      }
    }
    for (int o = 1; o < tpp; o <<= 1) {
      zxr += __shfl_xor(zxr, o, 64);
      zxi += __shfl_xor(zxi, o, 64);
      zyr += __shfl_xor(zyr, o, 64);
      zyi += __shfl_xor(zyi, o, 64);
      hq += __shfl_xor(hq, o, 64);
      q11 += __shfl_xor(q11, o, 64);
      q12 += __shfl_xor(q12, o, 64);
      q22 += __shfl_xor(q22, o, 64);
      bx += __shfl_xor(bx, o, 64);
      by += __shfl_xor(by, o, 64);
    }
    if (act && lane == 0) {
      if (on) {
        if (insp) {
          const int jf = ip - p0;
          const double a11 = 1.0 + q11, a12 = q12, a22 = 1.0 + q22;
          const double dxr = dl[4 * jf], dxi = dl[4 * jf + 1], dyr = dl[4 * jf + 2],
                       dyi = dl[4 * jf + 3];
          zxr += dxr * a11 + dyr * a12;
          zxi += dxi * a11 + dyi * a12;
          zyr += dxr * a12 + dyr * a22;
          zyi += dxi * a12 + dyi * a22;
          hq += dxr * bx + dyr * by;
          Qd[3 * jf] = q11;
          Qd[3 * jf + 1] = q12;
          Qd[3 * jf + 2] = q22;
        }
        gdet[2 * ip] = -zxr;
        gdet[2 * ip + 1] = -zyr;
        acc_g2 += pick2(s.hbs2m, ti) * (zxi * zxi + zyi * zyi);
        if (ti == 0) acc_h0 -= hq;
        else acc_h1 -= hq;
      } else {
        gdet[2 * ip] = 0.0;
        gdet[2 * ip + 1] = 0.0;
      }
    }
  }
  acc_g2 = block_sum(acc_g2, red);
  acc_h0 = block_sum(acc_h0, red);
  acc_h1 = block_sum(acc_h1, red);
  if (tid == 0) {
    dsc[DS_H0] = acc_h0;
    dsc[DS_H1] = acc_h1;
    dsc[DS_G2] = acc_g2;
  }
}

// ---------------------------------------------------------------------------
// k_final: one wavefront per walker.  delta is the current time step (the
// COMMON delta that kinetic's drift cutoff reads, reptation.f:2755).
//
// Without backflow (s.plain) the Jacobian is the identity, and what k_fgrad
// and k_cross compute reduces to F's diagonal d_j: the drift is -Re d_j, the
// cross term sum_j Re(d_j . d_j), and the second-derivative term, a trace,
// sum_j (A^-1 G^2 A)_jj = -sum_k |g_k|^2.  Those two kernels are not launched
// (at N=26, 256 walkers 31 of an 82 us VMC step, at N=122 1.05 of a 1.9 ms
// evaluation).
//
// Bound by latency: one wavefront per block, so that a few hundred walkers
// reach every CU, what it reads fetched before anything depends on it, and
// sums of property slots formed in registers (with four walkers per block and
// slots read back after their stores 6.8 us at N = 26, 256 walkers, now 4.9 us).
__global__ __launch_bounds__(64) void k_final(DevSys s, WsLayout L, double* __restrict__ ws,
                                              double* __restrict__ props,
                                              double* __restrict__ gout,
                                              double* __restrict__ hout,
                                              double* __restrict__ grad2,
                                              int32_t* __restrict__ status,
                                              double delta) {
  const int w = blockIdx.x;
  const int lane = threadIdx.x & 63;
  if (s.nact && w >= *s.nact) return;
  const int N = s.nptot;
  const double* __restrict__ wsw = ws + (int64_t)w * L.per_walker;
  const double* sc = wsw + L.off_sc;
  double ltf = sc[SC_LTF];
  double h[2] = {sc[SC_H0], sc[SC_H1]};
  const double pv[3] = {sc[SC_P0], sc[SC_P1], sc[SC_PT]};
  const double g2in = grad2[w];
  bool sing = false, guard = false;
  double hd[2] = {0.0, 0.0}, g2ph = 0.0;
  if (s.has_det) {
#pragma unroll
    for (int sp = 0; sp < 2; sp++) {
      if (sp >= s.ntypes || s.np[sp] == 0) continue;
      const double* dsc = wsw + L.off_det[sp];
      ltf -= dsc[DS_LOGDET];
      if (dsc[DS_SING] != 0.0) sing = true;
      if (s.plain) continue;
      hd[0] += dsc[DS_H0] + dsc[DS_X0];
      hd[1] += dsc[DS_H1] + dsc[DS_X1];
      g2ph += dsc[DS_G2];
    }
    // underflow guard of slater_excitations (reptation.f:10087-10092)
    guard = !(exp(-ltf * 2.0) > 0.0);
  }
  const bool use_det = s.has_det && !guard && !sing;
  if (use_det) {
    h[0] += hd[0];
    h[1] += hd[1];
  }
  double* gw = gout + (int64_t)w * 2 * N;
  double g2t[2] = {0.0, 0.0}, ggs = 0.0;
  double dd[2] = {0.0, 0.0}, im2 = 0.0;  // s.plain: Re sum d.d per type, fixed-phase term
  for (int i = lane; i < N; i += 64) {
    double gx = wsw[L.off_gj + 2 * i], gy = wsw[L.off_gj + 2 * i + 1];
    if (use_det && s.plain) {
      // particles of a type couple to their own spin's orbitals alone
      const int t = ptype(s, i);
      if (t ? s.iub_flag[1][1] : s.iub_flag[0][0]) {
        const double* Fd =
            wsw + pick2(L.off_det, t) + DS_N + 2 * N + 3 * pick2(s.np, t) + 4 * (i - pick2(s.ipf, t));
        const double xr = Fd[0], xi = Fd[1], yr = Fd[2], yi = Fd[3];
        gx -= xr;
        gy -= yr;
        const double v = (xr * xr - xi * xi) + (yr * yr - yi * yi);
        if (t == 0) dd[0] += v;
        else dd[1] += v;
        im2 += pick2(s.hbs2m, t) * (xi * xi + yi * yi);
      }
    } else if (use_det) {
      for (int sp = 0; sp < s.ntypes; sp++) {
        if (pick2(s.np, sp) == 0) continue;
        const double* gd = wsw + pick2(L.off_det, sp) + DS_N;
        gx += gd[2 * i];
        gy += gd[2 * i + 1];
      }
    }
    const int t = ptype(s, i);
    const double x2 = gx * gx + gy * gy;
    if (s.adrift != 0.0) {
      // drift cutoff (kinetic, reptation.f:2747-2760), vari as sigma sets it
      // (reptation.f:855-870); every particle here has hbs2m != 0
      const double vari = 1.0 / (2.0 * pick2(s.hbs2m, t) * delta);
      double gg = x2 * s.adrift * delta * delta * vari;
      gg = (-1.0 + sqrt(1.0 + 2.0 * gg)) / gg;
      ggs += gg;
      gx *= gg;
      gy *= gg;
    }
    if (t == 0) g2t[0] += x2;
    else g2t[1] += x2;
    gw[2 * i] = gx;
    gw[2 * i + 1] = gy;
  }
  g2t[0] = wave_sum(g2t[0]);
  g2t[1] = wave_sum(g2t[1]);
  ggs = wave_sum(ggs);
  if (use_det && s.plain) {
    g2ph = wave_sum(im2);
#pragma unroll
    for (int t = 0; t < 2; t++)
      if (t < s.ntypes && s.np[t] > 0 && s.iub_flag[t][t]) h[t] += s.g2sum[t] + wave_sum(dd[t]);
  }
  if (lane == 0) {
    double* p = props + (int64_t)w * s.n_props;
    double kin0 = 0.0;
#pragma unroll
    for (int t = 0; t < 2; t++) {
      if (t >= s.ntypes) break;
      hout[(int64_t)w * 2 + t] = h[t];
      if (s.hbs2m[t] == 0.0) continue;  // no kinetic slots (reptation.f:2739)
      const double kin = s.hbs2m[t] * (h[t] - g2t[t]);
      kin0 += kin;
      p[s.jkin[t]] = kin / s.np[t];
      p[s.jun[t]] = 1.0 / sqrt(g2t[t]);
    }
    if (s.ntypes == 1) hout[(int64_t)w * 2 + 1] = 0.0;
    p[s.jgg] = (s.adrift == 0.0) ? 1.0 : ggs / s.npnorm;
    if (use_det) grad2[w] = g2ph;
    p[s.jltf] = ltf;
#pragma unroll
    for (int t = 0; t < 2; t++)
      if (t < s.ntypes && s.jpot[t] >= 0) p[s.jpot[t]] = (s.tailc[t] + pv[t]) / s.np[t];
    const double pkin = kin0 / s.npnorm;
    const double pefp = (s.ntheta != 0) ? (use_det ? g2ph : g2in) / s.npnorm : 0.0;
    const double ppot = (s.tailc_tot + pv[2] + s.v0) / s.npnorm;
    const double ptot = ppot + pkin + pefp;
    p[s.jkin0] = pkin;
    p[s.jefp] = pefp;
    p[s.jpot0] = ppot;
    p[s.jetot] = ptot;
    p[s.je2] = ptot * ptot;
    if (status) status[w] = (guard ? 1 : 0) | (sing ? 2 : 0);
  }
}
