// qmc_cross.hip -- backflow Laplacian cross term on the FP64 matrix cores.
//
// For every spin s and particle type t with backflow between them,
//   h_t += sum_{ip in t, idim} sum_{j,k} Re[(qa F)(qa F)]   (reptation.f:10241-10259)
//   h_t -= sum_{ip in t, idim} sum_j qa qa (F_a F_b)_jj     (reptation.f:10195-10240)
// of which the first is the symmetric contraction sum_{r,q} M[r][q] S_t[r][q] over rows
// r = (j, a) of the spin's particles (R = 2m <= 128 rows) with
//   M[(j,a),(k,b)] = Re(F_a(k,j) F_b(j,k))            (symmetric),
//   S_t = V_t V_t^T,  V_t[(j,a),(ip,idim)] = qa(a,idim,j,ip),
// qa being the backflow Jacobian: 1 + Q_j on the particle's own block and
// -(eta delta + eta' r u u) for a pair (reptation.f:10023-10058).
//
// One workgroup per (walker, spin).  S_t is a SYRK built from 16 x 16 tiles
// with v_mfma_f64_16x16x4f64, the tiles of the upper triangle shared between the
// wavefronts (XcShape).  V_t is staged in LDS 8 or 16 particles (KC columns) at
// a time, column-major so each MFMA operand is one 8-byte LDS read per lane.  M is formed from F (L2) tile by tile when S_t is
// complete, once for both particle types, so only the S accumulators stay in
// registers through the chunks and F is read once per (walker, spin); it is
// prefetched into L2 while the last chunk's products run.
#include <type_traits>

#include "qmc_dev.h"

typedef double xc_d4 __attribute__((ext_vector_type(4)));

// The kernel's shape for spins of up to 8 NB particles: NB 16-row tiles per
// side of S, of which the upper triangle goes to W wavefronts, and chunks of
// KC columns.  Padding to the full 128 rows made the tiles beyond the spin's the
// larger part of the work (33 of 36 tiles at 13 particles per spin, 26 of 36 at
// 29): N = 26, 4096 walkers 209 us (now 39), N = 58, 512 walkers 45 us (now 22),
// N = 74, 256 walkers 36 us (now 27).  Wavefronts and chunk: enough threads to
// form a chunk's entries in one or two turns, and LDS for as many blocks as the
// registers allow. (N = 58 with chunks of 32 columns 32 us, with 8 wavefronts 28; N
// = 26, 4096 walkers with 4 wavefronts 44, with one 45 us.)
template <int NB>
struct XcShape {
  static constexpr int W = NB >= 6 ? 8 : NB == 4 ? 4 : 2, T = 64 * W;
  static constexpr int KC = NB >= 6 ? 32 : 16;
  static constexpr int JR = 8 * NB;        // particles (rows of 2)
  static constexpr int RS = 16 * NB + 16;  // LDS row stride: the 16-lane groups of an operand read disjoint banks
  static constexpr int NTILE = NB * (NB + 1) / 2;
  static constexpr int TPW = (NTILE + W - 1) / W;  // most tiles per wavefront
  static constexpr int EPT = (JR * (KC / 2) + T - 1) / T;  // entries of a chunk per thread
  // tiles of wavefront w: the first NTILE % W take one more
  __host__ __device__ static constexpr int nt(int w) { return NTILE / W + (w < NTILE % W ? 1 : 0); }
  // tile q of wavefront w.  NB = 8: wavefronts g and g + 4 (one SIMD) share
  // block rows g and 7 - g, 5 + 4 tiles; else the triangle row by row.
  __host__ __device__ static constexpr int tile(int w, int q, bool col) {
    if (NB == 8) {
      const int g = w & 3, i = (w >> 2 ? 5 : 0) + q;
      const int tj = i < 8 - g ? g : 7 - g;
      return !col ? tj : i < 8 - g ? g + i : (7 - g) + (i - (8 - g));
    }
    int i = q;
    for (int v = 0; v < w; v++) i += nt(v);
    int tj = 0;
    while (i >= NB - tj) i -= NB - tj++;
    return col ? tj + i : tj;
  }
  __host__ __device__ static constexpr int tj(int w, int q) { return tile(w, q, false); }
  __host__ __device__ static constexpr int tk(int w, int q) { return tile(w, q, true); }
  __host__ __device__ static constexpr bool needs(int w, int b) {
    for (int q = 0; q < nt(w); q++)
      if (tj(w, q) == b || tk(w, q) == b) return true;
    return false;
  }
};

// f(integral_constant q) for q = 0..N-1.
template <int N, class F>
__device__ __forceinline__ void xc_each(F&& f) {
  if constexpr (N > 0) {
    xc_each<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

// f(integral_constant NB) for the larger spin's size.
template <class F>
static auto with_cross_shape(const DevSys& s, F&& f) {
  const int m = s.np[0] > s.np[1] ? s.np[0] : s.np[1];
  if (m <= 16) return f(std::integral_constant<int, 2>{});
  if (m <= 32) return f(std::integral_constant<int, 4>{});
  if (m <= 48) return f(std::integral_constant<int, 6>{});
  return f(std::integral_constant<int, 8>{});
}

// real part of the product of two elements of F (complex, or real orbitals')
__device__ __forceinline__ double xc_re(zd a, zd b) { return a.x * b.x - a.y * b.y; }
__device__ __forceinline__ double xc_re(double a, double b) { return a * b; }

// Empty statement that takes the accumulator in registers: the MFMAs that
// produce it are issued before this point.
__device__ __forceinline__ void xc_pin(xc_d4& a) { __asm__ volatile("" : "+v"(a)); }

// The 2 x 2 diagonal blocks of S_t (rows and columns (j, a), (j, b); the
// three distinct entries at index a + b), from the wavefronts that hold the
// diagonal tiles: sd[(t * 64 + j) * 3 + a + b].
template <int NB, int V>
__device__ __forceinline__ void xc_diag_blocks(const xc_d4 (&acc)[2][XcShape<NB>::TPW], double* __restrict__ sd, int lane) {
  xc_each<XcShape<NB>::nt(V)>([&](auto qc) {
    constexpr int q = decltype(qc)::value, TJ = XcShape<NB>::tj(V, q), TK = XcShape<NB>::tk(V, q);
    if constexpr (TJ != TK) return;
    const int c = lane & 15;
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int r = (lane >> 4) + 4 * v;
      if ((r >> 1) == (c >> 1) && r <= c) {
        const int e = (8 * TJ + (r >> 1)) * 3 + (r & 1) + (c & 1);
        sd[e] = acc[0][q][v];
        sd[192 + e] = acc[1][q][v];
      }
    }
  });
}

// Sums over the wavefront's tiles of M o (S_t - S_t's diagonal blocks), M
// formed from F here once for both particle types.  The diagonal blocks are
// the second-derivative terms sum_ab (F_a F_b)_jj S_t[(j,a),(j,b)]
// (reptation.f:10195-10240): (F_a F_b)_jj is the sum over k of M[(j,a),(k,b)],
// so each element of M takes both S_t[(j,a),(k,b)] and the block of its row.
// An element above the diagonal stands for its mirror image too, whose row is
// its column.  The accumulator of v_mfma_f64_16x16x4f64 holds, in lane l and
// register v, element (row l/16 + 4v, column l%16) of the 16 x 16 tile.
template <int NB, int V, typename Z>
__device__ __forceinline__ void xc_contract(const xc_d4 (&acc)[2][XcShape<NB>::TPW], const double* __restrict__ sd,
                                            const Z* __restrict__ Fg, int m, int lane_in, int nT, double& t0,
                                            double& t1) {
  const int R = 2 * m;
  // the addresses of F are formed here, not hoisted out of the chunk loops
  // (where they would have to be spilled)
  const Z* Fq = Fg;
  int lane = lane_in;
  __asm__ volatile("" : "+s"(Fq), "+v"(lane));
  t0 = t1 = 0.0;
  xc_each<XcShape<NB>::nt(V)>([&](auto qc) {
    constexpr int q = decltype(qc)::value, TJ = XcShape<NB>::tj(V, q), TK = XcShape<NB>::tk(V, q);
    if (TK < nT) {
      const int sc = 16 * TK + (lane & 15);
      const int ks = sc >> 1, bs = sc & 1;
      double u0 = 0.0, u1 = 0.0;
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int r = 16 * TJ + (lane >> 4) + 4 * v;
        if (r < R && sc < R) {
          const int jr = r >> 1, ar = r & 1;
          const double mv = xc_re(Fq[(ar * m + ks) * m + jr], Fq[(bs * m + jr) * m + ks]);
          const double* dj = sd + 3 * jr + ar + bs;
          if (TJ == TK) {
            u0 = fma(mv, acc[0][q][v] - dj[0], u0);
            u1 = fma(mv, acc[1][q][v] - dj[192], u1);
          } else {
            const double* dk = sd + 3 * ks + ar + bs;
            u0 = fma(mv, 2.0 * acc[0][q][v] - (dj[0] + dk[0]), u0);
            u1 = fma(mv, 2.0 * acc[1][q][v] - (dj[192] + dk[192]), u1);
          }
        }
      }
      t0 += u0;
      t1 += u1;
    }
    // one tile's F values in flight at a time
    __asm__ volatile("" ::: "memory");
  });
}

// Entry e (row j = e % JR, particle pc = e / JR) of the V chunk of
// particles c0..c0+cn-1: rows j beyond m and particles beyond cn are zero;
// the 2 x 2 block of (j, ip) is symmetric.  Consecutive threads take
// consecutive rows, so the column-major stores spread over the LDS banks.
template <int NB>
__device__ __forceinline__ void xc_entry(const DevSys& s, const double* __restrict__ Qd,
                                         const double* __restrict__ xs, double* __restrict__ Vt, TabRef tb,
                                         int e, int c0, int cn, int m, int p0) {
  typedef XcShape<NB> S;
  const int j = e % S::JR, pc = e / S::JR;
  if (S::JR * (S::KC / 2) % S::T != 0 && pc >= S::KC / 2) return;
  double v11 = 0, v12 = 0, v22 = 0;
  const int ip = c0 + pc;
  if (j < m && pc < cn) {
    const int jp = p0 + j;
    if (jp == ip) {
      v11 = 1.0 + Qd[3 * j];
      v12 = Qd[3 * j + 1];
      v22 = 1.0 + Qd[3 * j + 2];
    } else if (tb.row0 >= 0) {
      const double2 xj2 = ld2(xs, jp), xi2 = ld2(xs, ip);
      PairGeo pg = pair_geo(s, xj2.x, xj2.y, xi2.x, xi2.y);
      double eta, deta, ddeta;
      spline3(s, tb, pg.ind, pg.rem, eta, deta, ddeta);
      const double cb = deta * pg.byr;
      v11 = -(eta + cb * pg.ux * pg.ux);
      v12 = -(cb * pg.ux * pg.uy);
      v22 = -(eta + cb * pg.uy * pg.uy);
    }
  }
  // rows 2j, 2j+1 of each of the two columns: one 16-byte store each
  // (RS is even, so both are 16-byte aligned)
  *reinterpret_cast<double2*>(Vt + (2 * pc) * S::RS + 2 * j) = make_double2(v11, v12);
  *reinterpret_cast<double2*>(Vt + (2 * pc + 1) * S::RS + 2 * j) = make_double2(v12, v22);
}

// Destination of the L2 prefetch of F: one wavefront's 64 x 16 bytes, never read.
__shared__ __attribute__((aligned(16))) unsigned xc_sink[256];

// Body of wavefront V.  The V_t chunks (KC / 2 particles of one type at a time,
// over the types with backflow to this spin) are double-buffered: while the
// matrix cores take this chunk's products the vector units build the next chunk
// into the other buffer (EPT entries per thread, one or two, placed between the
// MFMA steps), so a chunk costs one barrier.
template <int NB, int V, typename Z>
__device__ __forceinline__ void xc_body(const DevSys& s, double* __restrict__ dsc, const double* __restrict__ Qd,
                                        const Z* __restrict__ Fg, const double* __restrict__ xs,
                                        double* __restrict__ Vt, double* red, int sp, int m, int p0, int tid) {
  typedef XcShape<NB> S;
  constexpr int XC_KC = S::KC, XC_RS = S::RS, XC_THREADS = S::T;
  const int lane = tid & 63;
  const int nT = (2 * m + 15) >> 4;
  // S_t accumulators of both particle types (zero for a type without
  // backflow to this spin), contracted with M in one pass over F at the end
  xc_d4 acc[2][S::TPW];
#pragma unroll
  for (int t = 0; t < 2; t++)
#pragma unroll
    for (int q = 0; q < S::TPW; q++) acc[t][q] = xc_d4{0.0, 0.0, 0.0, 0.0};
  bool act[2];
#pragma unroll
  for (int t = 0; t < 2; t++)
    act[t] = t < s.ntypes && (sp ? pick2(s.iub_flag[1], t) : pick2(s.iub_flag[0], t)) && pick2(s.np, t) > 0;
  const int ft = act[0] ? 0 : (act[1] ? 1 : -1);
  if (ft >= 0) {
    const int c0 = pick2(s.ipf, ft), cn = min(XC_KC / 2, pick2(s.np, ft));
    const TabRef tb = tabref<TK_B>(s, tpair(sp, ft));
    for (int e = tid; e < S::JR * (XC_KC / 2); e += XC_THREADS) xc_entry<NB>(s, Qd, xs, Vt, tb, e, c0, cn, m, p0);
  }
  block_sync();
  int cur = 0;
#pragma unroll
  for (int t = 0; t < 2; t++) {
    if (!act[t]) continue;
    const int ia = pick2(s.ipf, t), ib = ia + pick2(s.np, t);
    for (int c0 = ia; c0 < ib; c0 += XC_KC / 2) {
      // the next chunk: the rest of this type, then the other type
      int nt = t, nc0 = c0 + XC_KC / 2;
      if (nc0 >= ib) {
        nt = (t == 0 && act[1]) ? 1 : -1;
        nc0 = nt >= 0 ? pick2(s.ipf, 1) : 0;
      }
      const int ncn = nt >= 0 ? min(XC_KC / 2, pick2(s.ipf, nt) + pick2(s.np, nt) - nc0) : 0;
      const TabRef ntb = nt >= 0 ? tabref<TK_B>(s, tpair(sp, nt)) : TabRef{-1, 0};
      double* Vn = Vt + (cur ^ 1) * (XC_KC * XC_RS);
      const double* base = Vt + cur * (XC_KC * XC_RS) + (lane >> 4) * XC_RS + (lane & 15);
      // particles in this chunk: its columns 2 cn and beyond are zero, and
      // a step whose four columns all are is skipped
      const int cn = min(XC_KC / 2, ib - c0);
#pragma unroll
      for (int ks = 0; ks < XC_KC / 4; ks++) {
        if (2 * ks < cn) {
          // rows beyond 2m are zero in LDS, so tiles past the last block row
          // add zeros and need no branch here
          double blk[NB];
          xc_each<NB>([&](auto bc) {
            constexpr int b = decltype(bc)::value;
            if constexpr (XcShape<NB>::needs(V, b)) blk[b] = base[ks * 4 * XC_RS + 16 * b];
          });
          xc_each<XcShape<NB>::nt(V)>([&](auto qc) {
            constexpr int q = decltype(qc)::value, TJ = XcShape<NB>::tj(V, q), TK = XcShape<NB>::tk(V, q);
            acc[t][q] = __builtin_amdgcn_mfma_f64_16x16x4f64(blk[TJ], blk[TK], acc[t][q], 0, 0, 0);
          });
#pragma unroll
          for (int q = 0; q < XcShape<NB>::nt(V); q++) xc_pin(acc[t][q]);
        }
        if (nt >= 0 && (ks == 1 || (S::EPT == 2 && ks == 1 + XC_KC / 8)))
          xc_entry<NB>(s, Qd, xs, Vn, ntb, tid + (ks == 1 ? 0 : XC_THREADS), nc0, ncn, m, p0);
        // during the last chunk, F of this (walker, spin) is fetched into
        // the L2 cache (16 bytes a lane, into an LDS sink nothing reads), a
        // part at every other step, so the contraction below reads it
        // from there instead of waiting on HBM tile by tile
        if (nt < 0 && (ks & 1)) {
          const int nz = 2 * m * m * (int)sizeof(Z) / 16;
          for (int i = tid + (ks >> 1) * XC_THREADS; i < nz; i += XC_KC / 8 * XC_THREADS)
            __builtin_amdgcn_global_load_lds((const void*)((const double2*)Fg + i), (void __attribute__((address_space(3)))*)xc_sink,
                                             16, 0, 0);
        }
        // the next step's operands are read after this step's MFMAs issue
        __asm__ volatile("" ::: "memory");
      }
      block_sync();
      cur ^= 1;
    }
  }
  // the chunk buffers are free: the diagonal blocks go there
  xc_diag_blocks<NB, V>(acc, Vt, lane);
  block_sync();
  double u0, u1;
  xc_contract<NB, V>(acc, Vt, Fg, m, lane, nT, u0, u1);
  u0 = block_sum<XC_THREADS>(u0, red);
  u1 = block_sum<XC_THREADS>(u1, red);
  if (tid == 0) {
    dsc[DS_X0] = u0;
    dsc[DS_X1] = u1;
  }
}

// LDS: xs[2N], then two Vt[KC][RS] chunk buffers (column = (particle, idim) of
// the chunk, row = (j, a)).  Z: zd (complex F: k_gjc, k_det) or double (k_gjr).
template <typename Z, int NB>
__global__ __launch_bounds__(XcShape<NB>::T, 4) void k_cross(DevSys s, WsLayout L, const double* __restrict__ x,
                                                             double* __restrict__ ws,
                                                             const double* __restrict__ Fbuf) {
  constexpr int W = XcShape<NB>::W;
  extern __shared__ __attribute__((aligned(16))) double sm[];
  __shared__ double red[W];
  // walkers and spins in the reverse of the order in which the determinant
  // kernel wrote their F, so the first workgroups find theirs still in the
  // memory-side cache
  const int w = gridDim.x - 1 - blockIdx.x, sp = gridDim.y - 1 - blockIdx.y;
  if (s.nact && w >= *s.nact) return;
  const int m = pick2(s.np, sp);
  if (m == 0) return;
  const int N = s.nptot, p0 = pick2(s.ipf, sp);
  const int tid = threadIdx.x;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  double* wsw = ws + (int64_t)w * L.per_walker;
  double* dsc = wsw + pick2(L.off_det, sp);
  if (dsc[DS_SING] != 0.0) return;
  const double* Qd = dsc + DS_N + 2 * N;
  const Z* Fg = (const Z*)(Fbuf + (int64_t)w * L.f_per_walker + pick2(L.f_off, sp));
  double* xs = sm;
  double* Vt = sm + 2 * N;
  const double* xw = x + (int64_t)w * 2 * N;
  for (int k = tid; k < 2 * N; k += 64 * W) xs[k] = xw[k];
  block_sync();
#define XC_CASE(v)                                                                              \
  case v:                                                                                       \
    if constexpr (v < W) xc_body<NB, v>(s, dsc, Qd, Fg, xs, Vt, red, sp, m, p0, tid);           \
    break;
  switch (wv) { XC_CASE(0) XC_CASE(1) XC_CASE(2) XC_CASE(3) XC_CASE(4) XC_CASE(5) XC_CASE(6) XC_CASE(7) }
#undef XC_CASE
}

void launch_cross(const DevSys& s, const WsLayout& L, int nw, bool real, const double* x, double* ws,
                  const double* F, hipStream_t st) {
  with_cross_shape(s, [&](auto nb) {
    constexpr int NB = decltype(nb)::value;
    typedef XcShape<NB> S;
    const size_t lds = sizeof(double) * (2 * s.nptot + 2 * S::KC * S::RS);
    const dim3 grid(nw, s.ntypes);
    if (real) hipLaunchKernelGGL((k_cross<double, NB>), grid, dim3(S::T), lds, st, s, L, x, ws, F);
    else hipLaunchKernelGGL((k_cross<zd, NB>), grid, dim3(S::T), lds, st, s, L, x, ws, F);
  });
}
