// qmc_pairs.h -- the schedule on which the pair kernels (k_pairs, k_fgrad) visit
// a walker's pairs.
#pragma once
#include <type_traits>

#include "qmc_dev.h"

// The pair passes visit every unordered pair once, on a round-robin
// schedule over blocks of P lanes, P = 16, 32 or 64 the power of two that
// holds the larger type: the particles of type t sit in lanes 0..np_t-1 of a
// block, and step d of block pair (I, J) pairs lane l of I with lane
// (l + d) mod P of J, so within a step every lane has a distinct partner.
// Within one type d runs over 1..P/2 (d = P/2 on the lower half of the lanes
// only), across the two types over 0..P-1.  A wavefront takes 64 / P steps of
// one block pair at a time, one per group of P lanes (P^2 / 32 wavefront
// steps in all: with one group of 64 lanes for every size, N = 26 would take
// 128 steps of 13 live lanes instead of 8), and the wavefront steps are split
// into NW contiguous runs.  A pair's contribution to i stays in registers
// until the wavefront's run leaves block I; its contribution to j is added to
// the lane group's own partial sums in LDS (distinct j within a step, so no
// two lanes touch one address), and the NA = NW 64 / P partial sums are added
// in a fixed order afterwards: the result does not depend on scheduling.
// ONE: particles of one type alone, whose sums take half the LDS.
template <bool MIX, int P, bool ONE_ = false>
struct PairShape {
  static constexpr bool ONE = ONE_;
  static constexpr int NW = P == 16 || MIX ? 4 : 8;  // wavefronts
  static constexpr int T = 64 * NW, SUB = 64 / P, NA = NW * SUB;
  static constexpr int OWN = P / 2 / SUB, ACROSS = P / SUB;  // wavefront steps of a block pair
  static constexpr int NS = ONE ? P : 2 * P;  // particles a sum's row holds
  static constexpr int PART = 6 * NS;  // doubles of one group's partial sums (k_pairs)
};

// What the tables of a type pair are, read through the constant address space:
// scalar loads.  (Through a plain pointer they are vector loads of every step as
// soon as a statement that might write memory, such as a barrier's wait, stands
// before them: k_pairs of N = 122, 4096 walkers 498 us instead of 452.)
typedef const __attribute__((address_space(4))) TpInfo* TpPtr;

// The wavefront's run of pair steps: pair(T, tp, i, j) for each of its lanes'
// pairs (type pair tp), block(ti, tj) after each block pair's, end(ti) when the
// run leaves block ti.
template <class S, int P, class Pair, class Block, class End>
__device__ __forceinline__ void pair_run(const DevSys& s, int wv, int l, Pair&& pair, Block&& block, End&& end) {
  const int lp = l & (P - 1), sub = l / P;
  // schedule: both types present, or the one type t1
  const bool two = s.ntypes > 1 && s.np[0] > 0 && s.np[1] > 0;
  const int t1 = (s.ntypes > 1 && s.np[0] == 0) ? 1 : 0;
  const int nU = two ? 2 * S::OWN + S::ACROSS : S::OWN;
  const int u0 = wv * nU / S::NW, u1 = (wv + 1) * nU / S::NW;
  // blocks (0, 0), (0, 1), (1, 1): type 0's own and across are one stretch of i
  for (int blk = 0; blk < 3; blk++) {
    if (!two && blk > 0) break;
    const int ti = two ? (blk == 2 ? 1 : 0) : t1, tj = two ? (blk == 0 ? 0 : 1) : t1;
    const int b0 = blk == 0 ? 0 : (blk == 1 ? S::OWN : S::OWN + S::ACROSS);
    const int b1 = blk == 0 ? S::OWN : (blk == 1 ? S::OWN + S::ACROSS : 2 * S::OWN + S::ACROSS);
    const int a = max(u0, b0), b = min(u1, b1);
    if (a < b) {
      const int tp = tpair(ti, tj);
      const TpPtr T = (TpPtr)(s.tpi + tp);
      const int ni = pick2(s.np, ti), nj = pick2(s.np, tj), i = pick2(s.ipf, ti) + lp;
      for (int u = a; u < b; u++) {
        const int d = (u - b0) * S::SUB + sub + (ti == tj ? 1 : 0);
        const int jl = (lp + d) & (P - 1);
        if (lp < ni && jl < nj && (ti != tj || d < P / 2 || lp < P / 2)) pair(T, tp, i, pick2(s.ipf, tj) + jl);
      }
      block(ti, tj);
    }
    if (u0 < u1 && (blk == 2 || !two || (blk == 1 && u0 < b1))) end(ti);
  }
}

// Lanes per block of the pair schedule for a system.
static inline int pair_lanes(const DevSys& s) {
  const int m = s.np[0] > s.np[1] ? s.np[0] : s.np[1];
  return m <= 16 ? 16 : m <= 32 ? 32 : 64;
}

// Whether all particles are of one type.
static inline bool pair_one(const DevSys& s) { return s.ntypes == 1 || s.np[0] == 0 || s.np[1] == 0; }

// f(integral_constant P) for the system's lanes per block.
template <class F>
static auto with_lanes(const DevSys& s, F&& f) {
  switch (pair_lanes(s)) {
    case 16: return f(std::integral_constant<int, 16>{});
    case 32: return f(std::integral_constant<int, 32>{});
    default: return f(std::integral_constant<int, 64>{});
  }
}
