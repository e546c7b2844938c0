// qmc_sem.h -- what the single-electron move kernels share: exp and log of the
// move loop, the jobs of a packed launch, and the real-orbital launch.
#pragma once
#include "qmc_internal.h"

// exp and log for the move loop, their constants kept in scalar registers
// (qk<true>) so that the loop does not hold them in vector registers next to
// the inverse.  exp: Cody-Waite reduction x = n ln2 + r (ln2 over two
// doubles), |r| <= ln2 / 2, the Taylor series of e^r through r^13
// (truncation below 5e-18), scaled by 2^n; arguments are clamped to
// [-746, 710], beyond which the result is 0 or +inf.  log: x = m 2^e with
// m in [sqrt(1/2), sqrt(2)), log m = 2 atanh(s), s = (m - 1) / (m + 1),
// |s| <= 0.1716, the series through s^21 (truncation below 1e-18), plus
// e ln2; x > 0.
__device__ __forceinline__ double sem_exp(double x) {
  x = fmin(fmax(x, -746.0), 710.0);
  const double n = rint(x * qk<true>(0x1.71547652b82fep+0));
  double r = fma(-n, qk<true>(0x1.62e42fefa39efp-1), x);
  r = fma(-n, qk<true>(0x1.abc9e3b39803fp-56), r);
  double p = qk<true>(1.0 / 6227020800.0);
  p = fma(p, r, qk<true>(1.0 / 479001600.0));
  p = fma(p, r, qk<true>(1.0 / 39916800.0));
  p = fma(p, r, qk<true>(1.0 / 3628800.0));
  p = fma(p, r, qk<true>(1.0 / 362880.0));
  p = fma(p, r, qk<true>(1.0 / 40320.0));
  p = fma(p, r, qk<true>(1.0 / 5040.0));
  p = fma(p, r, qk<true>(1.0 / 720.0));
  p = fma(p, r, qk<true>(1.0 / 120.0));
  p = fma(p, r, qk<true>(1.0 / 24.0));
  p = fma(p, r, qk<true>(1.0 / 6.0));
  p = fma(p, r, 0.5);
  p = fma(p, r, 1.0);
  p = fma(p, r, 1.0);
  return ldexp(p, (int)n);
}

__device__ __forceinline__ double sem_log(double x) {
  int e;
  double m = frexp(x, &e);
  if (m < qk<true>(0x1.6a09e667f3bcdp-1)) {
    m *= 2.0;
    e -= 1;
  }
  const double sv = (m - 1.0) / (m + 1.0), s2 = sv * sv;
  double p = qk<true>(1.0 / 21.0);
  p = fma(p, s2, qk<true>(1.0 / 19.0));
  p = fma(p, s2, qk<true>(1.0 / 17.0));
  p = fma(p, s2, qk<true>(1.0 / 15.0));
  p = fma(p, s2, qk<true>(1.0 / 13.0));
  p = fma(p, s2, qk<true>(1.0 / 11.0));
  p = fma(p, s2, qk<true>(1.0 / 9.0));
  p = fma(p, s2, qk<true>(1.0 / 7.0));
  p = fma(p, s2, qk<true>(1.0 / 5.0));
  p = fma(p, s2, qk<true>(1.0 / 3.0));
  const double lm = 2.0 * fma(sv * s2, p, sv);
  const double de = (double)e;
  return fma(de, qk<true>(0x1.62e42fefa39efp-1), fma(de, qk<true>(0x1.abc9e3b39803fp-56), lm));
}

// One job of a launch: blocks w0 .. w0 + nw - 1 move electrons j0..j1-1 of its
// walkers, one block per walker (per two, narrow).
struct SemJob {
  const DevSys* sys;
  double* x;
  int64_t* rng;
  void* ainv;
  double* dlogpsi;
  double* nacc;
  double sigma;
  int w0, nw, j0, j1, mm;
  int tile[3];  // threads per row of spins of up to 16, 32, 64 rows
  int narrow;   // two walkers per block of two wavefronts, one each
};
#define SEM_MAX_PACK 16
struct SemJobs {
  SemJob job[SEM_MAX_PACK];
  int njobs;
};

// Moves of jobs of one kind of row (0 real, 1 complex FP64, 2 complex FP32) and
// wavefronts per walker (qmc_sem_moves.hip); nmax: electrons of the largest.
int launch_sem_moves(const SemJobs& jobs, int nblocks, int kind, int waves, bool u3, int nmax, hipStream_t st);
