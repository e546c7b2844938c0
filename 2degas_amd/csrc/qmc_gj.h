// qmc_gj.h -- what the augmented eliminations of qmc_gjr.hip (real orbitals) and
// qmc_gjc.hip (complex ones) share.
#pragma once
#include <type_traits>

#include "qmc_dev.h"

typedef double gr_d4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ gr_d4 gr_mfma(double a, double b, gr_d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// 1/d: hardware reciprocal and two Newton steps.
__device__ __forceinline__ double gr_rcp(double d) {
  double y = __builtin_amdgcn_rcp(d);
  double e = fma(-d, y, 1.0);
  y = fma(y, e, y);
  e = fma(-d, y, 1.0);
  return fma(y, e, y);
}

// LDS traffic between lanes of one wavefront.
__device__ __forceinline__ void gr_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Element i (uniform, run time) of a lane's 4 NT values of a part: register
// index mode on a tuple of 8 or 16 values, where a switch is a dozen branches.
typedef double gr_d8 __attribute__((ext_vector_type(8)));
typedef double gr_d16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ double gr_pick4(const gr_d4& a, int i) {
  const double x = i & 1 ? a[1] : a[0], y = i & 1 ? a[3] : a[2];
  return i & 2 ? y : x;
}
template <int NT>
__device__ __forceinline__ double gr_pick(const gr_d4 (&a)[NT], int i) {
  if constexpr (NT == 1) {
    return gr_pick4(a[0], i);
  } else if constexpr (NT == 2) {
    const gr_d8 v = __builtin_shufflevector(a[0], a[1], 0, 1, 2, 3, 4, 5, 6, 7);
    return v[i];
  } else {
    const gr_d8 v = __builtin_shufflevector(a[0], a[1], 0, 1, 2, 3, 4, 5, 6, 7);
    const gr_d8 w = __builtin_shufflevector(a[2], a[NT == 3 ? 2 : 3], 0, 1, 2, 3, 4, 5, 6, 7);
    const gr_d16 x = __builtin_shufflevector(v, w, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
    return x[i];
  }
}
