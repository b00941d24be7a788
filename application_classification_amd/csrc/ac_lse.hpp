// Log-sum-exp accumulators (ac::Lse, value = m + log1p(t)) shared by the fused kernels and the stage operators.
#pragma once

#include <hip/hip_runtime.h>

#include "ac_internal.hpp"

namespace ac {

// One exp per value and no branches: the exponent is always min - max of (x, m), which rescales t when x is a new
// maximum and is the new term otherwise.  exp(-inf) = 0 covers the empty accumulator.  min - max is formed as
// -|x - m|: rounding to nearest is sign-symmetric, so fl(min - max) = -|fl(x - m)| exactly, and x > m exactly when
// fl(x - m) > 0 (the difference of two distinct finite doubles never rounds to zero; m = -inf gives +inf).
__device__ __forceinline__ void lse_add(Lse& s, double x) {
  const bool valid = x != -__builtin_huge_val();
  const double d = x - s.m;  // NaN only for x = m = -inf, which is not valid
  const double e = (double)__expf((float)(-fabs(d)));
  const double t = d > 0.0 ? (1.0 + s.t) * e : s.t + e;
  s.t = valid ? t : s.t;
  s.m = valid ? fmax(x, s.m) : s.m;
}

// lse_add for a finite x (no -inf term to skip): the same result with fewer selects.  An empty accumulator
// (m = -inf) takes x as its maximum: exp(-inf) = 0 clears t.
__device__ __forceinline__ void lse_add_finite(Lse& s, double x) {
  const double d = x - s.m;
  const double e = (double)__expf((float)(-fabs(d)));
  s.t = d > 0.0 ? (1.0 + s.t) * e : s.t + e;
  s.m = fmax(x, s.m);
}

__device__ __forceinline__ Lse lse_merge(Lse a, Lse b) {
  if (b.m == -__builtin_huge_val()) return a;
  if (a.m == -__builtin_huge_val()) return b;
  if (a.m >= b.m) {
    a.t += (1.0 + b.t) * exp(b.m - a.m);
    return a;
  }
  b.t += (1.0 + a.t) * exp(a.m - b.m);
  return b;
}

// lse_merge with the exponential of the two maxima's difference in FP32 (__expf), as lse_add forms each term: for merges
// in a kernel's inner loop, where the FP64 exp would dominate.  The merged t keeps a relative error of about 1e-7.
__device__ __forceinline__ Lse lse_merge_fast(Lse a, Lse b) {
  if (b.m == -__builtin_huge_val()) return a;
  if (a.m == -__builtin_huge_val()) return b;
  if (a.m >= b.m) {
    a.t += (1.0 + b.t) * (double)__expf((float)(b.m - a.m));
    return a;
  }
  b.t += (1.0 + a.t) * (double)__expf((float)(a.m - b.m));
  return b;
}

// Merging many accumulators at once: M the largest of their maxima, then every accumulator's terms rescaled to M (one
// exponential each, independent of each other), then their sum, which leaves out one maximal element.
// lse_rescaled is an accumulator's share: (1 + t) exp(m - M), or, where its own maximum is M, -t: the sign bit (also of
// -0.0) marks a share whose maximal element is not counted.  lse_sum_step adds a share in order; seen: a maximal element
// has been left out already, so the next one counts.
__device__ __forceinline__ double lse_rescaled(const Lse& s, double M) {
  if (s.m == -__builtin_huge_val()) return 0.0;
  return s.m == M ? -s.t : (1.0 + s.t) * exp(s.m - M);
}

__device__ __forceinline__ void lse_sum_step(double& sum, bool& seen, double share) {
  if (signbit(share)) {
    sum += seen ? 1.0 - share : -share;
    seen = true;
  } else {
    sum += share;
  }
}

// One accumulator per lane over groups of `width` lanes (a power of two): every lane gets its group's.
__device__ __forceinline__ Lse lanes_lse_merge(const Lse& s, int width) {
  const int lane = threadIdx.x & 63;
  double M = s.m;
  for (int o = width >> 1; o > 0; o >>= 1) M = fmax(M, __shfl_xor(M, o, 64));
  unsigned long long holders = __ballot(s.m == M);
  if (width < 64) holders &= ((1ull << width) - 1ull) << (lane & ~(width - 1));
  double x = lse_rescaled(s, M);
  if (signbit(x)) x = lane == __ffsll((long long)holders) - 1 ? -x : 1.0 - x;
  for (int o = width >> 1; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
  return Lse{M, x};
}

// The largest m over a block of NT threads, in every thread.  sh: NT / 64 doubles, free when it returns.
template <int NT>
__device__ __forceinline__ double block_max(double m, double* sh) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = m;
  __syncthreads();
  m = sh[0];
#pragma unroll
  for (int w = 1; w < NT / 64; ++w) m = fmax(m, sh[w]);
  __syncthreads();
  return m;
}

// The sum of every thread's shares (lse_sum_step's sum and seen) over a block, in thread 0.  sh: NT / 32 doubles.
template <int NT>
__device__ __forceinline__ double block_lse_sum(double sum, bool seen, double* sh) {
  const int lane = threadIdx.x & 63;
  const unsigned long long holders = __ballot(seen);
  if (seen && lane != __ffsll((long long)holders) - 1) sum += 1.0;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
  if (lane == 0) {
    sh[threadIdx.x >> 6] = sum;
    sh[NT / 64 + (threadIdx.x >> 6)] = holders ? 1.0 : 0.0;
  }
  __syncthreads();
  double a = sh[0];
  bool any = sh[NT / 64] != 0.0;
#pragma unroll
  for (int w = 1; w < NT / 64; ++w) {
    a += sh[w];
    if (sh[NT / 64 + w] != 0.0) {
      if (any) a += 1.0;
      any = true;
    }
  }
  return a;
}

__device__ __forceinline__ Lse lse_empty() { return Lse{-__builtin_huge_val(), 0.0}; }

}  // namespace ac
