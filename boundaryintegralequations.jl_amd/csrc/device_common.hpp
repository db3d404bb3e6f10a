// Device helpers shared by the assembly kernels (gfx950).
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

namespace bie {
namespace {

// Workgroup barrier for LDS hand-offs only: waits for this wave's LDS (and scalar-load)
// operations, then s_barrier.  Unlike __syncthreads() it does not wait for outstanding
// global loads and stores, so prefetched table rows and the column stores of F and G stay
// in flight across it; nothing in global memory is exchanged between the waves of a
// workgroup through these barriers.  The memory clobber keeps the compiler from moving
// memory accesses across it.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Wave-uniform read of read-only data (the host-built slot schedules) through the scalar
// data cache: the load goes to an SGPR and is counted by lgkmcnt.  A vector load of the
// same value would be counted by vmcnt, which on gfx9-family GPUs retires loads and stores
// in issue order, so waiting for it would also wait for every column store issued before
// it.  Only for addresses that are the same in all active lanes and memory the kernel
// never writes.
template <class T>
__device__ __forceinline__ T sload(const T* p) {
  return *reinterpret_cast<const __attribute__((address_space(4))) T*>(
      reinterpret_cast<uintptr_t>(p));
}

// Two doubles as one 16-byte vector: a complex entry's (re, im) written by one store.
typedef double d2v __attribute__((ext_vector_type(2)));

// Julia Base n-ary hypot for Float64 (maxabs * sqrt(sum((x_i/maxabs)^2)), left to
// right), with no fused multiply-add so that the result is bit-identical to the CPU.
__device__ __forceinline__ double julia_hypot3_inline(double x, double y, double z) {
#pragma clang fp contract(off)
  const double ax = fabs(x), ay = fabs(y), az = fabs(z);
  if (isinf(ax) || isinf(ay) || isinf(az)) return INFINITY;
  if (isnan(ax) || isnan(ay) || isnan(az)) return NAN;
  double mx = ax > ay ? ax : ay;
  mx = mx > az ? mx : az;
  if (mx == 0.0) return mx;
  const double a = ax / mx, b = ay / mx, c = az / mx;
  double s = a * a;
  s = s + b * b;
  s = s + c * c;
  return mx * sqrt(s);
}

__device__ __noinline__ double julia_hypot3(double x, double y, double z) {
  return julia_hypot3_inline(x, y, z);
}

// The n-ary hypot that later Julia releases use for IEEE floats: the arguments scaled by
// 2^-E with E the exponent of maxabs (clamped to the normal range), squared and summed left
// to right, square-rooted and scaled back by 2^E.  The scalings are exact, so away from overflow and underflow this is
// sqrt((x^2 + y^2) + z^2) with every operation rounded once; no fused multiply-add, so the
// result is bit-identical to the CPU.
__device__ __forceinline__ double scaled_hypot3_inline(double x, double y, double z) {
#pragma clang fp contract(off)
  const double ax = fabs(x), ay = fabs(y), az = fabs(z);
  if (isinf(ax) || isinf(ay) || isinf(az)) return INFINITY;
  if (isnan(ax) || isnan(ay) || isnan(az)) return NAN;
  double mx = ax > ay ? ax : ay;
  mx = mx > az ? mx : az;
  if (mx == 0.0) return mx;
  int e = 0;
  (void)frexp(mx, &e);  // 2^E <= mx < 2^(E+1) with E = e - 1, clamped to the normal range
  const int E = max(-1022, min(1022, e - 1));
  const double inv = ldexp(1.0, -E), scale = ldexp(1.0, E);
  const double a = ax * inv, b = ay * inv, c = az * inv;
  double s = a * a;
  s = s + b * b;
  s = s + c * c;
  return scale * sqrt(s);
}

__device__ __noinline__ double scaled_hypot3(double x, double y, double z) {
  return scaled_hypot3_inline(x, y, z);
}

// 1-based rule index of the node nearest to x (first strict minimum of the Julia hypot
// distance; hyp 0: julia_hypot3, 1: scaled_hypot3).  A squared-distance filter decides
// every pair whose two nearest nodes are separated by more than 1e-12 relative (far beyond
// the few-ulp error of either distance, so the exact argmin is the same under either
// formula); near ties, zero, inf and NaN distances go through the exact sequence.  Index 0
// (no distance below Inf) maps to the last rule, as the reference's if/elseif chain does.
template <int NP>
__device__ __forceinline__ int select_rule(double x0, double x1, double x2,
                                           const double* __restrict__ P, int R, int hyp) {
  // quadrilaterals (node counts other than 3 and 6): one rule, nothing to select
  if (NP != 3 && NP != 6 && R == 1) return 1;
  double d2[NP];
#pragma unroll
  for (int s = 0; s < NP; ++s) {
    const double dx = P[4 * s] - x0, dy = P[4 * s + 1] - x1, dz = P[4 * s + 2] - x2;
    d2[s] = fma(dx, dx, fma(dy, dy, dz * dz));
  }
  int jb = 0;
  double b = d2[0];
#pragma unroll
  for (int s = 1; s < NP; ++s)
    if (d2[s] < b) {
      b = d2[s];
      jb = s;
    }
  const double lim = b * (1.0 + 1e-12);
  bool ok = (b <= 1.0e300);
#pragma unroll
  for (int s = 0; s < NP; ++s)
    if (s != jb && !(d2[s] > lim)) ok = false;
  int c;
  if (ok) {
    c = jb + 1;
  } else {
    double best = INFINITY;
    int idx = 0;
    for (int s = 0; s < NP; ++s) {
      const double dx = P[4 * s] - x0, dy = P[4 * s + 1] - x1, dz = P[4 * s + 2] - x2;
      const double d = hyp ? scaled_hypot3(dx, dy, dz) : julia_hypot3(dx, dy, dz);
      if (d < best) {
        best = d;
        idx = s + 1;
      }
    }
    c = idx;
  }
  if (c < 1 || c > R) c = R;
  return c;
}

}  // namespace
}  // namespace bie
