// Just enough of the HIP device language to run a kernel's bookkeeping on the
// host, one lane of one workgroup at a time: collectives across lanes see
// zeros from the other lanes, barriers do nothing.  Found before the real
// header by the tests that compile kernel sources for the CPU.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstring>

#define __global__
#define __device__
#define __host__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __shared__ thread_local
#define __align__(n) alignas(n)
struct int2 {
  int x, y;
};
struct int4 {
  int x, y, z, w;
};
struct double2 {
  double x, y;
};
struct float2 {
  float x, y;
};
struct dim3 {
  unsigned x = 1, y = 1, z = 1;
};
inline int2 make_int2(int x, int y) { return {x, y}; }
inline int4 make_int4(int x, int y, int z, int w) { return {x, y, z, w}; }
inline double2 make_double2(double x, double y) { return {x, y}; }
using hipStream_t = void*;
using hipEvent_t = void*;
using hipGraphExec_t = void*;
inline dim3 threadIdx{0, 0, 0}, blockIdx{0, 0, 0}, blockDim, gridDim;

inline void __syncthreads() {}
template <class T>
T __shfl_xor(T, int, int = 64) { return T(); }
template <class T>
T __shfl(T v, int, int = 64) { return v; }
template <class T>
T __shfl_down(T, int, int = 64) { return T(); }
inline unsigned long long __ballot(int p) { return p ? 1ull : 0ull; }
template <class T>
T atomicMax(T* p, T v) {
  const T o = *p;
  if (v > o) *p = v;
  return o;
}
template <class T>
T atomicMin(T* p, T v) {
  const T o = *p;
  if (v < o) *p = v;
  return o;
}
template <class T>
T atomicAdd(T* p, T v) {
  const T o = *p;
  *p += v;
  return o;
}
inline double __longlong_as_double(long long v) {
  double d;
  std::memcpy(&d, &v, 8);
  return d;
}
inline long long __double_as_longlong(double d) {
  long long v;
  std::memcpy(&v, &d, 8);
  return v;
}
#define amdgpu_waves_per_eu(...)
#define __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, x, y, z) (c)
#define __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, x, y, z) (c)
#define __builtin_amdgcn_update_dpp(o, s, c, r, b, f) (o)
#define __builtin_amdgcn_rcp(x) (1.0 / (x))
#define __builtin_amdgcn_rsq(x) (1.0 / std::sqrt(x))
#define __builtin_amdgcn_s_memrealtime() 0ull
using std::fabs;
using std::fmax;
using std::fmin;
using std::isfinite;
using std::max;
using std::min;
