// Device helpers shared by the HIP kernels (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>

namespace snu {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef double d4 __attribute__((ext_vector_type(4)));
// Pointers read from launch descriptors are generic; casting them to the
// global address space makes the compiler emit global_load/global_store
// (flat accesses also count against lgkmcnt, which would make every LDS wait
// drain the global prefetch as well).
typedef __attribute__((address_space(1))) const double gcdouble;
typedef __attribute__((address_space(1))) double gdouble;
__device__ __forceinline__ gcdouble *gptr(const double *p) { return (gcdouble *)p; }
__device__ __forceinline__ gdouble *gptr(double *p) { return (gdouble *)p; }
typedef __attribute__((address_space(1))) const float gcfloat;
typedef __attribute__((address_space(1))) float gfloat;
typedef __attribute__((address_space(1))) const long long gcint64;
__device__ __forceinline__ gcint64 *gptr(const long long *p) { return (gcint64 *)p; }
typedef __attribute__((address_space(1))) const int gcint;
__device__ __forceinline__ gcint *gptr(const int *p) { return (gcint *)p; }
__device__ __forceinline__ gcfloat *gptr(const float *p) { return (gcfloat *)p; }
__device__ __forceinline__ gfloat *gptr(float *p) { return (gfloat *)p; }

__device__ __forceinline__ int rl(int v, int l) {
  return __builtin_amdgcn_readlane(v, l);
}
__device__ __forceinline__ double rld(double v, int l) {
  long long x = __double_as_longlong(v);
  int lo = rl((int)(x & 0xffffffffLL), l);
  int hi = rl((int)(x >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ float rld(float v, int l) {
  return __int_as_float(rl(__float_as_int(v), l));
}

}  // namespace snu
