// Device helpers shared by the HIP kernels (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

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

// lane K's value in each group of 16 lanes
template <int K>
__device__ __forceinline__ float bcast16(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x150 + K, 0xf, 0xf, false));
}
template <int K>
__device__ __forceinline__ double bcast16(double v) {
  return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), 0x150 + K, 0xf, 0xf, false),
                          __builtin_amdgcn_mov_dpp(__double2loint(v), 0x150 + K, 0xf, 0xf, false));
}

// frexp, reciprocal, ldexp and division fixup in both precisions
__device__ __forceinline__ double frexp_m(double x) { return __builtin_amdgcn_frexp_mant(x); }
__device__ __forceinline__ float frexp_m(float x) { return __builtin_amdgcn_frexp_mantf(x); }
__device__ __forceinline__ int frexp_e(double x) { return __builtin_amdgcn_frexp_exp(x); }
__device__ __forceinline__ int frexp_e(float x) { return __builtin_amdgcn_frexp_expf(x); }
__device__ __forceinline__ double recip(double x) { return __builtin_amdgcn_rcp(x); }
__device__ __forceinline__ float recip(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ double scale2(double x, int e) { return __builtin_amdgcn_ldexp(x, e); }
__device__ __forceinline__ float scale2(float x, int e) { return __builtin_amdgcn_ldexpf(x, e); }
__device__ __forceinline__ double div_special(double q, double d, double a) { return __builtin_amdgcn_div_fixup(q, d, a); }
__device__ __forceinline__ float div_special(float q, float d, float a) { return __builtin_amdgcn_div_fixupf(q, d, a); }
// Quotients by one divisor with one reciprocal: a few Newton steps on its
// mantissa, and per quotient corrections by the exact remainder in FMA
// (Markstein's division).  The dividend is scaled by the divisor's exponent
// first, so that nothing on the way overflows where the quotient does not (a
// dividend beyond half the largest value did, taken whole).  Rounded as by a
// division while remainders are normal numbers (quotients above 2^-969, FP32
// 2^-101), within an ulp below.
template <typename T>
struct Divisor {
  T m, r;  // mantissa, its reciprocal
  int e;   // exponent
  __device__ __forceinline__ explicit Divisor(T d) : m(frexp_m(d)), e(frexp_e(d)) {
    r = recip(m);
    r = fma(fma(-m, r, T(1)), r, r);
    if constexpr (std::is_same<T, double>::value) r = fma(fma(-m, r, T(1)), r, r);
  }
  __device__ __forceinline__ T quotient(T a) const {
    const T n = scale2(a, -e);
    T q = n * r;
    q = fma(fma(-m, q, n), r, q);
    if constexpr (std::is_same<T, float>::value) q = fma(fma(-m, q, n), r, q);
    return div_special(q, m, n);
  }
};

// A pivot of a substitution: its reciprocal in two parts, whose product with the
// dividend has a division's rounding (to a few 2^-100) in two dependent
// operations, and its scale.  The dividend v - s is scaled by the pivot's
// exponent as it is formed, so that nothing on the way overflows where the
// quotient does not.  (Where a division gives an infinity: any value that is
// not finite.)
template <typename T>
struct Pivot {
  T r, lo;  // 1 / (pivot 2^-e)
  T neg;    // -2^-e
  Pivot() = default;
  __device__ __forceinline__ explicit Pivot(T d) {
    const int e = max(frexp_e(d), std::is_same<T, double>::value ? -1021 : -125);  // (2^-e is finite)
    const T m = scale2(d, -e);
    r = recip(m);
    r = fma(fma(-m, r, T(1)), r, r);
    if constexpr (std::is_same<T, double>::value) r = fma(fma(-m, r, T(1)), r, r);
    lo = fma(-m, r, T(1)) * r;
    neg = -scale2(T(1), -e);
  }
  __device__ __forceinline__ T scaled(T v) const { return -(v * neg); }
  // (v - s) / pivot, v scaled
  __device__ __forceinline__ T solve(T v, T s) const {
    const T n = fma(s, neg, v);
    return fma(n, r, n * lo);
  }
  // lane l's
  __device__ __forceinline__ Pivot of_lane(int l) const {
    Pivot p;
    p.r = rld(r, l), p.lo = rld(lo, l), p.neg = rld(neg, l);
    return p;
  }
};
// Of group G (of the four groups of 16 lanes) s[i], in group i, by permlane
// swaps (VALU, no LDS).
template <int G>
__device__ __forceinline__ unsigned spread_words(const unsigned (&x)[4]) {
  const auto a = __builtin_amdgcn_permlane16_swap(x[0], x[1], false, false);
  const auto b = __builtin_amdgcn_permlane16_swap(x[2], x[3], false, false);
  const auto p = __builtin_amdgcn_permlane32_swap(a[G & 1], b[G & 1], false, false);
  return p[G >> 1];
}
template <int G>
__device__ __forceinline__ float spread_group(const float (&s)[4]) {
  unsigned x[4];
#pragma unroll
  for (int i = 0; i < 4; i++) x[i] = __float_as_uint(s[i]);
  return __uint_as_float(spread_words<G>(x));
}
template <int G>
__device__ __forceinline__ double spread_group(const double (&s)[4]) {
  unsigned lo[4], hi[4];
#pragma unroll
  for (int i = 0; i < 4; i++) lo[i] = __double2loint(s[i]), hi[i] = __double2hiint(s[i]);
  return __hiloint2double((int)spread_words<G>(hi), (int)spread_words<G>(lo));
}

// MFMA fragments, 16x16x4 products.  A 16 x 16 block of a vector group (16 rows, 16 columns)
// is one fragment: register r of lane l holds row frag_row(r), column l % 16,
// which is both the layout the product leaves its result in and, taking the
// four rows of register r as one K step, the layout of its second operand.  So
// results feed the next product without passing through LDS; the first
// operand's K columns follow the same frag_row order.
template <typename T>
using Frag = T __attribute__((ext_vector_type(4)));
template <typename T>
__device__ __forceinline__ int frag_row(int r, int lk) {
  return std::is_same<T, double>::value ? 4 * r + lk : 4 * lk + r;
}
__device__ __forceinline__ Frag<double> mfma4(double a, double b, Frag<double> c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ Frag<float> mfma4(float a, float b, Frag<float> c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
template <typename T>
__device__ __forceinline__ Frag<T> frag_zero() {
  return Frag<T>{T(0), T(0), T(0), T(0)};
}

}  // namespace snu
