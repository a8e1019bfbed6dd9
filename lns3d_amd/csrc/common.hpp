// Shared device helpers for the LNS3D implicit-step kernels (gfx950).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

namespace lns3d {

// complex value with explicit real/imag parts; T = double or float
template <typename T> struct cx {
  T re, im;
};

template <typename T> __host__ __device__ __forceinline__ cx<T> operator+(cx<T> a, cx<T> b) { return {a.re + b.re, a.im + b.im}; }
template <typename T> __host__ __device__ __forceinline__ cx<T> operator-(cx<T> a, cx<T> b) { return {a.re - b.re, a.im - b.im}; }
template <typename T> __host__ __device__ __forceinline__ cx<T> operator-(cx<T> a) { return {-a.re, -a.im}; }
template <typename T> __host__ __device__ __forceinline__ cx<T> operator*(cx<T> a, cx<T> b) {
  return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
template <typename T> __host__ __device__ __forceinline__ cx<T> operator*(T s, cx<T> b) { return {s * b.re, s * b.im}; }
// acc + a*b
template <typename T> __host__ __device__ __forceinline__ cx<T> cfma(cx<T> a, cx<T> b, cx<T> acc) {
  acc.re = fma(a.re, b.re, acc.re);
  acc.re = fma(-a.im, b.im, acc.re);
  acc.im = fma(a.re, b.im, acc.im);
  acc.im = fma(a.im, b.re, acc.im);
  return acc;
}
// a*b with one rounding fewer per part than the textbook form
template <typename T> __host__ __device__ __forceinline__ cx<T> cmul(cx<T> a, cx<T> b) {
  T re = fma(a.re, b.re, -(a.im * b.im));
  T im = fma(a.re, b.im, a.im * b.re);
  return {re, im};
}
// a / b, Smith's algorithm (Smith, CACM 5(8), 1962)
template <typename T> __host__ __device__ __forceinline__ cx<T> cdiv(cx<T> a, cx<T> b) {
  if (fabs(b.re) >= fabs(b.im)) {
    T r = b.im / b.re, d = b.re + b.im * r;
    return {(a.re + a.im * r) / d, (a.im - a.re * r) / d};
  }
  T r = b.re / b.im, d = b.re * r + b.im;
  return {(a.re * r + a.im) / d, (a.im * r - a.re) / d};
}
template <typename T> __host__ __device__ __forceinline__ cx<T> crecip(cx<T> b) {
  return cdiv(cx<T>{T(1), T(0)}, b);
}

// The chip places workgroup b of a launch on XCD b % 8 (round robin over its
// eight XCDs, each with its own L2).  xcd_tile(b, nb) numbers the tiles so
// that each XCD works through a contiguous range of them (a bijection of
// [0, nb)): neighbouring tiles, which share stencil rows, share an L2.
__device__ __forceinline__ long xcd_tile(long b, long nb) {
  const long q = nb / 8, r = nb % 8, x = b % 8, k = b / 8;
  return x * q + (x < r ? x : r) + k;
}
// orders the LDS accesses of one wave before / after it (lanes of the wave
// exchanging values through LDS)
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The workgroup barrier of waves with copies in flight: their LDS accesses
// are complete (lgkmcnt 0) but the copies (or loads into registers) are not
// waited for, as a __syncthreads fence would (it treats global_load_lds as
// pending LDS writes).  The empty asm statements keep the compiler from moving memory
// accesses across the barrier.
__device__ __forceinline__ void loader_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);     // lgkmcnt(0); vmcnt, expcnt not waited for
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// finite-difference coefficient tables of the scheme (src/stencil.f90)
namespace st {
constexpr double ga1 = 8.333333333333333333333E-02, ga2 = -6.666666666666666666667E-01,
                 ga3 = 6.666666666666666666667E-01, ga4 = -8.333333333333333333333E-02;
constexpr double gc1 = -2.083333333333333333333E+00, gc2 = 4.000000000000000000000E+00,
                 gc3 = -3.000000000000000000000E+00, gc4 = 1.333333333333333333333E+00,
                 gc5 = -2.500000000000000000000E-01;
constexpr double gb1 = -2.500000000000000000000E-01, gb2 = -8.333333333333333333333E-01,
                 gb3 = 1.500000000000000000000E+00, gb4 = -5.000000000000000000000E-01,
                 gb5 = 8.333333333333333333333E-02;
constexpr double da1 = -8.333333333333333333333E-02, da2 = 1.333333333333333333333E+00,
                 da3 = -2.500000000000000000000E+00, da4 = 1.333333333333333333333E+00,
                 da5 = -8.333333333333333333333E-02;
constexpr double db1 = 9.166666666666666666667E-01, db2 = -1.666666666666666666667E+00,
                 db3 = 5.000000000000000000000E-01, db4 = 3.333333333333333333333E-01,
                 db5 = -8.333333333333333333333E-02;
constexpr double dd1 = 2.916666666666666666667E+00, dd2 = -8.666666666666666666667E+00,
                 dd3 = 9.500000000000000000000E+00, dd4 = -4.666666666666666666667E+00,
                 dd5 = 9.166666666666666666667E-01;
constexpr double pt66 = 6.6666666666666666666e-1;
}  // namespace st

#define LNS3D_CHECK(expr)                                                        \
  do {                                                                           \
    hipError_t e_ = (expr);                                                      \
    if (e_ != hipSuccess) return lns3d::set_error(__FILE__, __LINE__, hipGetErrorString(e_)); \
  } while (0)

int set_error(const char *file, int line, const char *msg);

}  // namespace lns3d
