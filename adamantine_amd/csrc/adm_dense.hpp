// Dense FP64 algebra of the EnKF analysis on the host: LU solve and products
// of small row-major matrices.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <utility>

namespace adm {

// The dense algebra of an analysis (64 members, 500 observations: 2.1 of its
// 2.2 ms before, with strided sums and a division per product; the whole
// analysis 0.89 ms now), written so that every inner loop runs
// over contiguous values of independent entries; each function has a body
// for any x86-64 and one for AVX2 with FMA (chosen when it runs).
#define ADM_BODY static inline __attribute__((always_inline))

// y -= f x, each with one rounding in both bodies: without the instruction
// the C library's fma gives the same bits, so that an analysis does not depend
// on the processor (LU of 200 rows, 32 right-hand sides: 0.87 ms with AVX2 and
// FMA, 11.6 ms in the plain body; the server processors beside this GPU have
// both)
ADM_BODY void axmy(size_t n, double f, const double *__restrict__ x,
                   double *__restrict__ y) {
  for (size_t k = 0; k < n; ++k) y[k] = __builtin_fma(-f, x[k], y[k]);
}

// (these two are not inlined: rare, beside the loops over rows below)
static __attribute__((noinline)) int all_finite(size_t n, const double *x) {
  for (size_t k = 0; k < n; ++k)
    if (!std::isfinite(x[k])) return 0;
  return 1;
}
// y -= f x with f = 0: not a number where x is not finite
static __attribute__((noinline)) void subtract_zero_times(
    size_t n, double f, const double *x, double *y) {
  for (size_t k = 0; k < n; ++k) y[k] = __builtin_fma(-f, x[k], y[k]);
}

// LU with partial pivoting: A X = B with B m x nrhs, both row-major and
// overwritten. False if a pivot is zero.
ADM_BODY bool lu_body(int m, double *A, int nrhs, double *B) {
  const size_t M = m, R = nrhs;
  for (size_t c = 0; c < M; ++c) {
    size_t pr = c;
    for (size_t r = c + 1; r < M; ++r)
      if (std::fabs(A[r * M + c]) > std::fabs(A[pr * M + c])) pr = r;
    if (A[pr * M + c] == 0.0) return false;
    if (pr != c) {
      for (size_t k = 0; k < M; ++k) std::swap(A[c * M + k], A[pr * M + k]);
      for (size_t k = 0; k < R; ++k) std::swap(B[c * R + k], B[pr * R + k]);
    }
    const double inv = 1.0 / A[c * M + c];
    int finite = -1;  // of B's row c; -1: not looked at yet
    for (size_t r = c + 1; r < M; ++r) {
      const double f = A[r * M + c] * inv;
      if (f == 0.0) {
        // B's row stays as it is, unless row c holds a value that is not
        // finite (a non-finite innovation must reach every gain)
        if (finite < 0) finite = all_finite(R, B + c * R);
        if (!finite) subtract_zero_times(R, f, B + c * R, B + r * R);
        continue;
      }
      axmy(M - c - 1, f, A + c * M + c + 1, A + r * M + c + 1);
      axmy(R, f, B + c * R, B + r * R);
    }
  }
  for (size_t r = M; r-- > 0;) {
    for (size_t k = r + 1; k < M; ++k)
      axmy(R, A[r * M + k], B + k * R, B + r * R);
    const double d = A[r * M + r];
    for (size_t k = 0; k < R; ++k) B[r * R + k] = B[r * R + k] / d;
  }
  return true;
}

// C (p x q, row-major) = sum over k of X[k][a] Y[k][b] (both row-major with
// m rows): rank-one updates, k in order
ADM_BODY void gram_body(int m, int p, const double *X, int q, const double *Y,
                        double *C) {
  std::fill(C, C + (size_t)p * q, 0.0);
  for (int a = 0; a < p; ++a)
    for (int k = 0; k < m; ++k)
      axmy(q, -X[(size_t)k * p + a], Y + (size_t)k * q, C + (size_t)a * q);
}

static bool lu_plain(int m, double *A, int nrhs, double *B) {
  return lu_body(m, A, nrhs, B);
}
static void gram_plain(int m, int p, const double *X, int q, const double *Y,
                       double *C) {
  gram_body(m, p, X, q, Y, C);
}
#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
__attribute__((target("avx2,fma"))) static bool lu_avx2(int m, double *A,
                                                        int nrhs, double *B) {
  return lu_body(m, A, nrhs, B);
}
__attribute__((target("avx2,fma"))) static void gram_avx2(
    int m, int p, const double *X, int q, const double *Y, double *C) {
  gram_body(m, p, X, q, Y, C);
}
static bool has_avx2() {
  static const bool yes =
      __builtin_cpu_supports("avx2") && __builtin_cpu_supports("fma");
  return yes;
}
#else
#define lu_avx2 lu_plain
#define gram_avx2 gram_plain
static bool has_avx2() { return false; }
#endif

// Whether every off-diagonal entry of an m x m row-major matrix is zero (a
// value that is not a number is not). Without a branch in a row: with one per
// entry an analysis of 2 members and 400 observations took 115 us, 139 once
// the code around it had changed, and takes 85 so.
static __attribute__((noinline)) bool is_diagonal(int m, const double *R) {
  for (int a = 0; a < m; ++a) {
    const double *row = R + (size_t)a * m;
    int other = 0;
    for (int b = 0; b < a; ++b) other |= row[b] != 0.0;
    for (int b = a + 1; b < m; ++b) other |= row[b] != 0.0;
    if (other) return false;
  }
  return true;
}

#undef ADM_BODY

}  // namespace adm
