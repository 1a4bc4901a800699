// FP64 Boys values from a table about nodes BOYSD_H apart (rows of an LDS copy,
// eri_pairs.h).  Needs no HIP, so that it can be compiled and run on a host.
#pragma once
#include <math.h>

namespace pscf {

constexpr int BOYSD_NT = 200, BOYSD_TERMS = 10, BOYSD_COLS = BOYSD_TERMS + 2;
constexpr double BOYSD_H = 0.2;
constexpr double BOYS_EDGE = 39.9;  // the tables serve arguments below, the asymptote from here on

__device__ constexpr double INV_FACT[11] = {1.0,       1.0,        1.0 / 2,     1.0 / 6,      1.0 / 24,     1.0 / 120,
                                            1.0 / 720, 1.0 / 5040, 1.0 / 40320, 1.0 / 362880, 1.0 / 3628800};

// Row for an argument of at most BOYS_EDGE.  The edge lies half a node past the
// last row and rounds to one more, which there is not.
__device__ __forceinline__ int boysd_node(double t) {
  const int i = (int)(t * (1.0 / BOYSD_H) + 0.5);
  return i < BOYSD_NT - 1 ? i : BOYSD_NT - 1;
}

// F_0 .. F_L from the table; t is clamped to it.
template <int L>
__device__ __forceinline__ void ep_boys(double t, const double* __restrict__ tab, double* f) {
  t = fmin(t, BOYS_EDGE);
  const int i = boysd_node(t);
  const double d = (double)i * BOYSD_H - t;
  const double* c = tab + i * BOYSD_COLS;
  double a = c[BOYSD_TERMS];
#pragma unroll
  for (int k = BOYSD_TERMS; k > 0; --k) a = fma(a, d, c[k - 1]);
  f[L] = a;
  if constexpr (L > 0) {
    double e = INV_FACT[9];  // exp(d), |d| <= 0.1
#pragma unroll
    for (int k = 8; k >= 0; --k) e = fma(e, d, INV_FACT[k]);
    e *= c[BOYSD_TERMS + 1];
#pragma unroll
    for (int m = L; m > 0; --m) f[m - 1] = fma(t + t, f[m], e) * (1.0 / (2 * m - 1));
  }
}

}  // namespace pscf
