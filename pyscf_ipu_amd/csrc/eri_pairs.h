// Packed s8 ERIs from shell-pair primitive lists (McMurchie-Davidson), the
// engine of pscf_eri_s8 and, in FP32, of the batched entries.
//
// The ERI work is bound by VALU issue, so the layout removes what a
// lane-per-contracted-quartet Rys form spends beyond the arithmetic itself:
//   * a workgroup takes a tile of bra shell pairs x ket shell pairs of one
//     angular class and computes every primitive pair of both sides once (the
//     exponential included), in FP64, into LDS; primitive pairs with a
//     negligible Gaussian-product prefactor are dropped there;
//   * lane = ket PRIMITIVE pair (whole shell pairs packed into 64-lane chunks),
//     the bra primitive pairs of one shell pair a wave-uniform loop: no lane
//     waits for another quartet's longer contraction;
//   * the integral is sum_h1 E_bra[h1] sum_h2 E_ket[h2] (-1)^|h2| R[h1 + h2]
//     over Hermite Gaussians: only Boys values and R are per primitive quartet,
//     no Rys roots (whose FP64 Hankel solve, acos and cos were most of the
//     p-class time).  The bra expansion goes into the inner loop, the ket
//     expansion after it, once per (bra pair, ket primitive);
//   * the sum over a ket pair's primitives is a segmented sum through LDS whose
//     outputs are spread over all lanes, so the scattered s8 stores are too.
// The results do not depend on the tile shape, the grid or the schedule.
// Measured against the lane-per-quartet Rys kernels: one 9-heavy-atom STO-3G
// molecule in FP64 449 -> 218 us, one 12-heavy-atom 6-31G molecule in FP32
// 16.5 -> 0.84 ms (its contractions, 1 to 36 primitives a pair, had diverged in
// a wave) and in FP64 26 -> 2.1 ms, 1024 nine-heavy-atom molecules in FP32 127
// -> 51 ms.  What bounds it now is VALU issue: about 33 (ss|ss) to 520 (pp|pp)
// instructions per primitive quartet at about two thirds of the issue rate, the
// rest staging, segmented sums and the ends of tiles.
#pragma once
#include "batch.h"
#include "boys_fp64.h"
#include "common.h"
#include "wave.h"

namespace pscf {

// Primitive pairs with |c_a c_b| exp(-mu R^2) / p below this are dropped.  A
// dropped pair adds at most 34.99 / (4 pi)^2 (angular factors of s shells) x the
// other side's prefactor (below 20 for same-centre 1s pairs) x R^2 for each p
// pair: 4.4e-20 R^2 in FP64 and 4.4e-15 R^2 in FP32, R the molecule's extent in
// Bohr.  At 15 that is 1e-17 and 1e-12 of an ERI of order 1, at 50 1e-16 and
// 1e-11: under the rounding of the types (measured: no change of the error
// against 64 bits).
template <typename T>
struct EpCut;
template <>
struct EpCut<double> {
  static constexpr double v = 1e-20;
};
template <>
struct EpCut<float> {
  static constexpr double v = 1e-15;
};

constexpr int EP_THREADS = 256, EP_WAVES = EP_THREADS / 64;
constexpr int EP_PAIRS = 64;    // shell pairs staged at once (one lane each)
constexpr int EP_RUN = 8;       // bra pairs a wave runs through with one ket chunk
constexpr int EP_CHUNKS = 80;   // 64-lane chunks of the staged ket primitives
constexpr int EP_ROWS = 9;      // values per lane of one segmented sum
constexpr int EP_SUM = 9;       // lanes a segmented sum reads at once
// Primitive pairs staged at once per side.  LDS sets the workgroups per CU:
// three in FP32 (576 kets: two, 1.05 instead of 0.84 ms for a 12-heavy-atom
// 6-31G molecule), two in FP64 (256 kets: one, 0.30 instead of 0.22 ms for a
// 9-heavy-atom STO-3G molecule).
template <typename T>
__host__ __device__ constexpr int ep_cap_ket(int Y) {
  return sizeof(T) == 8 ? 192 : (Y == 2 ? 416 : 448);
}
constexpr int EP_CAP_BRA = 288;

// ------------------------------------------------------------ Boys values ----
// FP32: cubic Taylor about nodes 1/16 apart (error below 2e-8), one 16-byte
// LDS read; FP64: 10 terms about nodes 0.2 apart, with exp(-T_i) beside them
// (19 KB; nodes 0.1 apart with 8 terms take 32 KB and a workgroup per CU), see
// boys_fp64.h.
constexpr int BOYSF_NT = 640, BOYSF_LMAX = 4;
__device__ float4 g_boysf[(BOYSF_LMAX + 1) * BOYSF_NT];

template <typename T>
struct EpTable;
template <>
struct EpTable<float> {
  using type = float4;
  static constexpr int bytes = BOYSF_NT * 16;
};
template <>
struct EpTable<double> {
  using type = double;
  static constexpr int bytes = BOYSD_NT * BOYSD_COLS * 8;
};

__device__ inline float rsq(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ inline double rsq(double x) {  // hardware estimate and one third-order step
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}

// F_0 .. F_L from the table; t is clamped to it.
template <int L>
__device__ __forceinline__ void ep_boys(float t, const float4* __restrict__ tab, float* f) {
  t = fminf(t, (float)BOYS_EDGE);
  const int i = (int)(t * 16.0f + 0.5f);
  const float d = (float)i * 0.0625f - t;
  const float4 c = tab[i];
  f[L] = c.x + d * (c.y + d * (c.z + d * c.w));
  if constexpr (L > 0) {
    const float e = __builtin_amdgcn_exp2f(-1.44269504f * t), t2 = t + t;
#pragma unroll
    for (int m = L; m > 0; --m) f[m - 1] = (t2 * f[m] + e) * (1.0f / (2 * m - 1));
  }
}
// F_0 = sqrt(pi / t) / 2 and upward recursion past the tables.
template <int L, typename T>
__device__ __forceinline__ void ep_boys_tail(T t, T* f) {
  const T s = rsq(t), inv = s * s;
  f[0] = T(0.88622692545275801365) * s;
#pragma unroll
  for (int m = 0; m < L; ++m) f[m + 1] = f[m] * T(m + 0.5) * inv;
}

template <int L>
__device__ inline void ep_stage_table(float4* tab, const double*) {
  for (int i = threadIdx.x; i < BOYSF_NT; i += EP_THREADS) tab[i] = g_boysf[L * BOYSF_NT + i];
}
template <int L>
__device__ inline void ep_stage_table(double* tab, const double* __restrict__ g) {
  for (int i = threadIdx.x; i < BOYSD_NT; i += EP_THREADS) {
    const double* s = g + 2 * i * BOYS_NM + L;  // every second node of the 0.1 grid
#pragma unroll
    for (int k = 0; k <= BOYSD_TERMS; ++k)  // (order 5: a term less, 9e-19 at most)
      tab[i * BOYSD_COLS + k] = L + k < BOYS_NM ? s[L + k < BOYS_NM ? k : 0] * INV_FACT[k] : 0.0;
    if constexpr (L > 0) tab[i * BOYSD_COLS + BOYSD_TERMS + 1] = exp(-(double)i * BOYSD_H);
  }
}

// -------------------------------------------------------- Hermite indices ----
// (t, u, v) numbered by order t + u + v, then u + v, then v.
__host__ __device__ constexpr int hidx(int t, int u, int v) {
  const int s = t + u + v, w = u + v;
  return s * (s + 1) * (s + 2) / 6 + w * (w + 1) / 2 + v;
}
__host__ __device__ constexpr int hcount(int L) { return (L + 1) * (L + 2) * (L + 3) / 6; }
struct HermiteTable {
  int up[35][3];             // index raised once along each axis (orders 0-4)
  int axis[56];              // an axis of the highest power
  int lo1[56], lo2[56];      // lowered once and twice along it
  int pow[56];               // the power after lowering once
};
constexpr HermiteTable make_hermite_table() {
  HermiteTable h{};
  for (int s = 0; s <= 5; ++s)
    for (int w = 0; w <= s; ++w)
      for (int v = 0; v <= w; ++v) {
        const int t[3] = {s - w, w - v, v};
        const int k = hidx(t[0], t[1], t[2]);
        for (int d = 0; d < 3; ++d)
          if (s < 5) h.up[k][d] = hidx(t[0] + (d == 0), t[1] + (d == 1), t[2] + (d == 2));
        if (s == 0) continue;
        const int d = t[0] >= t[1] && t[0] >= t[2] ? 0 : (t[1] >= t[2] ? 1 : 2);
        h.axis[k] = d;
        h.pow[k] = t[d] - 1;
        h.lo1[k] = hidx(t[0] - (d == 0), t[1] - (d == 1), t[2] - (d == 2));
        if (t[d] >= 2) h.lo2[k] = hidx(t[0] - 2 * (d == 0), t[1] - 2 * (d == 1), t[2] - 2 * (d == 2));
      }
  return h;
}
__device__ constexpr HermiteTable HT = make_hermite_table();

// R_tuv from b[n] = (-2 alpha)^n F_n times the prefactor, t + u + v <= L.
template <int L, typename T>
__device__ __forceinline__ void hermite_coulomb(const T (&x)[3], const T (&b)[L + 1], T (&R)[hcount(L)]) {
  T w[L + 1][hcount(L)];
#pragma unroll
  for (int n = 0; n <= L; ++n) w[n][0] = b[n];
#pragma unroll
  for (int s = 1; s <= L; ++s)
#pragma unroll
    for (int k = hcount(s - 1); k < hcount(s); ++k)
#pragma unroll
      for (int n = 0; n <= L - s; ++n) {
        T v = x[HT.axis[k]] * w[n + 1][HT.lo1[k]];
        if (HT.pow[k] > 0) v += T(HT.pow[k]) * w[n + 1][HT.lo2[k]];
        w[n][k] = v;
      }
#pragma unroll
  for (int k = 0; k < hcount(L); ++k) R[k] = w[0][k];
}

// ------------------------------------------------------------- LDS layout ----
template <typename T>
struct EpPrim {  // a primitive pair: exponent sum, centre, K / p, second exponent / p, 1 / (2 p), shell pair
  T p, x, y, z, k, w, u;
  int pair;
};
__host__ __device__ constexpr int ep_comps(int X) { return X == 0 ? 1 : (X == 1 ? 3 : 9); }
template <typename T, int X>
struct EpSide {
  int sh[EP_PAIRS][2];       // shells
  int off[EP_PAIRS + 1];     // first candidate primitive of each staged pair
  int cs[EP_PAIRS + 1];      // first kept primitive
  T ab[EP_PAIRS][3];         // centre of the first shell minus that of the second
  // packed AO pair index of each component, in its top bit whether both AOs are
  // the same; EP_SKIP for the upper components of a pair of one shell
  uint32_t idx[EP_PAIRS][ep_comps(X)];
  int n, next, next_f, cont; // pairs staged; where the next stage starts; pair 0 continues an earlier stage
};
constexpr uint32_t EP_SAME = 0x80000000u, EP_SKIP = 0xffffffffu;
template <typename T, int X, int Y>
struct EpShared {
  EpSide<T, X> bra;
  EpSide<T, Y> ket;
  int wave_cnt[EP_WAVES];
  int nchunk, split;
  int chunk[EP_CHUNKS][4];   // first kept primitive, lanes, first pair, pairs (negative: continues a pair)
  EpPrim<T> bprim[EP_CAP_BRA], kprim[ep_cap_ket<T>(Y)];
  T rows[EP_WAVES][EP_ROWS * 65 + EP_SUM];  // 64 lanes and a pad per row; emission reads up to EP_SUM past a row
};
__host__ __device__ inline uint32_t tri32(uint32_t i) { return i * (i + 1) / 2; }

// Where a molecule's shells and pairs come from.
struct EpMol {
  const int* atm;
  const int* bas;
  const double* env;
  const int* ao;     // first AO of each shell
  const int* pairs;  // explicit pair list, or
  const int* sl;     // class-sorted shells with ns s shells first
  int ns;
};

template <int X>
__device__ inline void ep_pair(const EpMol& M, int first, int a, int& i, int& j) {
  if (M.pairs) {
    i = M.pairs[2 * (first + a)];
    j = M.pairs[2 * (first + a) + 1];
  } else if (X == 1) {
    i = M.sl[M.ns + a / M.ns];
    j = M.sl[a % M.ns];
  } else {
    int t = (int)((sqrt(8.0 * (double)a + 1.0) - 1.0) * 0.5);
    while ((t + 1) * (t + 2) / 2 <= a) ++t;
    while (t * (t + 1) / 2 > a) --t;
    const int base = X == 0 ? 0 : M.ns;
    i = M.sl[base + t];
    j = M.sl[base + a - t * (t + 1) / 2];
  }
}

// Stages pairs s, s + 1, ... (below e) of class X, from primitive f of pair s,
// up to EP_PAIRS pairs and `cap` primitives: a pair with more primitives than
// `cap` is split over stages.  All threads of the workgroup call it.
template <typename T, int X>
__device__ inline void ep_stage(const EpMol& M, int first, int s, int f, int e, EpSide<T, X>& S, EpPrim<T>* prim, int cap,
                                double ang, int* wave_cnt) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (wave == 0) {
    int k = 0;
    if (s + lane < e) {
      int i, j;
      ep_pair<X>(M, first, s + lane, i, j);
      const int* bi = M.bas + i * BAS_SLOTS;
      const int* bj = M.bas + j * BAS_SLOTS;
      k = bi[2] * bj[2] - (lane == 0 ? f : 0);
      S.sh[lane][0] = i;
      S.sh[lane][1] = j;
      const uint32_t ai = M.ao[i], aj = M.ao[j];
#pragma unroll
      for (int fi = 0; fi < (X > 0 ? 3 : 1); ++fi)
#pragma unroll
        for (int fj = 0; fj < (X == 2 ? 3 : 1); ++fj) {
          const uint32_t p = ai + fi, q = aj + fj;
          S.idx[lane][fi * (X == 2 ? 3 : 1) + fj] = i == j && q > p
                                                        ? EP_SKIP
                                                        : (tri32(max(p, q)) + min(p, q)) | (p == q ? EP_SAME : 0u);
        }
      const double* ri = M.env + M.atm[bi[0] * ATM_SLOTS + 1];
      const double* rj = M.env + M.atm[bj[0] * ATM_SLOTS + 1];
      for (int d = 0; d < 3; ++d) S.ab[lane][d] = (T)(ri[d] - rj[d]);
    }
    int inc = k;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int v = __shfl_up(inc, d);
      if (lane >= d) inc += v;
    }
    const bool in = s + lane < e && inc <= cap;
    int n = __popcll(__ballot(in));
    const bool split = n == 0;
    if (split) {
      n = 1;
      inc = min(inc, cap);
      if (lane == 0) k = cap;
    }
    S.off[lane] = lane < n ? inc - k : 0;
    if (lane == n - 1) S.off[n] = inc;
    if (lane == 0) {
      S.n = n;
      S.cont = f > 0;
      S.next = split ? s : s + n;
      S.next_f = split ? f + cap : 0;
    }
  }
  __syncthreads();
  const int n = S.n, total = S.off[n];
  int base = 0;
  for (int c0 = 0; c0 < total; c0 += EP_THREADS) {
    const int c = c0 + tid;
    bool keep = false;
    int pair = 0;
    EpPrim<T> r;
    if (c < total) {
      int hi = n;
      while (hi - pair > 1) {
        const int mid = (pair + hi) >> 1;
        if (S.off[mid] <= c)
          pair = mid;
        else
          hi = mid;
      }
      const int* bi = M.bas + S.sh[pair][0] * BAS_SLOTS;
      const int* bj = M.bas + S.sh[pair][1] * BAS_SLOTS;
      const int q = c - S.off[pair] + (pair == 0 ? f : 0);
      const int npj = bj[2], pi = q / npj, pj = q - pi * npj;
      const double* ri = M.env + M.atm[bi[0] * ATM_SLOTS + 1];
      const double* rj = M.env + M.atm[bj[0] * ATM_SLOTS + 1];
      const double a = M.env[bi[5] + pi], b = M.env[bj[5] + pj], p = a + b, rp = 1.0 / p, w = b * rp;
      double r2 = 0.0, P[3];
      for (int d = 0; d < 3; ++d) {
        const double x = ri[d] - rj[d];
        r2 += x * x;
        P[d] = ri[d] - w * x;
      }
      const double k = M.env[bi[6] + pi] * M.env[bj[6] + pj] * exp(-a * w * r2) * rp;
      keep = !(fabs(k) < EpCut<T>::v);  // not-a-number stays
      r.p = (T)p;
      r.x = (T)P[0];
      r.y = (T)P[1];
      r.z = (T)P[2];
      r.k = (T)(k * ang);
      r.w = (T)w;
      r.u = (T)(0.5 * rp);
      r.pair = pair;
    }
    const uint64_t m = __ballot(keep);
    if (lane == 0) wave_cnt[wave] = __popcll(m);
    __syncthreads();
    int at = base;
    for (int v = 0; v < EP_WAVES; ++v) {
      if (v < wave) at += wave_cnt[v];
      base += wave_cnt[v];
    }
    at += __popcll(m & ((1ull << lane) - 1));
    if (keep) prim[at] = r;
    if (c < total && c == S.off[pair]) S.cs[pair] = at;
    __syncthreads();
  }
  if (tid == 0) S.cs[n] = base;
  __syncthreads();
}

// Cuts the staged ket primitives into chunks of at most 64 lanes holding whole
// shell pairs (a pair with more takes several chunks).  One wave calls it.
template <class Shared>
__device__ inline void ep_chunks(Shared& sh, int lane) {
  const auto& K = sh.ket;
  const int n = K.n, end = lane < n ? K.cs[lane + 1] : 0x7fffffff;
  int t = 0, pos = 0, c = 0, split = 0;
  while (t < n) {
    const int cnt = __popcll(__ballot(lane >= t && lane < n && end - pos <= 64));
    const int last = cnt ? K.cs[t + cnt] : pos + 64;
    const bool cont = pos > K.cs[t] || (t == 0 && K.cont);
    if (cnt == 0) split = 1;
    if (lane == 0) {
      sh.chunk[c][0] = pos;
      sh.chunk[c][1] = last - pos;
      sh.chunk[c][2] = t;
      sh.chunk[c][3] = cont ? -max(cnt, 1) : max(cnt, 1);
    }
    ++c;
    t += cnt;
    pos = last;
  }
  if (lane == 0) {
    sh.nchunk = c;
    sh.split = split;
  }
}

// Segmented sums of the wave's rows over each ket pair's lanes, and their
// stores: output o = (ket pair of the chunk, row) is spread over the lanes.
// Row r of a class with at least EP_ROWS components is component comp0 + r of
// bra pair bra0; otherwise component r % NC of bra pair bra0 + r / NC.
template <typename T, int X, int Y, int ROWS>
__device__ __forceinline__ void ep_emit(const EpShared<T, X, Y>& sh, const T* rows, int lane, int t0, int npair,
                                        int pos, int nl, bool kcont, int a, int b, int bra0, int comp0, int nrow,
                                        T* __restrict__ out, bool div) {
  constexpr int NK = ep_comps(Y), NC = ep_comps(X) * NK;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  const int nout = npair * ROWS;
#pragma unroll 1
  for (int o = lane; o < nout; o += 64) {
    const int seg = o / ROWS, row = o - seg * ROWS, t = t0 + seg;
    const int l0 = max(sh.ket.cs[t] - pos, 0), l1 = min(sh.ket.cs[t + 1] - pos, nl);
    const int bi = NC >= EP_ROWS ? bra0 : bra0 + row / NC;
    const int comp = NC >= EP_ROWS ? comp0 + row : row % NC;
    const uint32_t pqf = sh.bra.idx[min(bi, EP_PAIRS - 1)][comp / NK], rsf = sh.ket.idx[t][comp % NK];
    const T* rl = rows + row * 65;
    T sum = T(0);
    constexpr int NS = sizeof(T) == 4 ? EP_SUM : 4;
    for (int l = l0; l < l1; l += NS) {  // NS reads in flight, added in lane order
      T v[NS];
#pragma unroll
      for (int k = 0; k < NS; ++k) v[k] = rl[l + k];
#pragma unroll
      for (int k = 0; k < NS; ++k) sum += l + k < l1 ? v[k] : T(0);
    }
    const uint32_t pq = pqf & ~EP_SAME, rs = rsf & ~EP_SAME;
    bool skip = row >= nrow || pqf == EP_SKIP || rsf == EP_SKIP;
    // within one class: the ket pair at or below the bra pair, and of a pair
    // with itself the lower triangle
    if (X == Y) skip = skip || b + t > a + bi || (b + t == a + bi && rs > pq);
    if (!skip) {
      const uint32_t hi = max(pq, rs);
      const int64_t at = (int64_t)(((uint64_t)hi * (hi + 1)) >> 1) + min(pq, rs);
      // div: over the element's multiplicity 2^([p==q] + [r==s] + [pq==rs])
      if (div) sum *= T(1.0) / T(1 << ((pqf >> 31) + (rsf >> 31) + (pq == rs)));
      // a split pair (more primitives than a stage or a chunk holds) adds to what is there
      if ((kcont && seg == 0) || (sh.bra.cont && bi == 0)) sum += out[at];
      out[at] = sum;
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Expansions on the first bra centre that a bra class accumulates: 1 for ss, 3
// for ps, 9 for pp ((p_d|, then xx yy zz xy xz yz; the horizontal step to (pp|
// follows the primitive loop), or for one p component I of a pp pair's first
// shell 4 ((p_I|, then Ix Iy Iz).
__host__ __device__ constexpr int ep_rows(int X, int I) { return X == 0 ? 1 : (X == 1 ? 3 : (I >= 0 ? 4 : 9)); }
__device__ constexpr int EP_D[3][3] = {{3, 6, 7}, {6, 4, 8}, {7, 8, 5}};  // row of d component ij

// Bra primitives per step of the primitive loop: independent chains for the
// low classes, whose chains of dependent operations are latency-bound.
template <typename T>
__host__ __device__ constexpr int ep_unroll(int X, int Y) {
  return X + Y <= (sizeof(T) == 4 ? 2 : 1) ? 2 : 1;
}

// Adds U bra primitives (wave-uniform, from LDS) to the lane's accumulators.
template <typename T, int X, int Y, int I, int U, typename TabT>
__device__ __forceinline__ void ep_prims(const EpPrim<T>* prim, const T (&AB)[3], T q, const T (&Q)[3], const TabT* tab,
                                         T (&acc)[ep_rows(X, I)][hcount(Y)]) {
  constexpr int L = X + Y, H2 = hcount(Y);
  EpPrim<T> B[U];
  T x[U][3], F[U][L + 1], sc[U], al[U], t[U], tmax = T(0);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    B[u] = prim[u];
    x[u][0] = B[u].x - Q[0];
    x[u][1] = B[u].y - Q[1];
    x[u][2] = B[u].z - Q[2];
    const T rs = rsq(B[u].p + q);
    al[u] = B[u].p * q * rs * rs;
    sc[u] = B[u].k * rs;
    t[u] = al[u] * (x[u][0] * x[u][0] + x[u][1] * x[u][1] + x[u][2] * x[u][2]);
    tmax = u ? max(tmax, t[u]) : t[u];
    ep_boys<L>(t[u], tab, F[u]);
  }
  if (__any(tmax >= T(BOYS_EDGE))) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (t[u] >= T(BOYS_EDGE)) ep_boys_tail<L>(t[u], F[u]);
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    T bn[L + 1], R[hcount(L)];
#pragma unroll
    for (int n = 0; n <= L; ++n) {
      bn[n] = sc[u] * F[u][n];
      if (n < L) sc[u] *= T(-2) * al[u];
    }
    hermite_coulomb<L>(x[u], bn, R);
    if constexpr (X == 0) {
#pragma unroll
      for (int h = 0; h < H2; ++h) acc[0][h] += R[h];
    } else {
      const T h = B[u].u;  // 1 / (2 p)
      T PA[3];
#pragma unroll
      for (int d = 0; d < 3; ++d) PA[d] = -B[u].w * AB[d];
      if constexpr (X == 1) {
#pragma unroll
        for (int k = 0; k < H2; ++k)
#pragma unroll
          for (int d = 0; d < 3; ++d) acc[d][k] += PA[d] * R[k] + h * R[HT.up[k][d]];
      } else {
        const T h2 = h * h;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          if (I >= 0 && i != I) continue;
#pragma unroll
          for (int k = 0; k < H2; ++k) acc[I >= 0 ? 0 : i][k] += PA[i] * R[k] + h * R[HT.up[k][i]];
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            if (I < 0 && j < i) continue;
            const T e0 = PA[i] * PA[j] + (i == j ? h : T(0)), ei = PA[j] * h, ej = PA[i] * h;
#pragma unroll
            for (int k = 0; k < H2; ++k) {
              T v = e0 * R[k];
              if (i == j)
                v += (ei + ej) * R[HT.up[k][i]];
              else
                v += ei * R[HT.up[k][i]] + ej * R[HT.up[k][j]];
              acc[I >= 0 ? 1 + j : EP_D[i][j]][k] += v + h2 * R[HT.up[HT.up[k][i]][j]];
            }
          }
        }
      }
    }
  }
}

// ERIs of bra pairs [a0, a1) x ket pairs [b0, b1) (b <= a if X == Y); X <= Y:
// the class with more components is the lanes', whose expansion is outside the
// primitive loop.  I >= 0 ((pp|pp) only): the components of one p function of
// the bra's first shell, a third of the accumulators.
template <typename T, int X, int Y, int I, typename TabT>
__device__ inline void ep_tile(const EpMol& M, int xfirst, int yfirst, int a0, int a1, int b0, int b1, const TabT* tab,
                               EpShared<T, X, Y>& sh, T* __restrict__ out, bool div) {
  constexpr int NB = X == 0 ? 1 : (X == 1 || I >= 0 ? 3 : 9), NK = Y == 0 ? 1 : (Y == 1 ? 3 : 9);
  constexpr int H2 = hcount(Y), NC = NB * NK, NR = ep_rows(X, I), U = ep_unroll<T>(X, Y);
  constexpr int G = NC == 1 ? 8 : (NC == 3 ? 3 : 1);  // bra pairs per segmented sum
  constexpr int ROWS = NC >= EP_ROWS ? EP_ROWS : G * NC;
  // 2 pi^(5/2) and the s/p angular factors
  constexpr double ANGX = X == 0 ? ANG_S * ANG_S : (X == 1 ? ANG_S * ANG_P : ANG_P * ANG_P);
  constexpr double ANGY = Y == 0 ? ANG_S * ANG_S : (Y == 1 ? ANG_S * ANG_P : ANG_P * ANG_P);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  T* rows = sh.rows[wave];
  for (int b = b0, fb = 0; b < b1;) {
    ep_stage<T, Y>(M, yfirst, b, fb, b1, sh.ket, sh.kprim, ep_cap_ket<T>(Y), ANGY, sh.wave_cnt);
    if (wave == 0) ep_chunks(sh, lane);
    for (int a = a0, fa = 0; a < a1;) {
      ep_stage<T, X>(M, xfirst, a, fa, a1, sh.bra, sh.bprim, EP_CAP_BRA, 34.986836655249725 * ANGX, sh.wave_cnt);
      // items (ket chunk, run of bra pairs) dealt to the waves; where a ket pair
      // is split over chunks, one wave keeps a bra's chunks, in order
      const int nbra = sh.bra.n, run = min(EP_RUN, (nbra + EP_WAVES - 1) / EP_WAVES), nrun = (nbra + run - 1) / run;
      const int nitem = sh.nchunk * nrun, split = sh.split;
      for (int it = split ? 0 : wave; it < nitem; it += split ? 1 : EP_WAVES) {
        const int c = it / nrun, ir = it - c * nrun, r1 = min((ir + 1) * run, nbra);
        if (split && ir % EP_WAVES != wave) continue;
        const int pos = sh.chunk[c][0], nl = sh.chunk[c][1], t0 = sh.chunk[c][2];
        const bool kcont = sh.chunk[c][3] < 0;
        const int npair = abs(sh.chunk[c][3]);
        // ket pairs of this chunk all above the bra pairs before r0
        const int r0 = X == Y ? max(ir * run, b + t0 - a) : ir * run;
        if (r0 >= r1) continue;
        // this lane's ket primitive (idle lanes: a harmless one with zero prefactor)
        T q = T(1), Q[3] = {T(0), T(0), T(0)}, kk = T(0), QC[3], QD[3], uq = T(0);
        if (lane < nl) {
          const EpPrim<T> r = sh.kprim[pos + lane];
          q = r.p;
          Q[0] = r.x;
          Q[1] = r.y;
          Q[2] = r.z;
          kk = r.k;
          uq = r.u;
          if constexpr (Y > 0)
            for (int d = 0; d < 3; ++d) {
              const T cd = sh.ket.ab[r.pair][d];
              QC[d] = -r.w * cd;
              QD[d] = (T(1) - r.w) * cd;
            }
        } else {
          for (int d = 0; d < 3; ++d) QC[d] = QD[d] = T(0);
        }
#pragma unroll 1
        for (int ib = r0, g = 0, g0 = r0; ib < r1; ++ib) {
          const int s1 = __builtin_amdgcn_readfirstlane(sh.bra.cs[ib + 1]);
          int s = __builtin_amdgcn_readfirstlane(sh.bra.cs[ib]);
          T AB[3];
          for (int d = 0; d < 3; ++d) AB[d] = sh.bra.ab[ib][d];
          T acc[NR][H2];
#pragma unroll
          for (int i = 0; i < NR; ++i)
#pragma unroll
            for (int h = 0; h < H2; ++h) acc[i][h] = T(0);
#pragma unroll 1
          for (; s + U <= s1; s += U) ep_prims<T, X, Y, I, U>(sh.bprim + s, AB, q, Q, tab, acc);
          if constexpr (U > 1)
#pragma unroll 1
            for (; s < s1; ++s) ep_prims<T, X, Y, I, 1>(sh.bprim + s, AB, q, Q, tab, acc);
          // horizontal step, ket expansion, rows for the segmented sum
#pragma unroll
          for (int cb = 0; cb < NB; ++cb) {
            T v[H2];
#pragma unroll
            for (int h = 0; h < H2; ++h) {
              if constexpr (X < 2)
                v[h] = acc[cb][h];
              else if constexpr (I >= 0)
                v[h] = acc[1 + cb][h] + AB[cb] * acc[0][h];
              else
                v[h] = acc[EP_D[cb / 3][cb % 3]][h] + AB[cb % 3] * acc[cb / 3][h];
            }
            T val[NK];
            if constexpr (Y == 0) {
              val[0] = kk * v[0];
            } else if constexpr (Y == 1) {
#pragma unroll
              for (int d = 0; d < 3; ++d) val[d] = kk * (QC[d] * v[0] - uq * v[1 + d]);
            } else {
#pragma unroll
              for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int j = 0; j < 3; ++j)
                  val[i * 3 + j] = kk * ((QC[i] * QD[j] + (i == j ? uq : T(0))) * v[0] -
                                         uq * (QC[i] * v[1 + j] + QD[j] * v[1 + i]) +
                                         uq * uq * v[HT.up[1 + i][j]]);
            }
            const int row0 = NC >= EP_ROWS ? (cb * NK) % EP_ROWS : g * NC + cb * NK;
#pragma unroll
            for (int d = 0; d < NK; ++d) rows[(row0 + d) * 65 + lane] = val[d];
            const bool full = NC >= EP_ROWS ? (cb * NK) % EP_ROWS + NK == EP_ROWS
                                            : cb == NB - 1 && (g == G - 1 || ib == r1 - 1);
            if (full)
              ep_emit<T, X, Y, ROWS>(sh, rows, lane, t0, npair, pos, nl, kcont, a, b, NC >= EP_ROWS ? ib : g0,
                                     NC >= EP_ROWS ? ((I < 0 ? 0 : 3 * I) + cb) * NK / EP_ROWS * EP_ROWS : 0,
                                     NC >= EP_ROWS ? EP_ROWS : (g + 1) * NC, out, div);
          }
          if (NC < EP_ROWS && ++g == G) {
            g = 0;
            g0 = ib + 1;
          }
        }
      }
      fa = sh.bra.next_f;
      a = sh.bra.next;
      __syncthreads();
    }
    fb = sh.ket.next_f;
    b = sh.ket.next;
    __syncthreads();
  }
}

// Tile t of class (X, Y) with nx and ny pairs, na x nb pairs per tile (na
// divides nb): every tile, or for X == Y those with a ket at or below a bra.
template <int X, int Y>
__host__ __device__ inline int64_t ep_tiles(int64_t nx, int64_t ny, int na, int nb) {
  const int64_t ta = (nx + na - 1) / na, tb = (ny + nb - 1) / nb;
  if (X != Y) return ta * tb;
  const int r = nb / na;
  const int64_t g = ta / r, rest = ta - g * r;  // bra tiles g r .. take g + 1 ket tiles each
  return r * (g * (g + 1) / 2) + rest * (g + 1);
}
template <int X, int Y>
__device__ inline void ep_tile_at(int64_t t, int ny, int na, int nb, int& ta, int& tb) {
  if (X != Y) {
    const int n = (ny + nb - 1) / nb;
    ta = (int)(t / n);
    tb = (int)(t - (int64_t)ta * n);
  } else {
    const int r = nb / na;
    int64_t g = (int64_t)((sqrt(8.0 * (double)(t / r) + 1.0) - 1.0) * 0.5);
    while (r * ((g + 1) * (g + 2) / 2) <= t) ++g;
    while (r * (g * (g + 1) / 2) > t) --g;
    const int64_t rem = t - r * (g * (g + 1) / 2);
    ta = (int)(g * r + rem / (g + 1));
    tb = (int)(rem % (g + 1));
  }
}

// ---------------------------------------------------------------- kernels ----
// Classes (bra|ket): (pp|pp), (ps|pp), (ss|pp), (ps|ps), (ss|ps), (ss|ss), heaviest first.
constexpr int EP_CLASSES = 6;
constexpr int EP_X[EP_CLASSES] = {2, 1, 0, 1, 0, 0}, EP_Y[EP_CLASSES] = {2, 2, 2, 1, 1, 0};

// LDS of a workgroup: Boys table, then EpShared.
template <typename T, int C>
constexpr size_t ep_lds() {
  return EpTable<T>::bytes + sizeof(EpShared<T, EP_X[C], EP_Y[C]>);
}
template <typename T>
constexpr size_t ep_lds_max() {
  size_t m = ep_lds<T, 0>();
  m = ep_lds<T, 1>() > m ? ep_lds<T, 1>() : m;
  m = ep_lds<T, 2>() > m ? ep_lds<T, 2>() : m;
  m = ep_lds<T, 3>() > m ? ep_lds<T, 3>() : m;
  m = ep_lds<T, 4>() > m ? ep_lds<T, 4>() : m;
  return ep_lds<T, 5>() > m ? ep_lds<T, 5>() : m;
}

// Runs tile t of class C.  SPLIT: (pp|pp) comes as three tiles, one per p
// function of the bra's first shell (a third of the accumulators and three
// times the workgroups, for about 1.6 times the operations).
template <typename T, int C, bool SPLIT>
struct EpRun {
  static constexpr int X = EP_X[C], Y = EP_Y[C], parts = SPLIT && X == 2 ? 3 : 1;
  __host__ __device__ static int64_t tiles(int64_t nx, int64_t ny, int na, int nb) {
    return parts * ep_tiles<X, Y>(nx, ny, na, nb);
  }
  // bra pairs [a0, a1) x ket pairs [b0, b1), part i
  template <typename TabT>
  __device__ static inline void rect(const EpMol& M, int xfirst, int yfirst, int a0, int a1, int b0, int b1, int i,
                                     const TabT* tab, EpShared<T, X, Y>& sh, T* out, bool div) {
    if constexpr (parts == 1) {
      ep_tile<T, X, Y, -1>(M, xfirst, yfirst, a0, a1, b0, b1, tab, sh, out, div);
    } else {
      if (i == 0)
        ep_tile<T, X, Y, 0>(M, xfirst, yfirst, a0, a1, b0, b1, tab, sh, out, div);
      else if (i == 1)
        ep_tile<T, X, Y, 1>(M, xfirst, yfirst, a0, a1, b0, b1, tab, sh, out, div);
      else
        ep_tile<T, X, Y, 2>(M, xfirst, yfirst, a0, a1, b0, b1, tab, sh, out, div);
    }
  }
  template <typename TabT>
  __device__ static inline void tile(const EpMol& M, int xfirst, int yfirst, int nx, int ny, int na, int nb, int64_t t,
                                     const TabT* tab, EpShared<T, X, Y>& sh, T* out, bool div) {
    int ta, tb;
    ep_tile_at<X, Y>(t / parts, ny, na, nb, ta, tb);
    const int a0 = ta * na, a1 = min(a0 + na, nx), b0 = tb * nb, b1 = min(b0 + nb, X == Y ? a1 : ny);
    rect(M, xfirst, yfirst, a0, a1, b0, b1, (int)(t % parts), tab, sh, out, div);
  }
};

// One molecule, explicit class-sorted pair list: workgroups [b0[c], b0[c + 1])
// take the tiles of class c.
struct EpLaunch {
  int off[3], cnt[3];
  int na[EP_CLASSES], nb[EP_CLASSES];
  int b0[EP_CLASSES + 1];
};

template <typename T, int C>
__device__ inline void ep_launch_class(const EpMol& M, const EpLaunch& E, unsigned char* smem, T* out) {
  constexpr int X = EP_X[C], Y = EP_Y[C];
  auto* tab = reinterpret_cast<typename EpTable<T>::type*>(smem);
  ep_stage_table<X + Y>(tab, g_boys);
  auto& sh = *reinterpret_cast<EpShared<T, X, Y>*>(smem + EpTable<T>::bytes);
  EpRun<T, C, true>::tile(M, E.off[X], E.off[Y], E.cnt[X], E.cnt[Y], E.na[C], E.nb[C], (int)blockIdx.x - E.b0[C], tab,
                          sh, out, false);
}

template <typename T>
__global__ void __launch_bounds__(EP_THREADS, 2) eri_s8_kernel(const int* __restrict__ atm, const int* __restrict__ bas,
                                                            const double* __restrict__ env, int nbas,
                                                            const int* __restrict__ pairs, EpLaunch E,
                                                            T* __restrict__ out) {
  extern __shared__ __align__(16) unsigned char smem[];
  int* ao_loc = reinterpret_cast<int*>(smem + ep_lds_max<T>());
  stage_ao_loc(ao_loc, bas, nbas);
  __syncthreads();
  const EpMol M{atm, bas, env, ao_loc, pairs, pairs, 1};
  const int b = blockIdx.x;
  if (b < E.b0[1])
    ep_launch_class<T, 0>(M, E, smem, out);
  else if (b < E.b0[2])
    ep_launch_class<T, 1>(M, E, smem, out);
  else if (b < E.b0[3])
    ep_launch_class<T, 2>(M, E, smem, out);
  else if (b < E.b0[4])
    ep_launch_class<T, 3>(M, E, smem, out);
  else if (b < E.b0[5])
    ep_launch_class<T, 4>(M, E, smem, out);
  else
    ep_launch_class<T, 5>(M, E, smem, out);
}

// Pairs of class X in a molecule with ns s and np p shells.
__host__ __device__ inline int ep_count(int X, int ns, int np) {
  return X == 0 ? ns * (ns + 1) / 2 : (X == 1 ? ns * np : np * (np + 1) / 2);
}

// All molecules of an FP32 batch, one class: `per` workgroups share a molecule's
// tiles.  `per` is odd: neighbouring workgroups go to different XCDs, and with
// an even count the parts of molecules with few tiles all fell on the same few
// XCDs (1024 nine-heavy-atom molecules: 69 ms with 32, 51 ms with 31; 500: 33 ms
// with 64, 25.5 with 65).  The
// classes have a launch each: in one launch they would all take the registers
// and LDS of the heaviest (74 ms).
template <int C>
__global__ void __launch_bounds__(EP_THREADS, 2) eri_s8_mols_kernel(
    const BatchMol* __restrict__ mols, const int* __restrict__ order, int per, const int* __restrict__ atm,
    const int* __restrict__ bas, const double* __restrict__ env, const int* __restrict__ shell_ao,
    const int* __restrict__ shl, int na, int nb, float* __restrict__ out, int div) {
  using Run = EpRun<float, C, false>;
  extern __shared__ __align__(16) unsigned char smem[];
  const int mo = blockIdx.x / per, part = blockIdx.x - mo * per;
  const BatchMol B = mols[order ? order[mo] : mo];
  const int ns = (int)B.ns, np = (int)B.np, nx = ep_count(Run::X, ns, np), ny = ep_count(Run::Y, ns, np);
  const int64_t tiles = Run::tiles(nx, ny, na, nb);
  if (part >= tiles) return;
  auto* tab = reinterpret_cast<float4*>(smem);
  ep_stage_table<Run::X + Run::Y>(tab, g_boys);
  auto& sh = *reinterpret_cast<EpShared<float, Run::X, Run::Y>*>(smem + EpTable<float>::bytes);
  const EpMol M{atm, bas, env, shell_ao, nullptr, shl + B.shl0, ns};
  for (int64_t t = part; t < tiles; t += per) Run::tile(M, 0, 0, nx, ny, na, nb, t, tab, sh, out + B.eri0, div != 0);
}

// Work lists of (molecule, first quartet) entries of EP_LIST quartets each,
// quartets numbered row by row, a row being the quartets of one pair of the
// heavier class (the lower triangle within one class): a workgroup takes
// EP_GROUP entries and merges neighbours, so that a range of quartets is a few
// whole rows and a part of a row at either end.
constexpr int EP_LIST = 256, EP_GROUP = 16;
template <int C>
__global__ void __launch_bounds__(EP_THREADS, 2) eri_s8_list_kernel(
    const BatchMol* __restrict__ mols, const int* __restrict__ work, int nwork, const int* __restrict__ atm,
    const int* __restrict__ bas, const double* __restrict__ env, const int* __restrict__ shell_ao,
    const int* __restrict__ shl, float* __restrict__ out, int div) {
  using Run = EpRun<float, C, false>;
  constexpr bool TRI = Run::X == Run::Y;
  extern __shared__ __align__(16) unsigned char smem[];
  auto* tab = reinterpret_cast<float4*>(smem);
  ep_stage_table<Run::X + Run::Y>(tab, g_boys);
  auto& sh = *reinterpret_cast<EpShared<float, Run::X, Run::Y>*>(smem + EpTable<float>::bytes);
  const int w1 = min((int)(blockIdx.x + 1) * EP_GROUP, nwork);
  for (int w = blockIdx.x * EP_GROUP; w < w1;) {
    const int m = work[2 * w];
    int64_t q = work[2 * w + 1], q1 = q + EP_LIST;
    for (++w; w < w1 && work[2 * w] == m && work[2 * w + 1] == q1; ++w) q1 += EP_LIST;
    const BatchMol B = mols[m];
    const int ns = (int)B.ns, np = (int)B.np;
    const int64_t nrow = ep_count(Run::Y, ns, np), ncol = ep_count(Run::X, ns, np);
    const int64_t total = TRI ? tri(nrow) : nrow * ncol;
    q1 = q1 < total ? q1 : total;
    const EpMol M{atm, bas, env, shell_ao, nullptr, shl + B.shl0, ns};
    while (q < q1) {
      // row of q, its first quartet and length
      int64_t r = TRI ? (int64_t)((sqrt(8.0 * (double)q + 1.0) - 1.0) * 0.5) : q / ncol;
      if (TRI) {
        while (tri(r + 1) <= q) ++r;
        while (tri(r) > q) --r;
      }
      const int64_t row0 = TRI ? tri(r) : r * ncol, len = TRI ? r + 1 : ncol;
      int64_t r1 = r + 1, c0 = q - row0, c1 = q1 - row0 < len ? q1 - row0 : len;
      q = row0 + c1;
      if (c0 == 0 && c1 == len) {  // whole rows from here on
        while (r1 < nrow && q + (TRI ? r1 + 1 : ncol) <= q1) {
          q += TRI ? r1 + 1 : ncol;
          ++r1;
        }
        c1 = TRI ? r1 : ncol;
      }
      // rows are bra pairs in the triangle, else the lanes' ket pairs
      if (TRI)
        Run::rect(M, 0, 0, (int)r, (int)r1, (int)c0, (int)c1, 0, tab, sh, out + B.eri0, div != 0);
      else
        Run::rect(M, 0, 0, (int)c0, (int)c1, (int)r, (int)r1, 0, tab, sh, out + B.eri0, div != 0);
    }
  }
}

}  // namespace pscf
