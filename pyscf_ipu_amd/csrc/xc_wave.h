// Wave-private XC tiles: each wave takes 16 grid points through the whole
// pipeline -- AO values, X = phi0 D, densities, Y, V += phi0^T Y -- and the
// workgroup's four waves meet only for the pointwise functional, whose three
// parts take a wave each over the 64 points: two barriers per 64 points, so
// one wave's matrix products run beside another's loads or AO evaluation.
// Each lane forms exactly the Y and phi0 values that its GEMM-2 operands are
// (the points of a k step are the rows row(lg, k) of GEMM 1's accumulators), so
// Y never goes to LDS.  A wave keeps its whole V in registers, and its whole D
// operand too where both fit (DLDS otherwise).
//
// Measured against workgroup-wide tiles (five barriers per 32 points): 1024
// 9-heavy molecules, FP32, AO values evaluated in the kernel, one XC pass 9.3 ->
// 6.0 ms; one 9-heavy molecule at level 1 from a stored block, FP32, 62 -> 32 us.
// The direct form is bound by the sum of AO evaluation (a third of the time), matrix
// products (a third; their peak-rate time is 1.9 ms) and LDS traffic, which two
// waves a SIMD overlap only in part; the stored form in FP64 by matrix products and
// the functional, HBM time about a third.
#pragma once
#include "common.h"

namespace pscf {

// LDS layout (elements of T): waves' phi [4][PHI] (| D [NP][XD] with DLDS), or,
// at a flush, NVB partial V matrices; then rho [2][4][64], the functional's
// parts [9][64] and the waves' coefficients [4][4][16].
// STORED keeps an AO block's gradients in registers (LDS: phi0 alone, for GEMM
// 1's operand); the direct form transposes all four components through LDS.
template <typename T, int NP, bool STORED>
struct XW {
  typedef typename XMTraits<T>::v4 v4;
  static constexpr int NB = NP / 16, NK = NP / 4;
  // row stride: 16 consecutive rows spread over all 64 banks
  static constexpr int XS = NP + (STORED && sizeof(T) == 8 ? 2 : 4), XD = NP <= 16 ? 16 : (NP == 48 ? 48 : 80);
  // HS = 2: two waves share 16 points, each with half of the columns of X, Y and
  // V, where all of them (FP64, nao 64: 128 registers of V, 128 of AO values) leave
  // a wave nothing for the functional; 512 threads, two waves a SIMD (the SCF of a
  // molecule of nao 60: 4.39 ms, 4.50 with a wave per 16 points)
  static constexpr int HS = STORED && sizeof(T) == 8 && NP == 64 ? 2 : 1, THREADS = XC_THREADS * HS, NBH = NB / HS;
  static constexpr int PHI = (STORED ? HS : 4) * 16 * XS;  // HS = 2: phi0 of this tile and the last
  static constexpr bool DLDS = STORED && (sizeof(T) == 8 ? NP >= 48 : NP >= 64);
  static constexpr int ND = DLDS ? 1 : NB * NK;  // D registers
  static constexpr int NV = 2;                   // partial V matrices of a flush
  static constexpr int MAIN0 = 4 * PHI + (DLDS ? NP * XD : 0);
  static constexpr int MAIN = MAIN0 > NV * NP * NP ? MAIN0 : NV * NP * NP;
  static constexpr int RHO = 2 * HS * 4 * 64, PART = 9 * 64, COEF = HS * 4 * 64;
  static constexpr size_t lds_elems = (size_t)MAIN + RHO + PART + COEF;
  static constexpr size_t lds_bytes = (sizeof(T) * lds_elems + 31) & ~(size_t)31;
};

// LDS reads of a wave's own earlier writes (in order within the wave).
__device__ __forceinline__ void xw_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// D of GEMM 1: registers D[4 k + lane / 16][16 cb + lane % 16], or LDS.
template <typename T, int NP, bool STORED>
__device__ inline void xw_load_d(const T* __restrict__ dm, int N, T (&dreg)[XW<T, NP, STORED>::ND]) {
  typedef XW<T, NP, STORED> L;
  if constexpr (!L::DLDS) {
    const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
#pragma unroll
    for (int cb = 0; cb < L::NB; ++cb)
#pragma unroll
      for (int k = 0; k < L::NK; ++k) {
        const int row = 4 * k + lg, col = 16 * cb + li;
        dreg[cb * L::NK + k] = row < N && col < N ? dm[row * N + col] : T(0);
      }
  }
}

// Before the first tile of a sum: V = 0 and, with DLDS, D into LDS (a flush
// overwrites it); in the direct form the padding columns of the wave's Phi = 0.
template <typename T, int NP, bool STORED>
__device__ inline void xw_begin(T* smem, const T* __restrict__ dm, int N,
                                typename XW<T, NP, STORED>::v4 (&vacc)[XW<T, NP, STORED>::NB * XW<T, NP, STORED>::NBH]) {
  typedef XW<T, NP, STORED> L;
  if constexpr (!STORED) {
    T* Phi = smem + (threadIdx.x >> 6) * L::PHI + (threadIdx.x & 63) * L::XS;
    for (int mu = N; mu < NP; ++mu) Phi[mu] = T(0);
  }
  if constexpr (L::DLDS) {
    T* Dm = smem + 4 * L::PHI;
    for (int x = threadIdx.x; x < NP * NP; x += L::THREADS) {
      const int i = x / NP, j = x - i * NP;
      Dm[i * L::XD + j] = i < N && j < N ? dm[i * N + j] : T(0);
    }
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < L::NB * L::NBH; ++u) vacc[u] = (typename L::v4){T(0), T(0), T(0), T(0)};
}

// X = phi0 D of the wave's 16 points (A operand from LDS, read once per k step
// for all column blocks).
template <typename T, int NP, bool STORED>
__device__ inline void xw_gemm1(const T* Phi, const T* Dm, const T (&dreg)[XW<T, NP, STORED>::ND],
                                typename XMTraits<T>::v4 (&x)[XW<T, NP, STORED>::NBH], int col0) {
  typedef XW<T, NP, STORED> L;
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
#pragma unroll
  for (int cb = 0; cb < L::NBH; ++cb) x[cb] = (typename L::v4){T(0), T(0), T(0), T(0)};
#pragma unroll
  for (int k = 0; k < L::NK; ++k) {
    const T av = Phi[li * L::XS + 4 * k + lg];
#pragma unroll
    for (int cb = 0; cb < L::NBH; ++cb)
      x[cb] = XMTraits<T>::mfma(av, L::DLDS ? Dm[(4 * k + lg) * L::XD + col0 + 16 * cb + li] : dreg[L::DLDS ? 0 : cb * L::NK + k],
                                x[cb]);
  }
}

// Densities to coefficients: s[4 c + j] is this lane's share of rho_c at point
// row(lg, j) of the wave's 16; on return coef[4][16] holds c_0 .. c_3 of the
// wave's points.  odd alternates from tile to tile: a wave may write the next
// tile's rho while another still reads this one's.
template <typename T, int HS>
__device__ inline void xw_point(T (&s)[16], T* rho, T* part, T* coef, int p0, int g, T wt, T eps, double& e_loc) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), slot = wave / HS;
  const int li = lane & 15, lg = lane >> 4;
  const T tot = transpose_reduce16_row(s, lane);
  rho[((wave % HS) * 4 + (li >> 2)) * 64 + slot * 16 + XMTraits<T>::row(lg, li & 3)] = tot;
  __syncthreads();
  auto rc = [&](int c, int q) { return HS == 1 ? rho[c * 64 + q] : rho[c * 64 + q] + rho[(4 + c) * 64 + q]; };
  if (wave < 3) {  // part `wave` of the functional (Slater + VWN, B88, LYP) at 64 points
    T r, gam, e = T(0), vr = T(0), vn = T(0);
    b3lyp_inputs<T>(rc(0, lane), rc(1, lane), rc(2, lane), rc(3, lane), eps, r, gam);
    if (wave == 0)
      b3lyp_part<T, 0>(r, gam, e, vr, vn);
    else if (wave == 1)
      b3lyp_part<T, 1>(r, gam, e, vr, vn);
    else
      b3lyp_part<T, 2>(r, gam, e, vr, vn);
    part[(3 * wave) * 64 + lane] = e;
    part[(3 * wave + 1) * 64 + lane] = vr;
    part[(3 * wave + 2) * 64 + lane] = vn;
  }
  __syncthreads();
  if (lane < 16) {
    const int q = slot * 16 + lane;
    T c[4] = {T(0), T(0), T(0), T(0)};
    if (p0 + lane < g) {
      const T e = part[q] + part[3 * 64 + q] + part[6 * 64 + q];
      const T vr = part[64 + q] + part[4 * 64 + q] + part[7 * 64 + q];
      const T vn = part[2 * 64 + q] + part[5 * 64 + q] + part[8 * 64 + q];
      if (wave % HS == 0) e_loc += (double)rc(0, q) * (double)wt * (double)e;
      const T f = T(4) * vn * wt;
      c[0] = T(0.5) * vr * wt;
      c[1] = f * rc(1, q);
      c[2] = f * rc(2, q);
      c[3] = f * rc(3, q);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) coef[k * 16 + lane] = c[k];
  }
  xw_fence();
}

// AO values of a wave's 16 points in the accumulators' layout: f[c][b][j] =
// component c, AO 16 b + li, point row(lg, j), from element (c, mu, p) at
// ao[c sc + mu smu + p sp].  AOs and points past the end repeat the last one:
// D's padding is zero, coefficients past g are zero, and V's padding is not
// stored, so their values do not matter.  With smu = 1 a load takes 16
// consecutive AOs; with sp = 1 four lanes' consecutive points of 16 AOs (FP64),
// or four consecutive points a lane (FP32).
template <typename T, int NP>
struct XwStored {
  const T* ao;
  int sc, smu, sp, g, N;
  static constexpr int NBH = XW<T, NP, true>::NBH;
  int moff[NBH];
  __device__ inline void init(int col0) {
#pragma unroll
    for (int b = 0; b < NBH; ++b) {
      const int mu = col0 + 16 * b + (int)(threadIdx.x & 15);
      moff[b] = (mu < N ? mu : N - 1) * smu;
    }
  }
  template <int C0, int C1>
  __device__ inline void load(int p0, T (&f)[C1 - C0][NBH][4]) const {
    const int lg = (threadIdx.x & 63) >> 4;
    if (sizeof(T) == 4 && sp == 1 && p0 + 16 <= g) {
      const int po = p0 + 4 * lg;
#pragma unroll
      for (int c = C0; c < C1; ++c)
#pragma unroll
        for (int b = 0; b < NBH; ++b) __builtin_memcpy(f[c - C0][b], ao + (c * sc + moff[b] + po), 4 * sizeof(T));
    } else {
      int po[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int p = p0 + XMTraits<T>::row(lg, j);
        po[j] = (p < g ? p : g - 1) * sp;
      }
#pragma unroll
      for (int c = C0; c < C1; ++c)
#pragma unroll
        for (int b = 0; b < NBH; ++b)
#pragma unroll
          for (int j = 0; j < 4; ++j) f[c - C0][b][j] = ao[c * sc + moff[b] + po[j]];
    }
  }
};

// AO registers of the tile at hand, loaded one tile ahead.
template <typename T, int NP>
struct XwAO {
  T f0[1][XW<T, NP, true>::NBH][4], fg[3][XW<T, NP, true>::NBH][4];
};

// Tiles tile, tile + tstride, ... (64 points each) below tile_end, from a
// stored AO block; f holds the first tile's values, and on return those of
// tile next (if it is not negative).
template <typename T, int NP>
__device__ inline void xw_tiles_stored(const XCArgs<T>& a, T* smem, int tile, int tstride, int tile_end, int next,
                                       const XwStored<T, NP>& st, XwAO<T, NP>& ao,
                                       const T (&dreg)[XW<T, NP, true>::ND],
                                       typename XMTraits<T>::v4 (&vacc)[XW<T, NP, true>::NB * XW<T, NP, true>::NBH],
                                       double& e_loc) {
  typedef XW<T, NP, true> L;
  constexpr int NB = L::NB, NBH = L::NBH, HS = L::HS;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, lg = lane >> 4, slot = wave / HS, col0 = wave % HS * NBH * 16;
  const T* Dm = smem + 4 * L::PHI;
  T* rho = smem + L::MAIN;
  T* part = rho + L::RHO;
  T* coef = part + L::PART + wave * 64;
  for (int odd = 0; tile < tile_end; tile += tstride, odd ^= 1) {
    const int p0 = tile * 64 + slot * 16;
    T* Phi = smem + slot * L::PHI + (HS == 2 ? odd * 16 * L::XS : 0);
    const T wt = lane < 16 && p0 + lane < a.g ? a.w[p0 + lane] : T(0);
    xw_fence();  // the last tile's reads of Phi and coef
#pragma unroll
    for (int b = 0; b < NBH; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j) Phi[XMTraits<T>::row(lg, j) * L::XS + col0 + 16 * b + li] = ao.f0[0][b][j];
    if constexpr (HS == 2)
      __syncthreads();  // the other wave's half
    else
      xw_fence();
    {
      typename L::v4 x[NBH];
      xw_gemm1<T, NP, true>(Phi, Dm, dreg, x, col0);
      T s[16];
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          T v = T(0);
#pragma unroll
          for (int b = 0; b < NBH; ++b) v += x[b][j] * (c == 0 ? ao.f0[0][b][j] : ao.fg[c > 0 ? c - 1 : 0][b][j]);
          s[c * 4 + j] = v;
        }
      xw_point<T, HS>(s, rho + odd * HS * 4 * 64, part, coef, p0, a.g, wt, a.eps, e_loc);
    }
    T y[NBH][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      T c[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) c[q] = coef[q * 16 + XMTraits<T>::row(lg, j)];
#pragma unroll
      for (int b = 0; b < NBH; ++b)
        y[b][j] = c[0] * ao.f0[0][b][j] + c[1] * ao.fg[0][b][j] + c[2] * ao.fg[1][b][j] + c[3] * ao.fg[2][b][j];
    }
    const int nt = tile + tstride < tile_end ? tile + tstride : next;
    T fn[1][NBH][4];
    __builtin_amdgcn_sched_barrier(0);
    if (nt >= 0) {
      st.template load<0, 1>(nt * 64 + slot * 16, fn);
      st.template load<1, 4>(nt * 64 + slot * 16, ao.fg);
    }
    __builtin_amdgcn_sched_barrier(0);
    // GEMM 2: V[mu][nu] += sum_p phi0[p][mu] Y[p][nu]
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int m = 0; m < NB; ++m) {
        const T f0 = HS == 2 ? Phi[XMTraits<T>::row(lg, j) * L::XS + 16 * m + li] : ao.f0[0][m % NBH][j];
#pragma unroll
        for (int n = 0; n < NBH; ++n) vacc[m * NBH + n] = XMTraits<T>::mfma(f0, y[n][j], vacc[m * NBH + n]);
      }
    if (nt >= 0) {
#pragma unroll
      for (int b = 0; b < NBH; ++b)
#pragma unroll
        for (int j = 0; j < 4; ++j) ao.f0[0][b][j] = fn[0][b][j];
    }
  }
}

// Evaluates a wave's 16 points from the shell records: lane l takes point
// l % 16 and records l / 16, l / 16 + 4, ....
template <typename T, int NP>
struct XwDirect {
  XcShells<T> sh;
  const double* coords;  // the molecule's points, [g][3]
  int g;
  double px, py, pz;
  __device__ inline void load(int p0) {
    const int pt = p0 + (int)(threadIdx.x & 15);
    const bool in = pt < g;
    px = in ? coords[3 * pt] : 0.0;
    py = in ? coords[3 * pt + 1] : 0.0;
    pz = in ? coords[3 * pt + 2] : 0.0;
  }
  __device__ inline void operator()(T* Phi, int p0, int next) {
    const int lane = threadIdx.x & 63, p = lane & 15;
    const bool in = p0 + p < g;
    const double x = px, y = py, z = pz;
    load(next);
    for (int r = lane >> 4; r < sh.nrec; r += 4) xc_eval_record<T, 16, XW<T, NP, false>::XS>(sh, r, x, y, z, in, Phi, p);
  }
};

// xw_tiles_stored with the AO values evaluated from the shell records.
template <typename T, int NP>
__device__ inline void xw_tiles_direct(const XCArgs<T>& a, T* smem, int tile, int tile_end, XwDirect<T, NP>& stage,
                                       const T (&dreg)[XW<T, NP, false>::ND],
                                       typename XMTraits<T>::v4 (&vacc)[XW<T, NP, false>::NB * XW<T, NP, false>::NB],
                                       double& e_loc) {
  typedef XW<T, NP, false> L;
  constexpr int XS = L::XS, NB = L::NB;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, lg = lane >> 4;
  T* Phi = smem + wave * L::PHI;
  T* rho = smem + L::MAIN;
  T* part = rho + L::RHO;
  T* coef = part + L::PART + wave * 64;
  // two waves share a SIMD: by unequal priority the one in its vector phase
  // runs at full rate and the two drift apart, so that matrix products meet
  // AO evaluation instead of other matrix products
  if (__builtin_amdgcn_s_getreg(4 | (3 << 11)) & 1) __builtin_amdgcn_s_setprio(2);  // HW_ID.wave_id, bits 3:0
  for (int odd = 0; tile < tile_end; ++tile, odd ^= 1) {
    const int p0 = tile * 64 + wave * 16;
    const T wt = lane < 16 && p0 + lane < a.g ? a.w[p0 + lane] : T(0);
    xw_fence();  // the last tile's reads of Phi and coef
    stage(Phi, p0, p0 + 64);
    xw_fence();
    {
      typename L::v4 x[NB];
      xw_gemm1<T, NP, false>(Phi, nullptr, dreg, x, 0);
      T s[16];
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const T* f = Phi + (c * 16 + XMTraits<T>::row(lg, j)) * XS + li;
          T v = T(0);
#pragma unroll
          for (int b = 0; b < NB; ++b) v += x[b][j] * f[16 * b];
          s[c * 4 + j] = v;
        }
      xw_point<T, 1>(s, rho + odd * 4 * 64, part, coef, p0, a.g, wt, a.eps, e_loc);
    }
    // GEMM 2: V[mu][nu] += sum_p phi0[p][mu] Y[p][nu], points 4 k + lg
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int p = 4 * k + lg;
      T c[4], f0[NB], y[NB];
#pragma unroll
      for (int q = 0; q < 4; ++q) c[q] = coef[q * 16 + p];
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const T* f = Phi + p * XS + 16 * b + li;
        f0[b] = f[0];
        y[b] = c[0] * f0[b] + c[1] * f[16 * XS] + c[2] * f[2 * 16 * XS] + c[3] * f[3 * 16 * XS];
      }
#pragma unroll
      for (int m = 0; m < NB; ++m)
#pragma unroll
        for (int n = 0; n < NB; ++n) vacc[m * NB + n] = XMTraits<T>::mfma(f0[m], y[n], vacc[m * NB + n]);
    }
  }
}

// Adds the four waves' V, (w0 + w2) + (w1 + w3), and hands (i, j, V_ij, V_ji)
// of i, j < N to out.  Begins and ends with a barrier; overwrites Phi and D.
template <typename T, int NP, bool STORED, class Out>
__device__ inline void xw_flush(T* smem, int N,
                                const typename XMTraits<T>::v4 (&vacc)[XW<T, NP, STORED>::NB * XW<T, NP, STORED>::NBH],
                                Out out) {
  typedef XW<T, NP, STORED> L;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, lg = lane >> 4;
  const int slot = wave / L::HS, col0 = wave % L::HS * L::NBH * 16;
  T* V = smem + (slot & 1) * NP * NP + col0;
  __syncthreads();
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if ((slot >> 1) == h) {
#pragma unroll
      for (int m = 0; m < L::NB; ++m)
#pragma unroll
        for (int n = 0; n < L::NBH; ++n)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            T* v = V + (16 * m + XMTraits<T>::row(lg, j)) * NP + 16 * n + li;
            *v = h ? *v + vacc[m * L::NBH + n][j] : vacc[m * L::NBH + n][j];
          }
    }
    __syncthreads();
  }
  for (int x = threadIdx.x; x < N * N; x += L::THREADS) {
    const int i = x / N, j = x - i * N;
    out(i, j, smem[i * NP + j] + smem[NP * NP + i * NP + j], smem[j * NP + i] + smem[NP * NP + j * NP + i]);
  }
  __syncthreads();
}

}  // namespace pscf
