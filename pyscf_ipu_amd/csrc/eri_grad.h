// Two-electron part of the nuclear gradient (grad_elec,
// pyscf_ipu/nanoDFT/nanoDFT.py:403-433, where int2e_ip1 is contracted with dm0
// into vj and vk), on the shell-pair primitive lists of eri_pairs.h:
// E_2e = 1/2 sum (ij|kl) G_ijkl with
//   G_ijkl = D_ij D_kl - (hyb/4) (D_ik D_jl + D_il D_jk).
// Every ordered (bra, ket) pair of shell pairs is taken and only the ket's
// centres are differentiated: the other half of the derivative is the swapped
// pair's.  The bra expansion is then the energy's, accumulated per ket
// primitive over the bra primitives, one Hermite order higher on the ket side;
// once per (bra pair, ket primitive) the ket expansion E and its derivatives
// meet G:
//   d/dQ raises the Hermite index, d/d(C - D) acts on E and on the prefactor,
//   d/dC = (c / q) d/dQ + d/d(C - D),  d/dD = (d / q) d/dQ - d/d(C - D).
// Six sums per ket pair and run of bra pairs leave through exact atomics.  FP64
// only.
//
// VALU-bound, and for one molecule bound by how far it spreads: (bra, ket)
// tiles of primitive lists in place of a lane per contracted quartet, whose
// chain ran over up to 36 x 36 primitives on a few workgroups (4 heavy atoms,
// 6-31G: six launches of 0.7 to 2.4 ms, 7.3 ms in all; now 0.22 + 0.06 ms).
#pragma once
#include "eri_pairs.h"

namespace pscf {

// Order-independent accumulation: contributions are rounded to multiples of
// 2^-40, so their FP64 sums are exact (below 2^13) whatever the order.
__device__ __forceinline__ double grad_quant(double v) { return rint(v * 0x1p40) * 0x1p-40; }

template <int X, int Y>
struct EgShared {
  EpSide<double, X> bra;
  EpSide<double, Y> ket;
  int wave_cnt[EP_WAVES];
  int nchunk, split;
  int chunk[EP_CHUNKS][4];
  EpPrim<double> bprim[EP_CAP_BRA], kprim[ep_cap_ket<double>(Y)];
};

struct EgArgs {
  const double* dm;
  int N;
  double hq;  // hyb / 4
  double* g;  // [natm][3]: LDS, or the gradient itself
};

// Bra pairs [a0, a1) x ket pairs [b0, b1).  I >= 0 (X = 2): the components of
// one p function of the bra's first shell.
template <int X, int Y, int I>
__device__ inline void eg_tile(const EpMol& M, int xfirst, int yfirst, int a0, int a1, int b0, int b1,
                               const double* tab, EgShared<X, Y>& sh, const EgArgs& A) {
  constexpr int NB = X == 0 ? 1 : (X == 1 || I >= 0 ? 3 : 9), H2 = hcount(Y + 1);
  constexpr int NR = ep_rows(X, I), U = X + Y == 0 ? 2 : 1;
  constexpr int KC = Y > 0 ? 3 : 1, KD = Y == 2 ? 3 : 1;               // ket components: KC x KD
  constexpr double ANGX = X == 0 ? ANG_S * ANG_S : (X == 1 ? ANG_S * ANG_P : ANG_P * ANG_P);
  constexpr double ANGY = Y == 0 ? ANG_S * ANG_S : (Y == 1 ? ANG_S * ANG_P : ANG_P * ANG_P);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const double* dm = A.dm;
  const int N = A.N;
  for (int b = b0, fb = 0; b < b1;) {
    ep_stage<double, Y>(M, yfirst, b, fb, b1, sh.ket, sh.kprim, ep_cap_ket<double>(Y), ANGY, sh.wave_cnt);
    if (wave == 0) ep_chunks(sh, lane);
    for (int a = a0, fa = 0; a < a1;) {
      ep_stage<double, X>(M, xfirst, a, fa, a1, sh.bra, sh.bprim, EP_CAP_BRA, 34.986836655249725 * ANGX, sh.wave_cnt);
      const int nbra = sh.bra.n, run = min(EP_RUN, (nbra + EP_WAVES - 1) / EP_WAVES), nrun = (nbra + run - 1) / run;
      const int nitem = sh.nchunk * nrun;
      for (int it = wave; it < nitem; it += EP_WAVES) {
        const int c = it / nrun, ir = it - c * nrun, r0 = ir * run, r1 = min(r0 + run, nbra);
        const int pos = sh.chunk[c][0], nl = sh.chunk[c][1];
        if (nl <= 0) continue;  // every primitive dropped
        // this lane's ket primitive (idle lanes: the last one's with a zero prefactor)
        const EpPrim<double> K = sh.kprim[pos + min(lane, nl - 1)];
        const double q = K.p, Q[3] = {K.x, K.y, K.z}, uq = K.u, w = K.w;
        const int ks = sh.ket.sh[K.pair][0], ls = sh.ket.sh[K.pair][1], ak = M.ao[ks], al = M.ao[ls];
        const double kk = lane < nl ? K.k * (ks == ls ? 1.0 : 2.0) : 0.0;
        double CD[3], QC[3], QD[3], gC[3] = {0.0, 0.0, 0.0}, gD[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          CD[d] = sh.ket.ab[K.pair][d];
          QC[d] = -w * CD[d];
          QD[d] = (1.0 - w) * CD[d];
        }
#pragma unroll 1
        for (int ib = r0; ib < r1; ++ib) {
          const int s1 = __builtin_amdgcn_readfirstlane(sh.bra.cs[ib + 1]);
          int s = __builtin_amdgcn_readfirstlane(sh.bra.cs[ib]);
          double AB[3];
          for (int d = 0; d < 3; ++d) AB[d] = sh.bra.ab[ib][d];
          double acc[NR][H2];
#pragma unroll
          for (int i = 0; i < NR; ++i)
#pragma unroll
            for (int h = 0; h < H2; ++h) acc[i][h] = 0.0;
#pragma unroll 1
          for (; s + U <= s1; s += U) ep_prims<double, X, Y + 1, I, U>(sh.bprim + s, AB, q, Q, tab, acc);
          if constexpr (U > 1)
#pragma unroll 1
            for (; s < s1; ++s) ep_prims<double, X, Y + 1, I, 1>(sh.bprim + s, AB, q, Q, tab, acc);
          const int is = sh.bra.sh[ib][0], js = sh.bra.sh[ib][1], ai = M.ao[is], aj = M.ao[js];
          // sums over the components with G: S = integral, dQ and dE = its
          // derivatives by Q and by E's dependence on C - D, all over kk
          double S = 0.0, dQ[3] = {0.0, 0.0, 0.0}, dE[3] = {0.0, 0.0, 0.0};
#pragma unroll
          for (int cb = 0; cb < NB; ++cb) {
            const int p = ai + (X == 0 ? 0 : (X == 1 ? cb : (I >= 0 ? I : cb / 3)));
            const int r = aj + (X < 2 ? 0 : (I >= 0 ? cb : cb % 3));
            double G[KC][KD];
            {
              const double Dpr = dm[p * N + r];
#pragma unroll
              for (int i = 0; i < KC; ++i)
#pragma unroll
                for (int j = 0; j < KD; ++j)
                  G[i][j] = Dpr * dm[(ak + i) * N + al + j] - A.hq * (dm[p * N + ak + i] * dm[r * N + al + j] +
                                                                      dm[p * N + al + j] * dm[r * N + ak + i]);
            }
            double v[H2];
#pragma unroll
            for (int h = 0; h < H2; ++h) {
              if constexpr (X < 2)
                v[h] = acc[cb][h];
              else if constexpr (I >= 0)
                v[h] = acc[1 + cb][h] + AB[cb] * acc[0][h];
              else
                v[h] = acc[EP_D[cb / 3][cb % 3]][h] + AB[cb % 3] * acc[cb / 3][h];
            }
            if constexpr (Y == 0) {
              S += G[0][0] * v[0];
#pragma unroll
              for (int e = 0; e < 3; ++e) dQ[e] -= G[0][0] * v[1 + e];
            } else if constexpr (Y == 1) {
              double T0 = 0.0;
#pragma unroll
              for (int i = 0; i < 3; ++i) {
                T0 += G[i][0] * QC[i];
                S -= uq * G[i][0] * v[1 + i];
                dE[i] -= w * G[i][0] * v[0];
              }
              S += T0 * v[0];
#pragma unroll
              for (int e = 0; e < 3; ++e) {
                double t = -T0 * v[1 + e];
#pragma unroll
                for (int i = 0; i < 3; ++i) t += uq * G[i][0] * v[HT.up[1 + i][e]];
                dQ[e] += t;
              }
            } else {
              double T0 = 0.0, T1[3] = {0.0, 0.0, 0.0}, T2[6];
#pragma unroll
              for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                  T0 += G[i][j] * (QC[i] * QD[j] + (i == j ? uq : 0.0));
                  T1[j] += uq * G[i][j] * QC[i];
                  T1[i] += uq * G[i][j] * QD[j];
                  const double tj = QD[j] * v[0] - uq * v[1 + j], ti = QC[i] * v[0] - uq * v[1 + i];
                  dE[i] -= w * G[i][j] * tj;
                  dE[j] += (1.0 - w) * G[i][j] * ti;
                }
              const double u2 = uq * uq;
#pragma unroll
              for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int j = i; j < 3; ++j)
                  T2[HT.up[1 + i][j] - 4] = u2 * (i == j ? G[i][i] : G[i][j] + G[j][i]);
              S += T0 * v[0];
#pragma unroll
              for (int k = 0; k < 3; ++k) S -= T1[k] * v[1 + k];
#pragma unroll
              for (int k = 0; k < 6; ++k) S += T2[k] * v[4 + k];
#pragma unroll
              for (int e = 0; e < 3; ++e) {
                double t = -T0 * v[1 + e];
#pragma unroll
                for (int k = 0; k < 3; ++k) t += T1[k] * v[HT.up[1 + k][e]];
#pragma unroll
                for (int k = 0; k < 6; ++k) t -= T2[k] * v[HT.up[4 + k][e]];
                dQ[e] += t;
              }
            }
          }
          const double f = is == js ? kk : 2.0 * kk, mu2 = 2.0 * w * (1.0 - w) * q;
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            const double dr = f * (dE[d] - mu2 * CD[d] * S), dq = f * dQ[d];
            gC[d] += (1.0 - w) * dq + dr;
            gD[d] += w * dq - dr;
          }
        }
        // sums over each ket pair's lanes (neighbours), in its first lane: fewer
        // atomics, and fewer roundings to their quantum
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
          const bool same = __shfl_down(K.pair, off) == K.pair && lane + off < 64;
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            const double c = __shfl_down(gC[d], off), e = __shfl_down(gD[d], off);
            gC[d] += same ? c : 0.0;
            gD[d] += same ? e : 0.0;
          }
        }
        const int before = __shfl_up(K.pair, 1);
        if (lane < nl && (lane == 0 || before != K.pair)) {
          const int atC = M.bas[ks * BAS_SLOTS], atD = M.bas[ls * BAS_SLOTS];
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            atomicAdd(A.g + 3 * atC + d, grad_quant(gC[d]));
            atomicAdd(A.g + 3 * atD + d, grad_quant(gD[d]));
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

// Ordered classes (bra|ket), heaviest first; the first EG_HEAVY, whose
// accumulators take a wave's whole register file, have a launch of their own,
// so that the others run two workgroups per CU.
constexpr int EG_CLASSES = 9, EG_HEAVY = 3;
constexpr int EG_X[EG_CLASSES] = {2, 1, 2, 0, 2, 1, 0, 1, 0}, EG_Y[EG_CLASSES] = {2, 2, 1, 2, 0, 1, 1, 0, 0};
// relative cost of a shell quartet (operations per primitive quartet)
constexpr double EG_COST[EG_CLASSES] = {30, 9, 9, 4, 3, 4, 2, 1.6, 1};
__host__ __device__ constexpr int eg_parts(int c) { return EG_X[c] == 2 && EG_Y[c] == 2 ? 3 : 1; }

struct EgLaunch {
  int off[3], cnt[3];
  int na[EG_CLASSES], nb[EG_CLASSES];
  int b0[EG_CLASSES + 1];  // first workgroup of each class of the launch
};

template <int C>
constexpr size_t eg_lds() {
  return EpTable<double>::bytes + sizeof(EgShared<EG_X[C], EG_Y[C]>);
}
template <int C0, int C1>
constexpr size_t eg_lds_max() {
  if constexpr (C0 + 1 == C1)
    return eg_lds<C0>();
  else
    return eg_lds<C0>() > eg_lds_max<C0 + 1, C1>() ? eg_lds<C0>() : eg_lds_max<C0 + 1, C1>();
}

template <int C, int C1>
__device__ inline void eg_class(const EpMol& M, const EgLaunch& E, unsigned char* smem, const EgArgs& A) {
  if (C + 1 < C1 && (int)blockIdx.x >= E.b0[C + 1]) {
    if constexpr (C + 1 < C1) eg_class<C + 1, C1>(M, E, smem, A);
    return;
  }
  constexpr int X = EG_X[C], Y = EG_Y[C], parts = eg_parts(C);
  double* tab = reinterpret_cast<double*>(smem);
  ep_stage_table<X + Y + 1>(tab, g_boys);
  auto& sh = *reinterpret_cast<EgShared<X, Y>*>(smem + EpTable<double>::bytes);
  const int u = (int)blockIdx.x - E.b0[C], t = u / parts, i = u - t * parts;
  const int na = E.na[C], nb = E.nb[C], nx = E.cnt[X], ny = E.cnt[Y], ntb = (ny + nb - 1) / nb;
  const int a0 = t / ntb * na, b0 = t % ntb * nb, a1 = min(a0 + na, nx), b1 = min(b0 + nb, ny);
  if constexpr (parts == 1) {
    eg_tile<X, Y, -1>(M, E.off[X], E.off[Y], a0, a1, b0, b1, tab, sh, A);
  } else {
    if (i == 0)
      eg_tile<X, Y, 0>(M, E.off[X], E.off[Y], a0, a1, b0, b1, tab, sh, A);
    else if (i == 1)
      eg_tile<X, Y, 1>(M, E.off[X], E.off[Y], a0, a1, b0, b1, tab, sh, A);
    else
      eg_tile<X, Y, 2>(M, E.off[X], E.off[Y], a0, a1, b0, b1, tab, sh, A);
  }
}

// Classes [C0, C1) of one molecule with a class-sorted pair list.  g_lds: the
// gradient's sums fit the LDS beside the tiles; otherwise the lanes' sums go
// to memory one by one.
template <int C0, int C1>
__global__ void __launch_bounds__(EP_THREADS, C0 == 0 ? 1 : 2) eri_grad_kernel(
    const int* __restrict__ atm, int natm, const int* __restrict__ bas, const double* __restrict__ env, int nbas,
    const int* __restrict__ pairs, EgLaunch E, const double* __restrict__ dm, int N, double hq, int g_lds,
    double* __restrict__ grad) {
  extern __shared__ __align__(16) unsigned char smem[];
  double* g = reinterpret_cast<double*>(smem + eg_lds_max<C0, C1>());
  int* ao_loc = reinterpret_cast<int*>(g + (g_lds ? 3 * natm : 0));
  stage_ao_loc(ao_loc, bas, nbas);
  if (g_lds)
    for (int i = threadIdx.x; i < 3 * natm; i += EP_THREADS) g[i] = 0.0;
  __syncthreads();
  const EpMol M{atm, bas, env, ao_loc, pairs, pairs, 1};
  eg_class<C0, C1>(M, E, smem, EgArgs{dm, N, hq, g_lds ? g : grad});
  __syncthreads();
  if (g_lds)
    for (int i = threadIdx.x; i < 3 * natm; i += EP_THREADS)
      if (g[i] != 0.0) atomicAdd(grad + i, g[i]);
}

}  // namespace pscf
