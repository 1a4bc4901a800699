// Learned initial guess on gfx950: atom-pair features, an MLP trained with
// BF16 MFMA (FP32 accumulation, FP32 master weights, Adam), and assembly of
// the predicted STO-3G density blocks into per-molecule density matrices.
//
// There is no counterpart in the reference (its SCF always starts from PySCF's
// MINAO guess, pyscf_ipu/nanoDFT/nanoDFT.py:233).  Network: per ordered atom
// pair, 43 inputs (one-hot H/C/N/O of both atoms, 32 Gaussian RBFs of the
// distance on 0..5 Angstrom with sigma 0.15 Angstrom, unit direction) ->
// 256 -> 256 -> 256 (SiLU) -> 25 (the 5x5 block of AOs of atom a x AOs of b).
#include <string.h>

#include "batch.h"
#include "common.h"
#include "wave.h"

namespace pscf {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short bf16_t;

__host__ __device__ inline bf16_t f2bf(float x) {  // round to nearest even
#ifdef __HIP_DEVICE_COMPILE__
  unsigned u = __float_as_uint(x);
#else
  unsigned u;
  memcpy(&u, &x, 4);
#endif
  u += 0x7fffu + ((u >> 16) & 1u);
  return (bf16_t)(u >> 16);
}
__device__ inline float bf2f(bf16_t h) { return __uint_as_float(((unsigned)h) << 16); }
__device__ inline float silu(float z) { return z / (1.0f + expf(-z)); }
__device__ inline float dsilu(float z) {
  const float s = 1.0f / (1.0f + expf(-z));
  return s * (1.0f + z * (1.0f - s));
}

enum Epilogue : int {
  EPI_BIAS_SILU = 0,  // Z = acc + b (FP32 out), H = silu(Z) (BF16 out2)
  EPI_BIAS = 1,       // out = acc + b (FP32)
  EPI_DSILU = 2,      // dZ = acc * dsilu(Zprev) -> FP32 out and BF16 out2
  EPI_ATOMIC = 3,     // out += acc (FP32 atomics; split-K)
  EPI_DSILU_SUM = 4,  // out2 = dZ = acc * dsilu(Zprev) (BF16), out[n] += sum_m dZ[m][n] (FP32 atomics)
};

constexpr int GBM = 64, GBN = 64, GBK = 16;

// What to do with one accumulated element (row, col).
template <int EPI>
__device__ __forceinline__ float gemm_store(float v, int row, int col, int64_t o, const float* __restrict__ bias,
                                            const float* __restrict__ aux, float* __restrict__ out,
                                            bf16_t* __restrict__ out2) {
  if (EPI == EPI_BIAS_SILU) {
    const float z = v + bias[col];
    out[o] = z;
    out2[o] = f2bf(silu(z));
  } else if (EPI == EPI_BIAS) {
    out[o] = v + bias[col];
  } else if (EPI == EPI_DSILU || EPI == EPI_DSILU_SUM) {
    v *= dsilu(aux[o]);
    if (EPI == EPI_DSILU) out[o] = v;
    out2[o] = f2bf(v);
  } else {
    atomicAdd(out + o, v);
  }
  return v;
}

// ------------------------------------------------------------ tiled GEMM ----
// The same product for operands with 16-byte aligned rows (every layer of the
// network): 16-byte global loads one K step ahead of the MFMAs, both operands
// staged as [row][k] (a k-major operand is transposed on the way, four k rows
// at a time), fragments read as one ds_read_b64.  Each output accumulates k in
// steps of 16 in order, as in gemm_bf16_kernel: same bits.
// 16384 rows: a hidden layer 28 -> 17 us (its 34 MB take 7 at HBM rate; 128 x
// 128 tiles, one workgroup per CU: 25), backward data 38 -> 17 us, a weight
// gradient 64 -> 19 us; a training step 658 -> 217 us.
// Row stride of the staged operands, 36 elements for 32 of k and 144 for 128: the
// fragment reads (16 rows, 8 bytes) and the transposing writes fall on all banks.
constexpr int tile_stride(int TK) { return TK == 32 ? 36 : TK + 16; }

// Stages rows [r0, r0 + R) x k [k0, k0 + TK) of a [row][k] operand (T: stored
// [k][row]).  TAIL: its stored rows are not whole 8-element pieces.
template <int R, int TK, bool T, bool TAIL>
struct TileLoad {
  static constexpr int KP = TK / 8, NT = (R * KP + 255) / 256;  // 16-byte pieces per row, per thread
  static constexpr int KQ = TK / 4, TASKS = KQ * R / 8;         // T: blocks of four k rows x eight rows
  static_assert(!T || TASKS <= 256, "one transposing block per thread");
  uint4 v[T ? 4 : NT];
  // n elements from p, in one 16-byte load.  TAIL: n may be less than 8; what lies
  // behind the elements is in the same row's padding or, in the last row, may be
  // behind the allocation, so that its end is read element by element
  __device__ static inline uint4 piece(const bf16_t* __restrict__ p, int n, bool last) {
    if (!TAIL || n >= 8 || !last) return *reinterpret_cast<const uint4*>(p);
    unsigned w[4] = {0, 0, 0, 0};
#pragma unroll 1
    for (int q = 0; q < n; ++q) w[q / 2] |= (unsigned)p[q] << (16 * (q % 2));
    return uint4{w[0], w[1], w[2], w[3]};
  }
  __device__ inline void load(const bf16_t* __restrict__ P, int ld, int r0, int rows, int k0, int kend) {
    const int tid = threadIdx.x;
    if constexpr (!T) {
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const int e = tid + 256 * i, r = e / KP, k = k0 + (e % KP) * 8;
        uint4 x = {0, 0, 0, 0};
        if (r < R && r0 + r < rows && k < kend) {
          x = piece(P + (int64_t)(r0 + r) * ld + k, kend - k, r0 + r == rows - 1);
          if (TAIL && k + 8 > kend) {  // the tail of the last piece is not part of K
            unsigned* w = reinterpret_cast<unsigned*>(&x);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              if (k + 2 * q >= kend) w[q] = 0;
              else if (k + 2 * q + 1 >= kend) w[q] &= 0xffffu;
            }
          }
        }
        v[i] = x;
      }
    } else {
      const int kq = tid % KQ, r = tid / KQ * 8;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int k = k0 + kq * 4 + q;
        v[q] = tid < TASKS && k < kend && r0 + r < rows
                   ? piece(P + (int64_t)k * ld + r0 + r, rows - r0 - r, k == kend - 1)
                   : uint4{0, 0, 0, 0};
      }
    }
  }
  __device__ inline void store(bf16_t* __restrict__ S) {
    constexpr int TS = tile_stride(TK);
    const int tid = threadIdx.x;
    if constexpr (!T) {
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const int e = tid + 256 * i, r = e / KP;
        if (r < R) {
          uint2* d = reinterpret_cast<uint2*>(S + r * TS + (e % KP) * 8);
          d[0] = uint2{v[i].x, v[i].y};
          d[1] = uint2{v[i].z, v[i].w};
        }
      }
    } else if (tid < TASKS) {
      const int kq = tid % KQ, r = tid / KQ * 8;
      const unsigned* w0 = reinterpret_cast<const unsigned*>(&v[0]);
      const unsigned* w1 = reinterpret_cast<const unsigned*>(&v[1]);
      const unsigned* w2 = reinterpret_cast<const unsigned*>(&v[2]);
      const unsigned* w3 = reinterpret_cast<const unsigned*>(&v[3]);
#pragma unroll
      for (int p = 0; p < 4; ++p) {  // rows r + 2p and r + 2p + 1
        *reinterpret_cast<uint2*>(S + (r + 2 * p) * TS + kq * 4) =
            uint2{(w0[p] & 0xffffu) | (w1[p] << 16), (w2[p] & 0xffffu) | (w3[p] << 16)};
        *reinterpret_cast<uint2*>(S + (r + 2 * p + 1) * TS + kq * 4) =
            uint2{(w0[p] >> 16) | (w1[p] & 0xffff0000u), (w2[p] >> 16) | (w3[p] & 0xffff0000u)};
      }
    }
  }
};

// Workgroup tile BM x BN, K in steps of TK, 4 waves of (BM / WM) x
// (BN / (4 / WM)).  TA, TB as in gemm_bf16_kernel; blockIdx.z splits the K
// steps (EPI_ATOMIC only).  A workgroup walks the row tiles blockIdx.y,
// blockIdx.y + gridDim.y, ...
template <int BM, int BN, int TK, int WM, bool TA, bool TB, int EPI, bool TAIL>
__global__ void __launch_bounds__(256) gemm_tile_kernel(int M, int N, int K, const bf16_t* __restrict__ A, int lda,
                                                        const bf16_t* __restrict__ B, int ldb,
                                                        const float* __restrict__ bias, const float* __restrict__ aux,
                                                        float* __restrict__ out, bf16_t* __restrict__ out2, int ldc) {
  constexpr int WN = 4 / WM, FM = BM / WM / 16, FN = BN / WN / 16, TS = tile_stride(TK);
  __shared__ __align__(16) bf16_t As[BM * TS];
  __shared__ __align__(16) bf16_t Bs[BN * TS];
  __shared__ float csum[EPI == EPI_DSILU_SUM ? WM * BN : 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, lg = lane >> 4;
  const int n0 = blockIdx.x * BN;
  const int wm = (wave / WN) * (BM / WM), wn = (wave % WN) * (BN / WN);
  const int steps = (K + TK - 1) / TK, per = (steps + gridDim.z - 1) / gridDim.z;
  const int s0 = blockIdx.z * per, s1 = min(steps, s0 + per);
  // nothing to add; the other epilogues store their result for K = 0 too
  if (EPI == EPI_ATOMIC && s0 >= s1) return;
  float sum[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) sum[j] = 0.f;
  for (int m0 = blockIdx.y * BM; m0 < M; m0 += gridDim.y * BM) {
    f32x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    TileLoad<BM, TK, TA, TAIL> la;
    TileLoad<BN, TK, !TB, TAIL> lb;
    la.load(A, lda, m0, M, s0 * TK, K);
    lb.load(B, ldb, n0, N, s0 * TK, K);
    for (int s = s0; s < s1; ++s) {
      __syncthreads();  // the last step's fragments are read
      la.store(As);
      lb.store(Bs);
      __syncthreads();
      if (s + 1 < s1) {
        la.load(A, lda, m0, M, (s + 1) * TK, K);
        lb.load(B, ldb, n0, N, (s + 1) * TK, K);
      }
#pragma unroll
      for (int kk = 0; kk < TK; kk += 16) {
        bf16x4 a[FM], b[FN];
#pragma unroll
        for (int i = 0; i < FM; ++i)
          a[i] = *reinterpret_cast<const bf16x4*>(As + (wm + i * 16 + li) * TS + kk + 4 * lg);
#pragma unroll
        for (int j = 0; j < FN; ++j)
          b[j] = *reinterpret_cast<const bf16x4*>(Bs + (wn + j * 16 + li) * TS + kk + 4 * lg);
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[i], b[j], acc[i][j], 0, 0, 0);
      }
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int col = n0 + wn + j * 16 + li;
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int row = m0 + wm + i * 16 + 4 * lg + q;
          if (row < M && col < N)
            sum[j] += gemm_store<EPI>(acc[i][j][q], row, col, (int64_t)row * ldc + col, bias, aux, out, out2);
        }
    }
  }
  if constexpr (EPI == EPI_DSILU_SUM) {  // one atomic per column and workgroup
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const float t = xor32_sum(xor16_sum(sum[j]));
      if (lg == 0) csum[(wave / WN) * BN + wn + j * 16 + li] = t;
    }
    __syncthreads();
    for (int c = threadIdx.x; c < BN; c += 256) {
      float t = 0.f;
#pragma unroll
      for (int w = 0; w < WM; ++w) t += csum[w * BN + c];
      if (n0 + c < N) atomicAdd(out + n0 + c, t);
    }
  }
}

// C[M][N] = op(A)[M][K] * op(B)[K][N], BF16 operands, FP32 accumulation on
// v_mfma_f32_16x16x16bf16_1k, for any alignment.  A(m,k) = TA ? A[k*lda+m] : A[m*lda+k];
// B(k,n) = TB ? B[n*ldb+k] : B[k*ldb+n].  Workgroup: 64x64 tile, 4 waves of
// 32x32 (2x2 MFMA blocks).  blockIdx.z splits K into gridDim.z ranges (only
// with EPI_ATOMIC).  Out-of-range rows/cols/ks are zero-filled.
template <bool TA, bool TB, int EPI>
__global__ void __launch_bounds__(256) gemm_bf16_kernel(int M, int N, int K, const bf16_t* __restrict__ A, int lda,
                                                        const bf16_t* __restrict__ B, int ldb,
                                                        const float* __restrict__ bias, const float* __restrict__ aux,
                                                        float* __restrict__ out, bf16_t* __restrict__ out2, int ldc) {
  __shared__ bf16_t As[GBM][GBK + 4];
  __shared__ bf16_t Bs[GBK][GBN + 4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m0 = blockIdx.y * GBM, n0 = blockIdx.x * GBN;
  const int kchunk = (K + gridDim.z - 1) / gridDim.z;
  const int kbeg = blockIdx.z * kchunk, kend = min(K, kbeg + kchunk);
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  for (int k0 = kbeg; k0 < kend; k0 += GBK) {
    // stage 64x16 of A and 16x64 of B (4 elements per thread each)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int e = tid + r * 256;
      const int am = e / GBK, ak = e % GBK;
      const int gm = m0 + am, gk = k0 + ak;
      bf16_t va = 0;
      if (gm < M && gk < kend) va = TA ? A[(int64_t)gk * lda + gm] : A[(int64_t)gm * lda + gk];
      As[am][ak] = va;
      const int bk = e / GBN, bn = e % GBN;
      const int gk2 = k0 + bk, gn = n0 + bn;
      bf16_t vb = 0;
      if (gn < N && gk2 < kend) vb = TB ? B[(int64_t)gn * ldb + gk2] : B[(int64_t)gk2 * ldb + gn];
      Bs[bk][bn] = vb;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        bf16x4 a, b;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          a[q] = (short)As[wm + i * 16 + (lane & 15)][4 * (lane >> 4) + q];
          b[q] = (short)Bs[4 * (lane >> 4) + q][wn + j * 16 + (lane & 15)];
        }
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[i][j], 0, 0, 0);
      }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = m0 + wm + i * 16 + 4 * (lane >> 4) + q;
        const int col = n0 + wn + j * 16 + (lane & 15);
        if (row >= M || col >= N) continue;
        gemm_store<EPI>(acc[i][j][q], row, col, (int64_t)row * ldc + col, bias, aux, out, out2);
      }
}

// g = 2 (pred - Y) mask / nvalid on the padded output (ld = 32); BF16 and
// FP32 copies of g; loss accumulated into *loss (FP64).  At most 512
// workgroups: the loss is one address, and with an atomic per 256 elements
// that was the time (27 -> 9 us for 16384 rows).
__global__ void __launch_bounds__(256) mse_grad_kernel(int64_t n, const float* __restrict__ pred,
                                                       const float* __restrict__ Y, const float* __restrict__ mask,
                                                       float inv_n, float* __restrict__ g32, bf16_t* __restrict__ g16,
                                                       double* __restrict__ loss) {
  __shared__ double red[4];
  double l = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const float d = (pred[i] - Y[i]) * mask[i];
    l += (double)d * d * inv_n;
    const float g = 2.0f * d * inv_n;
    g32[i] = g;
    g16[i] = f2bf(g);
  }
  l = wave_sum_last(l);
  if ((threadIdx.x & 63) == 63) red[threadIdx.x >> 6] = l;
  __syncthreads();
  if (threadIdx.x == 0) atomicAdd(loss, red[0] + red[1] + red[2] + red[3]);
}

// db[n] = sum_m dZ[m][n] in a fixed order, so that a bias gradient repeats bit
// for bit (Adam divides small gradients by themselves: a last bit here moves the
// next step's loss by up to 1e-8): CS_ROWS chains over every CS_ROWS-th row, then
// a tree.  The chains of 32 columns x 8 rows a workgroup, whole cache lines, all
// CUs; the tree is colsum_kernel over their results.  Memory-bound: 16384 x 256
// in 9 us with the tree (the matrix at HBM rate: 4), 27 with colsum_kernel
// alone, whose few workgroups take 16-byte pieces, 32 with a workgroup per column.
constexpr int CS_ROWS = 256, CS_COLS = 4;

template <int AHEAD>
__device__ __forceinline__ float colsum_chain(int M, const float* __restrict__ dz, int ld, int t, int n) {
  float s = 0.f;
  for (int64_t m = t; m < M; m += CS_ROWS * AHEAD) {
    float v[AHEAD];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) v[u] = m + u * CS_ROWS < M ? dz[(m + u * CS_ROWS) * ld + n] : 0.f;
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) s += v[u];
  }
  return s;
}

__global__ void __launch_bounds__(256) colsum_chain_kernel(int M, int N, const float* __restrict__ dz, int ld,
                                                           float* __restrict__ part) {
  const int n = blockIdx.x * 32 + threadIdx.x % 32, t = blockIdx.y * 8 + threadIdx.x / 32;
  if (n < N) part[t * N + n] = colsum_chain<32>(M, dz, ld, t, n);
}

__global__ void __launch_bounds__(CS_COLS * CS_ROWS) colsum_kernel(int M, int N, const float* __restrict__ dz, int ld,
                                                                   float* __restrict__ db) {
  __shared__ float red[CS_ROWS][CS_COLS];
  const int c = threadIdx.x % CS_COLS, t = threadIdx.x / CS_COLS, n = blockIdx.x * CS_COLS + c;
  red[t][c] = n < N ? colsum_chain<8>(M, dz, ld, t, n) : 0.f;
  for (int off = 32; off > 0; off >>= 1) {
    __syncthreads();
    if (t % 64 < off) red[t][c] += red[t + off][c];
  }
  __syncthreads();
  if (t == 0 && n < N) db[n] = red[0][c] + red[64][c] + red[128][c] + red[192][c];
}

// Adam on FP32 master weights; BF16 working copy refreshed.
__global__ void adam_kernel(int64_t n, float* __restrict__ w, bf16_t* __restrict__ w16, const float* __restrict__ g,
                            float* __restrict__ m, float* __restrict__ v, float lr, float b1, float b2, float eps,
                            float c1, float c2) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float wi = w[i] - lr * (mi * c1) / (sqrtf(vi * c2) + eps);
  w[i] = wi;
  if (w16) w16[i] = f2bf(wi);
}

// Pair features.  pairs[p] = (global atom a, global atom b); rows padded to 64
// BF16 columns (43 used) and an FP32 copy (ld 64) for checks.
__global__ void pair_features_kernel(int64_t P, const int* __restrict__ pairs, const int* __restrict__ atm,
                                     const double* __restrict__ env, bf16_t* __restrict__ X16,
                                     float* __restrict__ X32, unsigned char* __restrict__ valid) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= P) return;
  const int a = pairs[2 * p], b = pairs[2 * p + 1];
  const double* Ra = env + atm[a * ATM_SLOTS + 1];
  const double* Rb = env + atm[b * ATM_SLOTS + 1];
  const double bohr = 0.52917721092;
  const double vx = (Rb[0] - Ra[0]) * bohr, vy = (Rb[1] - Ra[1]) * bohr, vz = (Rb[2] - Ra[2]) * bohr;
  const double d = sqrt(vx * vx + vy * vy + vz * vz);
  float f[64];
#pragma unroll
  for (int k = 0; k < 64; ++k) f[k] = 0.f;
  const int za = atm[a * ATM_SLOTS], zb = atm[b * ATM_SLOTS];
  const int ea = za == 1 ? 0 : (za == 6 ? 1 : (za == 7 ? 2 : 3));
  const int eb = zb == 1 ? 0 : (zb == 6 ? 1 : (zb == 7 ? 2 : 3));
  f[ea] = 1.f;
  f[4 + eb] = 1.f;
#pragma unroll
  for (int k = 0; k < 32; ++k) {
    const double mu = 5.0 * k / 31.0;
    const double t = (d - mu) / 0.15;
    f[8 + k] = (float)exp(-0.5 * t * t);
  }
  if (d > 0.0) {
    f[40] = (float)(vx / d);
    f[41] = (float)(vy / d);
    f[42] = (float)(vz / d);
  }
#pragma unroll
  for (int k = 0; k < 64; ++k) {
    X16[p * 64 + k] = f2bf(f[k]);
    if (X32) X32[p * 64 + k] = f[k];
  }
  valid[p] = d < 5.0 ? 1 : 0;
}

// Targets: Y[p][r*5+c] = D[AO(a)+r][AO(b)+c] of the pair's molecule (ld 32),
// mask 1 where r < nao(a), c < nao(b) and the pair is within the cutoff.
__global__ void pair_targets_kernel(int64_t P, const int* __restrict__ pinfo, const unsigned char* __restrict__ valid,
                                    const BatchMol* __restrict__ mols, const double* __restrict__ D,
                                    float* __restrict__ Y, float* __restrict__ mask) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= P * 32) return;
  const int64_t p = t >> 5;
  const int e = (int)(t & 31);
  const int* q = pinfo + 5 * p;  // mol, ao_a, n_a, ao_b, n_b
  const int r = e / 5, c = e % 5;
  float y = 0.f, mk = 0.f;
  if (e < 25 && r < q[2] && c < q[4] && valid[p]) {
    const BatchMol Mo = mols[q[0]];
    y = (float)D[Mo.mat0 + (int64_t)(q[1] + r) * Mo.nao + q[3] + c];
    mk = 1.f;
  }
  Y[t] = y;
  mask[t] = mk;
}

// Predicted blocks into D (zero-initialised by the caller); pairs beyond the
// cutoff contribute nothing.
__global__ void pair_assemble_kernel(int64_t P, const int* __restrict__ pinfo, const unsigned char* __restrict__ valid,
                                     const BatchMol* __restrict__ mols, const float* __restrict__ pred,
                                     double* __restrict__ D) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= P * 32) return;
  const int64_t p = t >> 5;
  const int e = (int)(t & 31);
  const int* q = pinfo + 5 * p;
  const int r = e / 5, c = e % 5;
  if (e < 25 && r < q[2] && c < q[4] && valid[p]) {
    const BatchMol Mo = mols[q[0]];
    D[Mo.mat0 + (int64_t)(q[1] + r) * Mo.nao + q[3] + c] = (double)pred[t];
  }
}

__global__ void f32_to_bf16_kernel(int64_t n, const float* __restrict__ x, bf16_t* __restrict__ y) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = f2bf(x[i]);
}

template <int BM, int BN, int TK, int WM, bool TA, bool TB, int EPI>
static void launch_tile(int M, int N, int K, const void* A, int lda, const void* B, int ldb, const float* bias,
                        const float* aux, float* out, void* out2, int ldc, int rows, int ksplit, hipStream_t st) {
  dim3 grid((N + BN - 1) / BN, rows, ksplit);
  auto run = [&](auto kernel) {
    kernel<<<grid, 256, 0, st>>>(M, N, K, (const bf16_t*)A, lda, (const bf16_t*)B, ldb, bias, aux, out, (bf16_t*)out2,
                                 ldc);
  };
  if ((TA ? M : K) % 8 || (TB ? K : N) % 8)
    run(gemm_tile_kernel<BM, BN, TK, WM, TA, TB, EPI, true>);
  else
    run(gemm_tile_kernel<BM, BN, TK, WM, TA, TB, EPI, false>);
}

// Tiled form where every row starts 16-byte aligned and the rows are a multiple
// of 8 elements apart (the pieces it loads): 64 x 64 tiles, 64 x 32 for the
// narrow layer.
template <bool TA, bool TB, int EPI>
static int launch_gemm(int M, int N, int K, const void* A, int lda, const void* B, int ldb, const float* bias,
                       const float* aux, float* out, void* out2, int ldc, int ksplit, hipStream_t st) {
  const bool aligned = (((uintptr_t)A | (uintptr_t)B) & 15) == 0 && lda % 8 == 0 && ldb % 8 == 0 &&
                       ((TA ? M : K) + 7) / 8 * 8 <= lda && ((TB ? K : N) + 7) / 8 * 8 <= ldb;
  // the grid's y extent is limited to 65535; column sums: few workgroups per
  // column, each of which adds to the same addresses
  const int mt = (M + 63) / 64, rows = EPI == EPI_DSILU_SUM ? (mt < 256 ? mt : 256) : (mt < 65535 ? mt : 65535);
  if (aligned) {
    if constexpr (EPI == EPI_ATOMIC) {
      // steps of 128 k: the loop is bound by the latency of its loads.  K
      // ranges for two workgroups per CU: every range adds all outputs
      const int tiles = mt * ((N + 63) / 64), want = (512 + tiles - 1) / tiles;
      const int ks = ksplit < want ? ksplit : want;
      if (N <= 32)
        launch_tile<64, 32, 128, 4, TA, TB, EPI>(M, N, K, A, lda, B, ldb, bias, aux, out, out2, ldc, rows, ks, st);
      else
        launch_tile<64, 64, 128, 2, TA, TB, EPI>(M, N, K, A, lda, B, ldb, bias, aux, out, out2, ldc, rows, ks, st);
    } else if (N <= 32) {
      launch_tile<64, 32, 32, 4, TA, TB, EPI>(M, N, K, A, lda, B, ldb, bias, aux, out, out2, ldc, rows, 1, st);
    } else {
      launch_tile<64, 64, 32, 2, TA, TB, EPI>(M, N, K, A, lda, B, ldb, bias, aux, out, out2, ldc, rows, 1, st);
    }
  } else if constexpr (EPI == EPI_DSILU_SUM) {
    PSCF_REQUIRE(false, "pscf_mlp_gemm: op 4 needs 16-byte aligned rows");
  } else {
    dim3 grid((N + GBN - 1) / GBN, (M + GBM - 1) / GBM, ksplit);
    gemm_bf16_kernel<TA, TB, EPI><<<grid, 256, 0, st>>>(M, N, K, (const bf16_t*)A, lda, (const bf16_t*)B, ldb, bias,
                                                        aux, out, (bf16_t*)out2, ldc);
  }
  PSCF_HIP(hipGetLastError());
  return PSCF_OK;
}

}  // namespace pscf

using namespace pscf;

// op: 0 = forward hidden (X W + b, SiLU; out = Z FP32, out2 = H BF16)
//     1 = forward output (X W + b; out FP32)
//     2 = backward data (dY W^T, times dsilu(aux = Z of the layer below); out FP32, out2 BF16)
//     3 = weight gradient (X^T dY accumulated into out with atomics; ksplit > 1 allowed)
//     4 = as 2, but no FP32 copy: out2 BF16, and out[n] += the column sums (the bias gradient)
extern "C" int pscf_mlp_gemm(int op, int M, int N, int K, const void* d_A, int lda, const void* d_B, int ldb,
                             const float* d_bias, const float* d_aux, float* d_out, void* d_out2, int ldc, int ksplit,
                             void* stream) {
  PSCF_REQUIRE(M >= 0 && N >= 0 && K >= 0 && d_A && d_B && d_out, "pscf_mlp_gemm: bad arguments");
  PSCF_REQUIRE(ksplit >= 1 && (ksplit == 1 || op == 3), "pscf_mlp_gemm: ksplit > 1 only for weight gradients");
  if (M == 0 || N == 0) return PSCF_OK;
  hipStream_t st = (hipStream_t)stream;
  switch (op) {
    case 0:
      PSCF_REQUIRE(d_bias && d_out2, "pscf_mlp_gemm: forward needs bias and BF16 output");
      return launch_gemm<false, false, EPI_BIAS_SILU>(M, N, K, d_A, lda, d_B, ldb, d_bias, nullptr, d_out, d_out2, ldc,
                                                      1, st);
    case 1:
      PSCF_REQUIRE(d_bias, "pscf_mlp_gemm: forward needs bias");
      return launch_gemm<false, false, EPI_BIAS>(M, N, K, d_A, lda, d_B, ldb, d_bias, nullptr, d_out, nullptr, ldc, 1,
                                                 st);
    case 2:
      PSCF_REQUIRE(d_aux && d_out2, "pscf_mlp_gemm: backward needs Z and BF16 output");
      return launch_gemm<false, true, EPI_DSILU>(M, N, K, d_A, lda, d_B, ldb, nullptr, d_aux, d_out, d_out2, ldc, 1,
                                                 st);
    case 4:
      PSCF_REQUIRE(d_aux && d_out2, "pscf_mlp_gemm: backward needs Z and BF16 output");
      return launch_gemm<false, true, EPI_DSILU_SUM>(M, N, K, d_A, lda, d_B, ldb, nullptr, d_aux, d_out, d_out2, ldc,
                                                     1, st);
    case 3:
      return launch_gemm<true, false, EPI_ATOMIC>(M, N, K, d_A, lda, d_B, ldb, nullptr, nullptr, d_out, nullptr, ldc,
                                                  ksplit, st);
    default:
      break;
  }
  PSCF_REQUIRE(false, "pscf_mlp_gemm: bad op %d", op);
  return PSCF_EINVAL;
}

extern "C" int pscf_mlp_mse_grad(int B, const float* d_pred, const float* d_Y, const float* d_mask, float inv_n,
                                 float* d_g32, void* d_g16, double* d_loss, void* stream) {
  PSCF_REQUIRE(B >= 0 && d_pred && d_Y && d_mask && d_g32 && d_g16 && d_loss, "pscf_mlp_mse_grad: bad arguments");
  if (B == 0) return PSCF_OK;
  const int64_t n = (int64_t)B * 32, blocks = (n + 255) / 256;
  mse_grad_kernel<<<(unsigned)(blocks < 512 ? blocks : 512), 256, 0, (hipStream_t)stream>>>(
      n, d_pred, d_Y, d_mask, inv_n, d_g32, (bf16_t*)d_g16, d_loss);
  PSCF_HIP(hipGetLastError());
  return PSCF_OK;
}

static int colsum(int M, int N, const float* dz, int ld, float* db, float* ws, hipStream_t st) {
  if (ws) {
    colsum_chain_kernel<<<dim3((N + 31) / 32, CS_ROWS / 8), 256, 0, st>>>(M, N, dz, ld, ws);
    PSCF_HIP(hipGetLastError());
  }
  colsum_kernel<<<(N + CS_COLS - 1) / CS_COLS, CS_COLS * CS_ROWS, 0, st>>>(ws ? CS_ROWS : M, N, ws ? ws : dz,
                                                                          ws ? N : ld, db);
  PSCF_HIP(hipGetLastError());
  return PSCF_OK;
}

extern "C" int pscf_mlp_colsum(int M, int N, const float* d_dz, int ld, float* d_db, void* stream) {
  PSCF_REQUIRE(M >= 0 && N > 0 && d_dz && d_db, "pscf_mlp_colsum: bad arguments");
  return colsum(M, N, d_dz, ld, d_db, nullptr, (hipStream_t)stream);
}

extern "C" int pscf_mlp_colsum_ws(int M, int N, const float* d_dz, int ld, float* d_db, float* d_ws, void* stream) {
  PSCF_REQUIRE(M >= 0 && N > 0 && N <= 1 << 20 && d_dz && d_db && d_ws, "pscf_mlp_colsum_ws: bad arguments");
  return colsum(M, N, d_dz, ld, d_db, d_ws, (hipStream_t)stream);
}

extern "C" int pscf_mlp_adam(int64_t n, float* d_w, void* d_w16, const float* d_g, float* d_m, float* d_v, float lr,
                             float b1, float b2, float eps, int step, void* stream) {
  PSCF_REQUIRE(n >= 0 && step >= 1 && d_w && d_g && d_m && d_v, "pscf_mlp_adam: bad arguments");
  if (n == 0) return PSCF_OK;
  const float c1 = 1.f / (1.f - powf(b1, (float)step)), c2 = 1.f / (1.f - powf(b2, (float)step));
  adam_kernel<<<(unsigned)((n + 255) / 256), 256, 0, (hipStream_t)stream>>>(n, d_w, (bf16_t*)d_w16, d_g, d_m, d_v, lr,
                                                                          b1, b2, eps, c1, c2);
  PSCF_HIP(hipGetLastError());
  return PSCF_OK;
}

extern "C" int pscf_mlp_to_bf16(int64_t n, const float* d_x, void* d_y, void* stream) {
  PSCF_REQUIRE(n >= 0 && (n == 0 || (d_x && d_y)), "pscf_mlp_to_bf16: bad arguments");
  if (n == 0) return PSCF_OK;
  f32_to_bf16_kernel<<<(unsigned)((n + 255) / 256), 256, 0, (hipStream_t)stream>>>(n, d_x, (bf16_t*)d_y);
  PSCF_HIP(hipGetLastError());
  return PSCF_OK;
}

extern "C" int pscf_pair_features(int64_t P, const int* d_pairs, const int* d_atm, const double* d_env, void* d_X16,
                                  float* d_X32, unsigned char* d_valid, void* stream) {
  PSCF_REQUIRE(P >= 0 && (P == 0 || (d_pairs && d_atm && d_env && d_X16 && d_valid)), "pscf_pair_features: bad arguments");
  if (P == 0) return PSCF_OK;
  pair_features_kernel<<<(unsigned)((P + 255) / 256), 256, 0, (hipStream_t)stream>>>(P, d_pairs, d_atm, d_env,
                                                                                   (bf16_t*)d_X16, d_X32, d_valid);
  PSCF_HIP(hipGetLastError());
  return PSCF_OK;
}

extern "C" int pscf_pair_targets(int64_t P, const int* d_pinfo, const unsigned char* d_valid, const void* d_mols,
                                 const double* d_D, float* d_Y, float* d_mask, void* stream) {
  PSCF_REQUIRE(P >= 0 && (P == 0 || (d_pinfo && d_valid && d_mols && d_D && d_Y && d_mask)),
               "pscf_pair_targets: bad arguments");
  if (P == 0) return PSCF_OK;
  pair_targets_kernel<<<(unsigned)((P * 32 + 255) / 256), 256, 0, (hipStream_t)stream>>>(
      P, d_pinfo, d_valid, (const BatchMol*)d_mols, d_D, d_Y, d_mask);
  PSCF_HIP(hipGetLastError());
  return PSCF_OK;
}

extern "C" int pscf_pair_assemble(int64_t P, const int* d_pinfo, const unsigned char* d_valid, const void* d_mols,
                                  const float* d_pred, double* d_D, void* stream) {
  PSCF_REQUIRE(P >= 0 && (P == 0 || (d_pinfo && d_valid && d_mols && d_pred && d_D)),
               "pscf_pair_assemble: bad arguments");
  if (P == 0) return PSCF_OK;
  pair_assemble_kernel<<<(unsigned)((P * 32 + 255) / 256), 256, 0, (hipStream_t)stream>>>(
      P, d_pinfo, d_valid, (const BatchMol*)d_mols, d_pred, d_D);
  PSCF_HIP(hipGetLastError());
  return PSCF_OK;
}
