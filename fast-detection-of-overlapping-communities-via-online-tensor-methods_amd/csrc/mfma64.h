// FP64 MFMA output tiles shared by the whitening's tall products, the adjoint and the power method (device code).
#pragma once

#include "common.h"

namespace mmsb {

// A T x T block of the output (T = 32 or 64) per workgroup of four waves, each wave a (T/2) x (T/2)
// quadrant of 16 x 16 v_mfma_f64_16x16x4f64 blocks (lane l supplies A[l % 16][l / 16] and
// B[l / 16][l % 16]; accumulator register g of lane l holds D[4 g + l / 16][l % 16]). The reduction runs
// in LDS stages of KS, the next stage's global loads in flight in registers during the MFMAs.
// Row-major stages pad a row to KS + 4 doubles and k-major ones to T + 16, which spreads the 16 rows
// (and the 4 k of a lane group) of a fragment read over all banks.
template <int T>
constexpr int stage_k() { return T == 32 ? 32 : 16; }

__device__ inline doublex4 mma64(double a, double b, doublex4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }

template <int NP, int T>
struct NnStage {
  double a[NP][T][stage_k<T>() + 4];
  double b[stage_k<T>()][T + 16];
};

template <int T>
struct TnStage {
  double a[stage_k<T>()][T + 16];
  double b[stage_k<T>()][T + 16];
};

// acc[p] += X_p[row0 .. row0 + T, :] C[:, c0 .. c0 + T) for NP operands sharing C [kk x q] (row-major, leading
// dimension q); rows from `rows` and columns from q on read as zero. With NM > 0 also msum[s] = the
// calling thread's part of sum_i mu_s[i] C[i][c0 + threadIdx.x % T].
template <int NP, int T, int NM, typename TX>
__device__ inline void nn_tile(doublex4 (&acc)[NP][T / 32][T / 32], NnStage<NP, T>& S, const TX* const (&X)[NP], int64_t ldx,
                               int64_t row0, int64_t rows, const double* __restrict__ C, int32_t kk, int32_t q, int32_t c0,
                               const double* const* mu, double* msum) {
  constexpr int KS = stage_k<T>(), E = T * KS / 256, U = T / 32;
  const int t = threadIdx.x, l = t & 63, w = t >> 6;
  const int ai = (T / 2) * (w >> 1), bj = (T / 2) * (w & 1);
  const int xk = t % KS, xr = t / KS, cc = t % T, ck = T == 64 ? __builtin_amdgcn_readfirstlane(t >> 6) : t / T;
  TX rx[NP][E];
  double rc[E];
  auto load = [&](int kb) {
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int64_t row = row0 + xr + (256 / KS) * e;
        rx[p][e] = (kb + xk < kk && row < rows) ? X[p][row * ldx + kb + xk] : (TX)0;
      }
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int k = kb + ck + (256 / T) * e;
      const bool in = k < kk && c0 + cc < q;
      rc[e] = in ? C[(int64_t)k * q + c0 + cc] : 0.0;
      if constexpr (NM > 0) {
#pragma unroll
        for (int m = 0; m < NM; ++m) msum[m] = fma(k < kk ? mu[m][k] : 0.0, rc[e], msum[m]);
      }
    }
  };
  load(0);
  for (int kb = 0; kb < kk; kb += KS) {
    __syncthreads();
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
      for (int e = 0; e < E; ++e) S.a[p][xr + (256 / KS) * e][xk] = (double)rx[p][e];
#pragma unroll
    for (int e = 0; e < E; ++e) S.b[ck + (256 / T) * e][cc] = rc[e];
    __syncthreads();
    if (kb + KS < kk) load(kb + KS);
#pragma unroll
    for (int k4 = 0; k4 < KS; k4 += 4) {
      double b[U];
#pragma unroll
      for (int v = 0; v < U; ++v) b[v] = S.b[k4 + (l >> 4)][bj + 16 * v + (l & 15)];
#pragma unroll
      for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const double a = S.a[p][ai + 16 * u + (l & 15)][k4 + (l >> 4)];
#pragma unroll
          for (int v = 0; v < U; ++v) acc[p][u][v] = mma64(a, b[v], acc[p][u][v]);
        }
    }
  }
}

// acc += A[r0 .. r1, i0 .. i0 + T)^T B[r0 .. r1, j0 .. j0 + T); columns from p (A) and q (B) on read as zero.
template <int T, typename TA, typename TB>
__device__ inline void tn_tile(doublex4 (&acc)[T / 32][T / 32], TnStage<T>& S, const TA* __restrict__ A, int64_t lda, int32_t p,
                               int32_t i0, const TB* __restrict__ B, int64_t ldb, int32_t q, int32_t j0, int64_t r0,
                               int64_t r1) {
  constexpr int KS = stage_k<T>(), E = T * KS / 256, U = T / 32;
  const int t = threadIdx.x, l = t & 63, w = t >> 6;
  const int ai = (T / 2) * (w >> 1), bj = (T / 2) * (w & 1);
  const int cc = t % T, cx = t / T;
  TA ra[E];
  TB rb[E];
  auto load = [&](int64_t base) {
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int64_t x = base + cx + (256 / T) * e;
      ra[e] = (x < r1 && i0 + cc < p) ? A[x * lda + i0 + cc] : (TA)0;
      rb[e] = (x < r1 && j0 + cc < q) ? B[x * ldb + j0 + cc] : (TB)0;
    }
  };
  load(r0);
  for (int64_t base = r0; base < r1; base += KS) {
    __syncthreads();
#pragma unroll
    for (int e = 0; e < E; ++e) {
      S.a[cx + (256 / T) * e][cc] = (double)ra[e];
      S.b[cx + (256 / T) * e][cc] = (double)rb[e];
    }
    __syncthreads();
    if (base + KS < r1) load(base + KS);
#pragma unroll
    for (int k4 = 0; k4 < KS; k4 += 4) {
      double a[U], b[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        a[u] = S.a[k4 + (l >> 4)][ai + 16 * u + (l & 15)];
        b[u] = S.b[k4 + (l >> 4)][bj + 16 * u + (l & 15)];
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int v = 0; v < U; ++v) acc[u][v] = mma64(a[u], b[v], acc[u][v]);
    }
  }
}

// Visits the calling lane's elements of a T x T block: f(row, col, u, v, g) with row, col within the block.
template <int T, typename F>
__device__ inline void each_elem(F f) {
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int ai = (T / 2) * (w >> 1), bj = (T / 2) * (w & 1);
#pragma unroll
  for (int v = 0; v < T / 32; ++v)
#pragma unroll
    for (int u = 0; u < T / 32; ++u)
#pragma unroll
      for (int g = 0; g < 4; ++g) f(ai + 16 * u + 4 * g + (l >> 4), bj + 16 * v + (l & 15), u, v, g);
}

}  // namespace mmsb
