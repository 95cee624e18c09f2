// FP64 one-sided (Hestenes) Jacobi SVD of a small square matrix.
//
// Replaces the k x k culaDgesvd calls of the Nystrom helpers (gemm_pinv_nys.c:288,299) and
// serves both small factorisations of the whitening stage: the SVD of the r x r triangular factor
// of the randomized range of P_BC, and (after a positive shift) the eigendecomposition of the
// r x r Rayleigh-Ritz matrix of M2. Columns are orthogonalised pairwise by plane rotations
// A <- A J, V <- V J; at convergence sigma_j = ||A_j||, U_j = A_j / sigma_j.
//
// Blocks of B consecutive columns are paired by the round-robin (circle) schedule: nblk - 1 rounds
// of disjoint block pairs per sweep. One launch per round: the workgroup of block pair (P, Q) loads
// their 2B columns of A (and of V when it is accumulated) into LDS, orthogonalises every column pair
// among them (one inner sweep of 2B - 1 inner rounds of B disjoint pairs, one wave per pair), writes
// them back and adds its rotation count to the sweep's counter, which the host reads from the fourth
// sweep on (one without rotations ends the factorisation). Plain launches keep the
// factorisation free of cooperative launches, whose global-wave-sync resource only one process on a
// GPU can hold, and a launch boundary costs less than a grid-wide barrier on this part.
#include "common.h"
#include "dense.h"
#include "wave.h"

namespace mmsb {

static constexpr int kMaxSweeps = 40;
// Widest column block of the rotations (8, 4, 2 or 1); narrower blocks are taken when the wider do
// not fit in LDS.
#ifndef MMSB_JACOBI_BMAX
#define MMSB_JACOBI_BMAX 8
#endif
// counters: [0, kMaxSweeps) rotations per sweep. A sweep without rotations ends the factorisation: every later
// round sees its predecessor's zero and returns.

size_t jacobi_workspace_bytes(int32_t r) {
  return sizeof(double) * ((size_t)r * r + (size_t)r) + sizeof(int32_t) * kMaxSweeps + 64;
}

__device__ inline double block_sum(double v, double* red) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) red[w] = v;
  __syncthreads();
  double s = 0.0;
  for (int i = 0; i < (int)(blockDim.x >> 6); ++i) s += red[i];
  return s;
}

__device__ inline void pair_of(int rp, int round, int idx, int& p, int& q) {
  // circle method: player rp-1 fixed, the others rotate
  const int m = rp - 1;
  if (idx == 0) {
    p = m;
    q = round % m;
  } else {
    p = (round + idx) % m;
    q = (round - idx + m) % m;
  }
  if (p > q) {
    const int t = p;
    p = q;
    q = t;
  }
}

__global__ void jacobi_init_kernel(int32_t r, double* __restrict__ Vw, int32_t* __restrict__ counters) {
  const int64_t rr = (int64_t)r * r;
  const int64_t gtid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t gsz = (int64_t)gridDim.x * blockDim.x;
  if (Vw)
    for (int64_t e = gtid; e < rr; e += gsz) Vw[e] = ((e / r) == (e % r)) ? 1.0 : 0.0;
  for (int64_t e = gtid; e < kMaxSweeps; e += gsz) counters[e] = 0;
}

// One round of a sweep: workgroup b handles block pair b of the round (grid = block pairs), wave g the pair g of
// every inner round. Bound by the chain of one inner round -- dot products, three wave sums, the rotation's
// divisions and square roots, the barrier -- 15 times per launch. MIN <= r <= 64 RM: a lane keeps its RM entries
// of both columns in registers from the dot products to the rotation (RM = 0: any r, entries re-read); the wave
// sums stay out of LDS (wave.h), V's columns are read while the rotation is formed, and every wave moves two
// columns between HBM and LDS with all its loads in flight. The arithmetic and its order are those of a
// lane-strided sum and a shuffle butterfly. With 8 waves two share a SIMD, so every instruction of that chain
// counts twice: 3000 cycles per inner round at r = 110 before the sums were packed and the square roots paired,
// 1600 after. A launch at r = 110 takes 16.9 us with V and 15.8 without (33.6 and 30.8 with re-read columns, LDS
// shuffles and loads in turn); a 50k-node, k = 100 whitening 14.7 -> 10.7 ms.
template <int B, bool WV, int RM, int MIN>
__global__ __launch_bounds__(64 * B) void jacobi_round_kernel(int32_t r, double* __restrict__ A, double* __restrict__ Vw,
                                                              int32_t* __restrict__ counters, int32_t sweep, int32_t round) {
  constexpr int M = RM > 0 ? RM : 1;
  extern __shared__ double lds[];          // [2B][r] columns of A, then (WV) [2B][r] columns of V
  __shared__ int nrot;
  const int32_t live = sweep > 0 ? counters[sweep - 1] : 1;  // tested once the columns' loads are on their way
  double* la = lds;
  double* lv = lds + (int64_t)2 * B * r;
  const int nblk = (r + B - 1) / B;
  const int nbp = nblk + (nblk & 1);
  const int g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), tg = threadIdx.x & 63;
  int P, Q;
  pair_of(nbp, round, blockIdx.x, P, Q);
  auto gcol = [&](int lc) -> int {  // global column of local column lc, or -1
    const int blkid = lc < B ? P : Q;
    const int c = blkid * B + (lc % B);
    return (blkid < nblk && c < r) ? c : -1;
  };
  const int c0 = gcol(g), c1 = gcol(g + B);  // the columns this wave moves
  for (int base = 0; base < r; base += 64 * M) {
    double a0[M], a1[M], v0[M], v1[M];
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const int i = base + 64 * m + tg;
      a0[m] = (c0 >= 0 && i < r) ? A[(int64_t)c0 * r + i] : 0.0;
      a1[m] = (c1 >= 0 && i < r) ? A[(int64_t)c1 * r + i] : 0.0;
      if constexpr (WV) {
        v0[m] = (c0 >= 0 && i < r) ? Vw[(int64_t)c0 * r + i] : 0.0;
        v1[m] = (c1 >= 0 && i < r) ? Vw[(int64_t)c1 * r + i] : 0.0;
      }
    }
    if (live == 0) return;  // converged in an earlier sweep (uniform)
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const int i = base + 64 * m + tg;
      if (i < r) {
        la[g * r + i] = a0[m];
        la[(g + B) * r + i] = a1[m];
        if constexpr (WV) {
          lv[g * r + i] = v0[m];
          lv[(g + B) * r + i] = v1[m];
        }
      }
    }
  }
  if (threadIdx.x == 0) nrot = 0;
  __syncthreads();
  // entry 64 m + lane of a column, the last one for lanes past the end (whose value is then zeroed)
  int at[M];
  bool in[M];
#pragma unroll
  for (int m = 0; m < M; ++m) {
    in[m] = 64 * m + tg < r;
    at[m] = in[m] ? 64 * m + tg : r - 1;
  }
  int myrot = 0;
  for (int ir = 0; ir < 2 * B - 1; ++ir) {
    int lp, lq;
    pair_of(2 * B, ir, g, lp, lq);
    if (gcol(lp) >= 0 && gcol(lq) >= 0) {
      double* ap = la + lp * r;
      double* aq = la + lq * r;
      double* vp = lv + lp * r;
      double* vq = lv + lq * r;
      double x[M], y[M], vx[M], vy[M];
      double a = 0.0, b = 0.0, gg = 0.0;
      if constexpr (RM > 0) {
#pragma unroll
        for (int m = 0; m < M; ++m) {
          x[m] = ap[at[m]];
          y[m] = aq[at[m]];
        }
        if constexpr (WV) {
#pragma unroll
          for (int m = 0; m < M; ++m) {
            vx[m] = vp[at[m]];
            vy[m] = vq[at[m]];
          }
        }
#pragma unroll
        for (int m = 0; m < M; ++m) {
          if (64 * m + 64 > MIN) {
            x[m] = in[m] ? x[m] : 0.0;
            y[m] = in[m] ? y[m] : 0.0;
          }
          a = fma(x[m], x[m], a);
          b = fma(y[m], y[m], b);
          gg = fma(x[m], y[m], gg);
        }
      } else {
        for (int i = tg; i < r; i += 64) {
          const double p = ap[i], q = aq[i];
          a = fma(p, p, a);
          b = fma(q, q, b);
          gg = fma(p, q, gg);
        }
      }
      wave_sum3(a, b, gg);
      // the two square roots of the test and of the rotation's first step in one go, in the wave's two halves
      // (gg = 0 gives an infinite or undefined zeta that nothing uses)
      const double zeta = (b - a) / (2.0 * gg);
      const double root = sqrt(tg < 32 ? fma(zeta, zeta, 1.0) : a * b);
      if (gg != 0.0 && fabs(gg) > 1e-15 * read_lane(root, 32)) {
        const double t = (zeta >= 0.0 ? 1.0 : -1.0) / (fabs(zeta) + read_lane(root, 0));
        const double c = 1.0 / sqrt(fma(t, t, 1.0));
        const double sn = c * t;
        if constexpr (RM > 0) {
#pragma unroll
          for (int m = 0; m < M; ++m) {
            const int i = 64 * m + tg;
            if (64 * m + 64 <= MIN || in[m]) {
              ap[i] = fma(c, x[m], -(sn * y[m]));
              aq[i] = fma(sn, x[m], c * y[m]);
              if constexpr (WV) {
                vp[i] = fma(c, vx[m], -(sn * vy[m]));
                vq[i] = fma(sn, vx[m], c * vy[m]);
              }
            }
          }
        } else {
          for (int i = tg; i < r; i += 64) {
            const double p = ap[i], q = aq[i];
            ap[i] = fma(c, p, -(sn * q));
            aq[i] = fma(sn, p, c * q);
          }
          if constexpr (WV) {
            for (int i = tg; i < r; i += 64) {
              const double p = vp[i], q = vq[i];
              vp[i] = fma(c, p, -(sn * q));
              vq[i] = fma(sn, p, c * q);
            }
          }
        }
        if (tg == 0) ++myrot;
      }
    }
    __syncthreads();
  }
  if (tg == 0 && myrot) atomicAdd(&nrot, myrot);
  for (int i = tg; i < r; i += 64) {
    if (c0 >= 0) A[(int64_t)c0 * r + i] = la[g * r + i];
    if (c1 >= 0) A[(int64_t)c1 * r + i] = la[(g + B) * r + i];
    if constexpr (WV) {
      if (c0 >= 0) Vw[(int64_t)c0 * r + i] = lv[g * r + i];
      if (c1 >= 0) Vw[(int64_t)c1 * r + i] = lv[(g + B) * r + i];
    }
  }
  __syncthreads();
  if (threadIdx.x == 0 && nrot) atomicAdd(counters + sweep, nrot);
}

// sw[j] = ||A_j||, one workgroup per column.
__global__ __launch_bounds__(256) void jacobi_norms_kernel(int32_t r, const double* __restrict__ A, double* __restrict__ sw) {
  __shared__ double red[4];
  for (int j = blockIdx.x; j < r; j += gridDim.x) {
    const double* aj = A + (int64_t)j * r;
    double a = 0.0;
    for (int i = threadIdx.x; i < r; i += blockDim.x) a = fma(aj[i], aj[i], a);
    a = block_sum(a, red);
    if (threadIdx.x == 0) sw[j] = sqrt(a);
    __syncthreads();
  }
}

// Columns sorted by descending norm (stable): U = A_j / sigma_j, V, sigma; the sweep count.
__global__ __launch_bounds__(256) void jacobi_sort_kernel(int32_t r, const double* __restrict__ A, const double* __restrict__ Vw,
                                                          const double* __restrict__ sw, double* __restrict__ U,
                                                          double* __restrict__ sigma, double* __restrict__ V,
                                                          const int32_t* __restrict__ counters, int32_t* __restrict__ sweeps_out) {
  __shared__ double red[4];
  for (int j = blockIdx.x; j < r; j += gridDim.x) {
    const double sj = sw[j];
    int cnt = 0;
    for (int i = threadIdx.x; i < r; i += blockDim.x) {
      const double si = sw[i];
      cnt += (si > sj || (si == sj && i < j)) ? 1 : 0;
    }
    const int rank = (int)block_sum((double)cnt, red);
    const double inv = sj > 0.0 ? 1.0 / sj : 0.0;
    const double* aj = A + (int64_t)j * r;
    for (int i = threadIdx.x; i < r; i += blockDim.x) {
      U[(int64_t)rank * r + i] = aj[i] * inv;
      if (V) V[(int64_t)rank * r + i] = Vw[(int64_t)j * r + i];
    }
    if (threadIdx.x == 0) sigma[rank] = sj;
    __syncthreads();
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    int sweeps = 0;
    while (sweeps < kMaxSweeps && counters[sweeps]) ++sweeps;
    sweeps_out[0] = sweeps + 1;  // the last one rotated nothing
  }
}

template <int B, bool WV, int RM, int MIN>
static int run_sweeps_rm(hipStream_t s, int32_t r, double* A, double* Vw, int32_t* counters) {
  const void* fn = reinterpret_cast<const void*>(jacobi_round_kernel<B, WV, RM, MIN>);
  const size_t shm = sizeof(double) * (size_t)(WV ? 4 : 2) * B * r;
  MMSB_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm));
  const int nblk = (r + B - 1) / B;
  const int nbp = nblk + (nblk & 1);
  const int npairs = nbp / 2;
  int32_t rotations = 1;
  for (int sweep = 0; sweep < kMaxSweeps && rotations; ++sweep) {
    for (int round = 0; round < nbp - 1; ++round) {
      hipLaunchKernelGGL((jacobi_round_kernel<B, WV, RM, MIN>), dim3(npairs), dim3(64 * B), shm, s, r, A, Vw, counters, sweep,
                         round);
      MMSB_LAUNCH_CHECK();
    }
    // No matrix that is not already orthogonal converges in four sweeps (random ones take 10 at r = 110, 30 at 510):
    // until then the host does not wait, and the rounds after an early convergence return at once.
    if (sweep < 3) continue;
    MMSB_HIP(hipMemcpyAsync(&rotations, counters + sweep, sizeof(int32_t), hipMemcpyDeviceToHost, s));
    MMSB_HIP(hipStreamSynchronize(s));
  }
  if (rotations)  // every sweep still rotated: the factors are not converged, so say so instead of using them
    return set_error(MMSB_ERR_NUMERIC, "jacobi: no convergence after %d sweeps (r = %d)", kMaxSweeps, r);
  return MMSB_OK;
}

// Largest r whose 2B columns of A (and of V when it is wanted) fit in the 160 KiB of LDS.
template <int B, bool WV>
constexpr int sweep_r_max() { return (160 * 1024 - 256) / (int)(sizeof(double) * 2 * (WV ? 2 : 1) * B); }

// Smallest r that comes to blocks of B columns: jacobi_svd takes blocks twice as wide while they are allowed and fit.
template <int B, bool WV>
constexpr int sweep_r_min() { return 2 * B <= MMSB_JACOBI_BMAX ? sweep_r_max<2 * B, WV>() + 1 : 1; }

template <int B, bool WV>
static int run_sweeps(hipStream_t s, int32_t r, double* A, double* Vw, int32_t* counters) {
  if constexpr (B >= 4) {  // columns in registers: up to 20 entries per lane
#define MMSB_RM(RM, MIN)                                                            \
  if constexpr (MIN <= sweep_r_max<B, WV>() && 64 * RM >= sweep_r_min<B, WV>())      \
    if (r <= 64 * RM) return run_sweeps_rm<B, WV, RM, MIN>(s, r, A, Vw, counters);
    MMSB_RM(1, 1)
    MMSB_RM(2, 65)
    MMSB_RM(4, 129)
    MMSB_RM(6, 257)
    MMSB_RM(8, 385)
    MMSB_RM(12, 513)
    MMSB_RM(20, 769)
#undef MMSB_RM
  }
  if constexpr (B < 4 || sweep_r_max<B, WV>() > 64 * 20) return run_sweeps_rm<B, WV, 0, 0>(s, r, A, Vw, counters);
  return set_error(MMSB_ERR_ARG, "jacobi: no form for r=%d in blocks of %d columns", r, B);
}

int jacobi_svd(hipStream_t s, int32_t r, double* A, double* U, double* sigma, double* V, void* work, int32_t* sweeps_out) {
  MMSB_CHECK_ARG(r >= 1 && r <= 8192, "jacobi: r=%d out of range", r);
  double* Vw = static_cast<double*>(work);
  double* sw = Vw + (size_t)r * r;
  int32_t* counters = reinterpret_cast<int32_t*>(sw + r);
  // 8-column blocks while 2B columns of A (and of V when it is wanted) fit in the 160 KiB of LDS;
  // without V the rotations touch half the data. (16-column blocks, which V-free would allow at
  // r = 510, were slower: the longer inner rounds outweighed the halved round count.)
  auto fits = [&](int b, int arrays) { return sizeof(double) * (size_t)2 * arrays * b * r + 256 <= (size_t)160 * 1024; };
  const int grid = (int)std::min<int64_t>(std::max<int64_t>(1, ((int64_t)r * r + 255) / 256), 1024);
  hipLaunchKernelGGL(jacobi_init_kernel, dim3(grid), dim3(256), 0, s, r, V ? Vw : nullptr, counters);
  MMSB_LAUNCH_CHECK();
  const int arrays = V ? 2 : 1;
  int st;
  if (MMSB_JACOBI_BMAX >= 8 && fits(8, arrays))
    st = V ? run_sweeps<8, true>(s, r, A, Vw, counters) : run_sweeps<8, false>(s, r, A, Vw, counters);
  else if (MMSB_JACOBI_BMAX >= 4 && fits(4, arrays))
    st = V ? run_sweeps<4, true>(s, r, A, Vw, counters) : run_sweeps<4, false>(s, r, A, Vw, counters);
  else if (MMSB_JACOBI_BMAX >= 2 && fits(2, arrays))
    st = V ? run_sweeps<2, true>(s, r, A, Vw, counters) : run_sweeps<2, false>(s, r, A, Vw, counters);
  else if (fits(1, arrays))
    st = V ? run_sweeps<1, true>(s, r, A, Vw, counters) : run_sweeps<1, false>(s, r, A, Vw, counters);
  else
    return set_error(MMSB_ERR_ARG, "jacobi: r=%d does not fit the LDS of one workgroup", r);
  MMSB_TRY(st);
  const int cols = std::min(r, 1024);
  hipLaunchKernelGGL(jacobi_norms_kernel, dim3(cols), dim3(256), 0, s, r, A, sw);
  MMSB_LAUNCH_CHECK();
  hipLaunchKernelGGL(jacobi_sort_kernel, dim3(cols), dim3(256), 0, s, r, A, Vw, sw, U, sigma, V, counters, sweeps_out);
  MMSB_LAUNCH_CHECK();
  return MMSB_OK;
}

}  // namespace mmsb
