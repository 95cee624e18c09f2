// Loss and exact adjoint of the implicit tensor objective with respect to Phi.
//
//   L(Phi) = theta/2 sum_ij <phi_i, phi_j>^3 - sum_i T_b(phi_i, phi_i, phi_i)
//   T_b(u,v,w) = mean_x [c3 (y_A.u)(y_B.v)(y_C.w) + c1 ((y_A.u)(y_B.v)(mu_C.w) + (y_A.u)(mu_B.v)(y_C.w)
//                + (mu_A.u)(y_B.v)(y_C.w))] + c0 (mu_A.u)(mu_B.v)(mu_C.w)
//   dL/dPhi = 3 theta Phi (G o G) - [T(I,phi,phi) + T(phi,I,phi) + T(phi,phi,I)]   (G = Phi^T Phi)
//
// The reference's analytic gradient (Diff_Loss / The_second_term, CPU Util.cpp:257-304) is
// 3 theta Phi (G o G) - 3 T(phi,phi,I): it equals the exact adjoint when y_A = y_B = y_C and
// mu_A = mu_B = mu_C, and the GPU update direction (stpm.c:649-691) is that expression / 3 with
// theta = 1 in the scaling of init_buff. With A = Y_A Phi, B = Y_B Phi, C = Y_C Phi (b x k):
//   T(I,phi,phi) = Y_A^T K_A / b + mu_A kappa_A^T,  K_A = c3 B o C + c1 (B o m_C + m_B o C),
//                                                   kappa_A = c0 m_B o m_C + c1 mean_x(B o C)
// and likewise for the B and C modes. Everything accumulates in FP64; Y may be FP32 or FP64.
#include <mutex>

#include "common.h"
#include "dense.h"
#include "mfma64.h"

namespace mmsb {

// Column sums of a T x T block from each lane's partials s[v][0..NS) of its columns (bj + 16 v + l % 16):
// the four lanes of a column, then the two waves that share it; out[i * q + c0 + col]. Fixed order.
template <int T, int NS>
__device__ inline void block_colsum(double (&s)[T / 32][NS], double (&red)[2][NS][T], double* __restrict__ out, int32_t q,
                                    int32_t c0) {
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int v = 0; v < T / 32; ++v)
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      s[v][i] += __shfl_xor(s[v][i], 16);
      s[v][i] += __shfl_xor(s[v][i], 32);
      if (l < 16) red[w >> 1][i][(T / 2) * (w & 1) + 16 * v + l] = s[v][i];
    }
  __syncthreads();
  for (int e = threadIdx.x; e < NS * T; e += 256) {
    const int i = e / T, c = e % T;
    if (c0 + c < q) out[(int64_t)i * q + c0 + c] = red[0][i][c] + red[1][i][c];
  }
}

// m_s = Phi^T mu_s of the block's columns from the threads' parts (thread t holds column t % T).
template <int T, int NM>
__device__ inline void block_m(const double (&ms)[NM], double (&part)[NM][256], double (&m)[NM][T]) {
#pragma unroll
  for (int s = 0; s < NM; ++s) part[s][threadIdx.x] = ms[s];
  __syncthreads();
  for (int e = threadIdx.x; e < NM * T; e += 256) {
    const int s = e / T, c = e % T;
    double v = 0.0;
    for (int r = 0; r < 256 / T; ++r) v += part[s][c + T * r];
    m[s][c] = v;
  }
  __syncthreads();
}

// Adjoint, first launch. Workgroups [0, rt * ct): a T x T block of A = Y_A Phi, B = Y_B Phi, C = Y_C Phi (one
// pass over Phi for the three), turned into K_A, K_B, K_C in registers, with the column sums of B o C,
// A o C, A o B and of the loss terms over the block's rows (cpart [rt][4][k]) and m = Phi^T mu (by the first row
// of blocks). The ct * ct workgroups after them: H = (Phi^T Phi)^o2 and the sum of (Phi^T Phi)^o3 per block
// (gpart). Rows from nb and columns from k on stay out of the sums: an infinite entry of Phi makes NaN of their
// zeros. Two workgroups per CU: the 64 x 64 form needs the cap at 256 registers for it (502 -> 395 us per call
// at k = 500). The element-wise pass this replaces ran k threads over all nb rows (1.49 ms of 3.73 at k = 500,
// nb = 4000; 0.35 of 0.83 ms at k = 100, nb = 1024), and the products one vector-ALU launch each.
template <int T, typename TY>
__global__ __launch_bounds__(256, 2) void adj_products_kernel(int32_t nb, int32_t k, int32_t rt, int32_t ct, const TY* __restrict__ ya,
                                                           const TY* __restrict__ yb, const TY* __restrict__ yc, int32_t ldy,
                                                           const double* __restrict__ mua, const double* __restrict__ mub,
                                                           const double* __restrict__ muc, const double* __restrict__ phi,
                                                           double c3, double c1, double* __restrict__ KA,
                                                           double* __restrict__ KB, double* __restrict__ KC,
                                                           double* __restrict__ cpart, double* __restrict__ m,
                                                           double* __restrict__ H, double* __restrict__ gpart) {
  constexpr int U = T / 32;
  __shared__ union {
    NnStage<3, T> nn;
    TnStage<T> tn;
    struct {
      double part[3][256];
      double m[3][T];
      double red[2][4][T];
    } e;
    double red[256];
  } sm;
  const int64_t data = (int64_t)rt * ct;
  if (blockIdx.x >= data) {
    const int g = (int)(blockIdx.x - data), i0 = g / ct * T, j0 = g % ct * T;
    doublex4 acc[U][U] = {};
    tn_tile<T, double, double>(acc, sm.tn, phi, k, k, i0, phi, k, k, j0, 0, k);
    double s = 0.0;
    each_elem<T>([&](int r, int c, int u, int v, int gi) {
      const double x = acc[u][v][gi];
      if (i0 + r < k && j0 + c < k) {
        s = fma(x * x, x, s);
        H[(int64_t)(i0 + r) * k + j0 + c] = x * x;
      }
    });
    __syncthreads();
    sm.red[threadIdx.x] = s;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
      if ((int)threadIdx.x < off) sm.red[threadIdx.x] += sm.red[threadIdx.x + off];
      __syncthreads();
    }
    if (threadIdx.x == 0) gpart[g] = sm.red[0];
    return;
  }
  const int tr = (int)(blockIdx.x / ct), c0 = (int)(blockIdx.x % ct) * T;
  const int64_t x0 = (int64_t)tr * T;
  const TY* const Y[3] = {ya, yb, yc};
  const double* const mu[3] = {mua, mub, muc};
  doublex4 acc[3][U][U] = {};
  double ms[3] = {0.0, 0.0, 0.0};
  nn_tile<3, T, 3, TY>(acc, sm.nn, Y, ldy, x0, nb, phi, k, k, c0, mu, ms);
  __syncthreads();
  block_m<T, 3>(ms, sm.e.part, sm.e.m);
  double s[U][4] = {};
  each_elem<T>([&](int r, int c, int u, int v, int g) {
    const double a = acc[0][u][v][g], b = acc[1][u][v][g], cc = acc[2][u][v][g];
    const double ma = sm.e.m[0][c], mb = sm.e.m[1][c], mc = sm.e.m[2][c];
    if (x0 + r < nb) {
      s[v][0] += b * cc;
      s[v][1] += a * cc;
      s[v][2] += a * b;
      s[v][3] += c3 * a * b * cc + c1 * (a * b * mc + a * mb * cc + ma * b * cc);
      if (c0 + c < k) {
        const int64_t o = (x0 + r) * k + c0 + c;
        KA[o] = c3 * b * cc + c1 * (b * mc + mb * cc);
        KB[o] = c3 * a * cc + c1 * (a * mc + ma * cc);
        KC[o] = c3 * a * b + c1 * (a * mb + ma * b);
      }
    }
  });
  block_colsum<T, 4>(s, sm.e.red, cpart + (int64_t)tr * 4 * k, k, c0);
  if (tr == 0)
    for (int e = threadIdx.x; e < 3 * T; e += 256)
      if (c0 + e % T < k) m[(int64_t)(e / T) * k + c0 + e % T] = sm.e.m[e / T][e % T];
}

// Sums the row blocks' partials of column j (one of ns * k): fixed order, eight loads in flight.
__device__ inline double part_sum(const double* __restrict__ part, int64_t stride, int32_t n, int64_t j) {
  double a[8] = {};
  for (int32_t i = 0; i < n; i += 8)
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (i + u < n) a[u] += part[(int64_t)(i + u) * stride + j];
  return ((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]));
}

// Adjoint, second launch. Workgroups [0, S * ct * ct): block (i, j) of Y_A^T K_A + Y_B^T K_B + Y_C^T K_C over slice
// s of the rows (tpart [S][k * k]); then ct * ct blocks of Phi H; the rest sum the column partials into
// csum [4][k].
template <int T, typename TY>
__global__ __launch_bounds__(256) void adj_contract_kernel(int32_t nb, int32_t k, int32_t ct, int32_t S, int32_t rt,
                                                           const TY* __restrict__ ya, const TY* __restrict__ yb,
                                                           const TY* __restrict__ yc, int32_t ldy,
                                                           const double* __restrict__ KA, const double* __restrict__ KB,
                                                           const double* __restrict__ KC, double* __restrict__ tpart,
                                                           const double* __restrict__ phi, const double* __restrict__ H,
                                                           double* __restrict__ PhiH, const double* __restrict__ cpart,
                                                           double* __restrict__ csum) {
  constexpr int U = T / 32;
  __shared__ union {
    NnStage<1, T> nn;
    TnStage<T> tn;
  } sm;
  const int nt = ct * ct;
  const int blk = (int)blockIdx.x;
  if (blk < (S + 1) * nt) {
    const int tile = blk % nt, i0 = tile / ct * T, j0 = tile % ct * T;
    doublex4 acc[1][U][U] = {};
    double* out;
    if (blk < S * nt) {
      const int s = blk / nt;
      const int64_t r0 = (int64_t)nb * s / S, r1 = (int64_t)nb * (s + 1) / S;
      tn_tile<T, TY, double>(acc[0], sm.tn, ya, ldy, k, i0, KA, k, k, j0, r0, r1);
      tn_tile<T, TY, double>(acc[0], sm.tn, yb, ldy, k, i0, KB, k, k, j0, r0, r1);
      tn_tile<T, TY, double>(acc[0], sm.tn, yc, ldy, k, i0, KC, k, k, j0, r0, r1);
      out = tpart + (int64_t)s * k * k;
    } else {
      const double* const X[1] = {phi};
      nn_tile<1, T, 0, double>(acc, sm.nn, X, k, i0, k, H, k, k, j0, nullptr, nullptr);
      out = PhiH;
    }
    each_elem<T>([&](int r, int c, int u, int v, int g) {
      if (i0 + r < k && j0 + c < k) out[(int64_t)(i0 + r) * k + j0 + c] = acc[0][u][v][g];
    });
    return;
  }
  const int64_t j = (int64_t)(blk - (S + 1) * nt) * 256 + threadIdx.x;
  if (j < 4 * (int64_t)k) csum[j] = part_sum(cpart, 4 * (int64_t)k, rt, j);
}

// Adjoint, third launch: grad = 3 theta PhiH - (sum_s tpart / nb + mu_X kappa_X^T), one element per thread; the last
// workgroup forms loss = theta/2 sum G^3 - sum_j (mean_j + c0 m_A m_B m_C).
__global__ __launch_bounds__(256) void adj_final_kernel(int32_t nb, int32_t k, int32_t S, int32_t ngpart,
                                                        const double* __restrict__ m, const double* __restrict__ mua,
                                                        const double* __restrict__ mub, const double* __restrict__ muc,
                                                        const double* __restrict__ csum, const double* __restrict__ PhiH,
                                                        const double* __restrict__ tpart, const double* __restrict__ gpart,
                                                        double c1, double c0, double theta, double* __restrict__ grad,
                                                        double* __restrict__ loss) {
  const int64_t kk = (int64_t)k * k;
  const double inv = 1.0 / (double)nb;
  if (blockIdx.x + 1 < gridDim.x) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= kk) return;
    const int i = (int)(e / k), j = (int)(e % k);   // row i (component), column j (eigenvector)
    const double ma = m[j], mb = m[k + j], mc = m[2 * k + j];
    const double kA = c0 * mb * mc + c1 * (csum[j] * inv);
    const double kB = c0 * ma * mc + c1 * (csum[k + j] * inv);
    const double kC = c0 * ma * mb + c1 * (csum[2 * k + j] * inv);
    const double t = part_sum(tpart, kk, S, e) * inv + mua[i] * kA + mub[i] * kB + muc[i] * kC;
    grad[e] = 3.0 * theta * PhiH[e] - t;
    return;
  }
  __shared__ double red[256];
  const int t = threadIdx.x;
  double acc = 0.0;
  for (int g = t; g < ngpart; g += 256) acc += 0.5 * theta * gpart[g];
  for (int j = t; j < k; j += 256) acc -= csum[3 * k + j] * inv + c0 * m[j] * m[k + j] * m[2 * k + j];
  red[t] = acc;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if (t < off) red[t] += red[t + off];
    __syncthreads();
  }
  if (t == 0) loss[0] = red[0];
}

// Power method, one chunk of rows: B = Y_B Phi and C = Y_C Phi in T x T blocks (one pass over Phi for both), K_A = c3
// B o C + c1 (B o m_C + m_B o C) and the column sums of B o C over the block's rows (cpart [row block][k]) in the
// epilogue, and m_B, m_C (m [2][k]) by the first row of blocks. As a separate pass with k threads walking the
// chunk's 65536 rows the element-wise part alone took 16 ms per chunk at k = 100 (96 of 116 ms of three
// iterations over 100k nodes).
template <int T>
__global__ __launch_bounds__(256, 2) void pm_products_kernel(int32_t nb, int32_t k, int32_t ct, const float* __restrict__ yb,
                                                             const float* __restrict__ yc, int32_t ldy,
                                                             const double* __restrict__ mub, const double* __restrict__ muc,
                                                             const double* __restrict__ phi, double c3, double c1,
                                                             double* __restrict__ KA, double* __restrict__ cpart,
                                                             double* __restrict__ m) {
  constexpr int U = T / 32;
  __shared__ union {
    NnStage<2, T> nn;
    struct {
      double part[2][256];
      double m[2][T];
      double red[2][1][T];
    } e;
  } sm;
  const int tr = (int)(blockIdx.x / ct), c0 = (int)(blockIdx.x % ct) * T;
  const int64_t x0 = (int64_t)tr * T;
  const float* const Y[2] = {yb, yc};
  const double* const mu[2] = {mub, muc};
  doublex4 acc[2][U][U] = {};
  double ms[2] = {0.0, 0.0};
  nn_tile<2, T, 2, float>(acc, sm.nn, Y, ldy, x0, nb, phi, k, k, c0, mu, ms);
  __syncthreads();
  block_m<T, 2>(ms, sm.e.part, sm.e.m);
  double s[U][1] = {};
  each_elem<T>([&](int r, int c, int u, int v, int g) {
    const double b = acc[0][u][v][g], cc = acc[1][u][v][g];
    s[v][0] += b * cc;
    if (x0 + r < nb && c0 + c < k) KA[(x0 + r) * k + c0 + c] = c3 * b * cc + c1 * (b * sm.e.m[1][c] + sm.e.m[0][c] * cc);
  });
  block_colsum<T, 1>(s, sm.e.red, cpart + (int64_t)tr * k, k, c0);
  if (tr == 0)
    for (int e = threadIdx.x; e < 2 * T; e += 256)
      if (c0 + e % T < k) m[(int64_t)(e / T) * k + c0 + e % T] = sm.e.m[e / T][e % T];
}

// T[:, j] = T[:, j] / n + mu_A kappa_j, kappa = c0 m_B o m_C + c1 colsum / n (colsum from the nt row blocks'
// partials); lam_j = ||T[:, j]||^3, the reference's (sum phi^2)^(3/2) (Util.cpp:164-165); Phi[:, j] = T[:, j] / ||T[:, j]||
// (normc, Util.cpp:166). 16 columns per workgroup, 16 threads per column.
__global__ __launch_bounds__(256) void pm_finish_kernel(int32_t k, double inv_n, const double* __restrict__ T,
                                                        const double* __restrict__ mua, const double* __restrict__ m,
                                                        const double* __restrict__ cpart, int32_t nt, double c1, double c0,
                                                        double* __restrict__ phi, double* __restrict__ lam) {
  __shared__ double red[16][17];
  const int c = threadIdx.x & 15, g = threadIdx.x >> 4;
  const int j = blockIdx.x * 16 + c;
  const bool in = j < k;
  auto colsum16 = [&](double v) {  // over the column's 16 threads, fixed order
    __syncthreads();
    red[g][c] = v;
    __syncthreads();
    double t = 0.0;
    for (int i = 0; i < 16; ++i) t += red[i][c];
    return t;
  };
  double v = 0.0;
  if (in) {
#pragma unroll 8
    for (int t = g; t < nt; t += 16) v += cpart[(int64_t)t * k + j];
  }
  const double colsum = colsum16(v);
  const double kap = in ? c0 * m[j] * m[k + j] + c1 * colsum * inv_n : 0.0;
  double nn = 0.0;
  if (in)
    for (int i = g; i < k; i += 16) {
      const double x = T[(int64_t)i * k + j] * inv_n + mua[i] * kap;
      nn += x * x;
    }
  nn = colsum16(nn);
  if (!in) return;
  const double l = sqrt(nn);
  if (g == 0) lam[j] = l * l * l;
  const double sc = l > 0.0 ? 1.0 / l : 0.0;
  for (int i = g; i < k; i += 16) phi[(int64_t)i * k + j] = (T[(int64_t)i * k + j] * inv_n + mua[i] * kap) * sc;
}

// P = U V^T over the singular triplets (column-major U, V of the one-sided Jacobi SVD, whose U is zero in the
// columns with sigma = 0; out column-major), as blocks of sum_l V[l][j] U[l][i] over the buffers' rows l: 38 -> 5 us
// at k = 100 against one thread per element. Applied to the SVD of Phi^T (the row-major Phi buffer read
// column-major), out read row-major is the polar factor of Phi, the orthonormal matrix nearest to it.
__global__ __launch_bounds__(256) void polar_kernel(int32_t k, int32_t ct, const double* __restrict__ U,
                                                    const double* __restrict__ V, double* __restrict__ out) {
  __shared__ TnStage<32> sm;
  const int i0 = (int)blockIdx.x / ct * 32, j0 = (int)blockIdx.x % ct * 32;
  doublex4 acc[1][1] = {};
  tn_tile<32, double, double>(acc, sm, V, k, k, i0, U, k, k, j0, 0, k);
  each_elem<32>([&](int r, int c, int u, int v, int g) {
    if (i0 + r < k && j0 + c < k) out[(int64_t)(i0 + r) * k + j0 + c] = acc[u][v][g];
  });
}

static size_t align256(size_t b) { return (b + 255) / 256 * 256; }

// Row blocks of the products over n rows taken in chunks (the column partials of all chunks are kept).
static int power_tile(int32_t k, int64_t rows) { return ceil_div(rows, 64) * ceil_div(k, 64) >= 192 ? 64 : 32; }

static int64_t power_blocks(int64_t n, int32_t chunk) { return ceil_div(n, chunk) * ceil_div(chunk, 32); }

size_t power_workspace_bytes(int32_t k, int64_t n, int32_t chunk) {
  const size_t ck = sizeof(double) * (size_t)chunk * k, kk = sizeof(double) * (size_t)k * k;
  const size_t tn = tn_workspace_bytes(chunk, k, k);
  return align256(ck) + 4 * align256(kk) + 2 * align256(sizeof(double) * 4 * k) +
         align256(sizeof(double) * (size_t)power_blocks(n, chunk) * k) + align256(tn) +
         align256(jacobi_workspace_bytes(k)) + align256(64);
}

// One iteration of the batch implicit power method with the A mode free (CPU tensorDecom_alpha0,
// Util.cpp:131-206): Phi_j <- T(I, phi_j, phi_j) over all n rows, lambda_j = ||.||^3, columns
// normalised, then (optionally) the orthonormalisation Phi <- U V^T from the one-sided Jacobi SVD of
// Phi itself (the polar factor Phi (Phi^T Phi)^-1/2, without forming Phi^T Phi, whose condition
// number is cond(Phi)^2).
// Y_A, Y_B, Y_C row-major [nb x ldy] per chunk.
int power_iteration(hipStream_t s, int32_t k, int64_t n, const PowerRows& rows, int32_t ldy, const double* mua,
                    const double* mub, const double* muc, double c3, double c1, double c0, double* phi, double* lam,
                    int orthogonalize, int32_t chunk, void* work) {
  unsigned char* w = static_cast<unsigned char*>(work);
  auto take = [&](size_t bytes) { void* p = w; w += align256(bytes); return p; };
  const size_t kk = sizeof(double) * (size_t)k * k;
  double* KA = (double*)take(sizeof(double) * (size_t)chunk * k);
  double *T = (double*)take(kk), *G = (double*)take(kk), *Vj = (double*)take(kk), *Uj = (double*)take(kk);
  double *m = (double*)take(sizeof(double) * 4 * k), *sig = (double*)take(sizeof(double) * 4 * k);
  double* cpart = (double*)take(sizeof(double) * (size_t)power_blocks(n, chunk) * k);
  double* tn = (double*)take(tn_workspace_bytes(chunk, k, k));
  void* jw = take(jacobi_workspace_bytes(k));
  int32_t* sweeps = (int32_t*)take(64);
  int64_t nt = 0;  // row blocks so far
  for (int64_t r0 = 0; r0 < n; r0 += chunk) {
    const int32_t nb = (int32_t)std::min<int64_t>(chunk, n - r0);
    const float *ya = nullptr, *yb = nullptr, *yc = nullptr;
    MMSB_TRY(rows(r0, nb, &ya, &yb, &yc));
    const int t = power_tile(k, nb), ct = (int)ceil_div(k, t), rt = (int)ceil_div(nb, t);
    const dim3 g((unsigned)((int64_t)rt * ct));
    if (t == 64)
      hipLaunchKernelGGL(pm_products_kernel<64>, g, dim3(256), 0, s, nb, k, ct, yb, yc, ldy, mub, muc, phi, c3, c1, KA,
                         cpart + nt * k, m);
    else
      hipLaunchKernelGGL(pm_products_kernel<32>, g, dim3(256), 0, s, nb, k, ct, yb, yc, ldy, mub, muc, phi, c3, c1, KA,
                         cpart + nt * k, m);
    MMSB_LAUNCH_CHECK();
    nt += rt;
    MMSB_TRY((gemm_tn<float, double>(s, nb, k, k, 1.0, ya, ldy, KA, k, r0 == 0 ? 0.0 : 1.0, T, tn)));
  }
  hipLaunchKernelGGL(pm_finish_kernel, dim3((unsigned)ceil_div(k, 16)), dim3(256), 0, s, k, 1.0 / (double)n, T, mua, m, cpart,
                     (int32_t)nt, c1, c0, phi, lam);
  MMSB_LAUNCH_CHECK();
  if (orthogonalize) {  // Phi <- U V^T of Phi's own SVD (G holds a copy: the Jacobi SVD overwrites its input)
    hipError_t e = hipMemcpyAsync(G, phi, kk, hipMemcpyDeviceToDevice, s);
    if (e != hipSuccess) return set_error(MMSB_ERR_HIP, "power: %s", hipGetErrorString(e));
    MMSB_TRY(jacobi_svd(s, k, G, Uj, sig, Vj, jw, sweeps));
    const int ct = (int)ceil_div(k, 32);
    hipLaunchKernelGGL(polar_kernel, dim3((unsigned)(ct * ct)), dim3(256), 0, s, k, ct, Uj, Vj, phi);
    MMSB_LAUNCH_CHECK();
  }
  return MMSB_OK;
}

// The published workspace size (mmsb_stgd_grad_workspace): callers hold buffers of this size and the fixed
// scratch of the allocation-free form bounds (k, nb) by it, so it is a formula of its own: 6 b x k and
// 4 k x k matrices, 12 k-vectors, and the row-slice partials of a k x k product.
static int64_t grad_slices(int64_t n, int32_t k) {  // slices of a b-row product in that formula
  const int64_t t64 = ceil_div(k, 64) * ceil_div(k, 64);
  const int64_t s = std::min<int64_t>(ceil_div(2048, t64), std::max<int64_t>(1, n / 256));
  int64_t most = std::max<int64_t>(1, std::min<int64_t>(s, 512));
  if (k == 1 && n >= 65536) most = std::max(most, std::min<int64_t>(1024, n / 256));
  if (n >= 4096 && k >= 32) {
    const int64_t tp = ceil_div(k, 128), cap = std::max<int64_t>(1, (256ll << 20) / ((int64_t)k * k * 8));
    for (int64_t tiles : {tp * tp, tp * (tp + 1) / 2})
      most = std::max(most, std::max<int64_t>(1, std::min(std::min(std::max<int64_t>(1, 1024 / tiles), cap),
                                                          std::max<int64_t>(1, n / 1024))));
  }
  return most;
}

size_t grad_workspace_bytes(int32_t k, int32_t nb) {
  const size_t bk = sizeof(double) * (size_t)nb * k, kk = sizeof(double) * (size_t)k * k;
  size_t tn = (size_t)std::max(grad_slices(nb, k), grad_slices(k, k)) * kk;
  return 6 * align256(bk) + 4 * align256(kk) + 3 * align256(sizeof(double) * 4 * k) + align256(tn);
}

// Launch shape of the adjoint, a function of (k, nb) alone so that every entry point sums in the same order.
// 64 x 64 blocks read each operand half as often as 32 x 32 ones but leave CUs idle on small problems: they are
// taken for the products once they make 192 workgroups, and for the contraction above k = 256 (below it the
// k x k output has at most 16 of them): k = 500, nb = 4000 takes 387 us with 64 x 64 products, 431 with 32 x 32.
// The contraction's rows are cut into S slices of about 64 rows or more (nb = 65: 32 and 33), about 512 workgroups in all. A whole call
// (three launches instead of 22): k = 100, nb = 1024 in FP32 828 -> 49 us, of which 28 in kernels; k = 500,
// nb = 4000 in FP64 3.73 -> 0.39 ms, 32 TFLOP/s of FP64 MFMA.
struct AdjShape {
  int t1, rt, ct1, t2, ct2, S;
};

static AdjShape adj_shape(int32_t k, int32_t nb) {
  AdjShape a;
  a.t1 = ceil_div(nb, 64) * ceil_div(k, 64) >= 192 ? 64 : 32;
  a.rt = (int)ceil_div(nb, a.t1);
  a.ct1 = (int)ceil_div(k, a.t1);
  a.t2 = k > 256 ? 64 : 32;
  a.ct2 = (int)ceil_div(k, a.t2);
  // the partials lie in what the published size leaves: three b x k matrices less the column partials (at most
  // b k / 8 + 4 k values), and one k x k matrix
  const int64_t room = 1 + (3 * (int64_t)nb * k - (int64_t)a.rt * 4 * k) / ((int64_t)k * k);
  a.S = (int)std::max<int64_t>(1, std::min(std::min<int64_t>(ceil_div(512, a.ct2 * a.ct2), ceil_div(nb, 64)), room));
  return a;
}

template <typename TY>
int stgd_grad(hipStream_t s, int32_t k, int32_t nb, const TY* ya, const TY* yb, const TY* yc, int32_t ldy,
              const double* mua, const double* mub, const double* muc, const double* phi, double c3, double c1, double c0,
              double theta, double* grad, double* loss, void* work) {
  MMSB_CHECK_ARG(k >= 1 && nb >= 1 && ldy >= k, "grad: bad shape k=%d nb=%d ldy=%d", k, nb, ldy);
  MMSB_CHECK_ARG(ya && yb && yc && mua && mub && muc && phi && grad && loss && work, "grad: null pointer");
  const AdjShape a = adj_shape(k, nb);
  unsigned char* w = static_cast<unsigned char*>(work);
  auto take = [&](int64_t n) { double* p = reinterpret_cast<double*>(w); w += align256(sizeof(double) * (size_t)n); return p; };
  const int64_t bk = (int64_t)nb * k, kk = (int64_t)k * k;
  double *KA = take(bk), *KB = take(bk), *KC = take(bk);
  double *H = take(kk), *PhiH = take(kk);
  double *m = take(3 * (int64_t)k), *csum = take(4 * (int64_t)k), *gpart = take((int64_t)a.ct1 * a.ct1);
  double *cpart = take((int64_t)a.rt * 4 * k), *tpart = take(a.S * kk);
  MMSB_CHECK_ARG((size_t)(w - static_cast<unsigned char*>(work)) <= grad_workspace_bytes(k, nb), "grad: workspace layout");
  const dim3 g1((unsigned)((int64_t)a.rt * a.ct1 + (int64_t)a.ct1 * a.ct1));
  if (a.t1 == 64)
    hipLaunchKernelGGL((adj_products_kernel<64, TY>), g1, dim3(256), 0, s, nb, k, a.rt, a.ct1, ya, yb, yc, ldy, mua, mub, muc, phi,
                       c3, c1, KA, KB, KC, cpart, m, H, gpart);
  else
    hipLaunchKernelGGL((adj_products_kernel<32, TY>), g1, dim3(256), 0, s, nb, k, a.rt, a.ct1, ya, yb, yc, ldy, mua, mub, muc, phi,
                       c3, c1, KA, KB, KC, cpart, m, H, gpart);
  MMSB_LAUNCH_CHECK();
  const dim3 g2((unsigned)((int64_t)(a.S + 1) * a.ct2 * a.ct2 + ceil_div(4 * (int64_t)k, 256)));
  if (a.t2 == 64)
    hipLaunchKernelGGL((adj_contract_kernel<64, TY>), g2, dim3(256), 0, s, nb, k, a.ct2, a.S, a.rt, ya, yb, yc, ldy, KA, KB, KC,
                       tpart, phi, H, PhiH, cpart, csum);
  else
    hipLaunchKernelGGL((adj_contract_kernel<32, TY>), g2, dim3(256), 0, s, nb, k, a.ct2, a.S, a.rt, ya, yb, yc, ldy, KA, KB, KC,
                       tpart, phi, H, PhiH, cpart, csum);
  MMSB_LAUNCH_CHECK();
  hipLaunchKernelGGL(adj_final_kernel, dim3((unsigned)(ceil_div(kk, 256) + 1)), dim3(256), 0, s, nb, k, a.S, a.ct1 * a.ct1, m, mua,
                     mub, muc, csum, PhiH, tpart, gpart, c1, c0, theta, grad, loss);
  MMSB_LAUNCH_CHECK();
  return MMSB_OK;
}

template int stgd_grad<float>(hipStream_t, int32_t, int32_t, const float*, const float*, const float*, int32_t, const double*,
                              const double*, const double*, const double*, double, double, double, double, double*, double*,
                              void*);
template int stgd_grad<double>(hipStream_t, int32_t, int32_t, const double*, const double*, const double*, int32_t,
                               const double*, const double*, const double*, const double*, double, double, double, double,
                               double*, double*, void*);

}  // namespace mmsb

extern "C" size_t mmsb_stgd_grad_workspace(int32_t k, int32_t nb) {
  if (k < 1 || nb < 1) return 0;
  return mmsb::grad_workspace_bytes(k, nb);
}

extern "C" int mmsb_tensor_coeffs(double alpha0, int32_t scaling, double* out3) {
  mmsb::clear_error();
  MMSB_CHECK_ARG(out3 && alpha0 > 0.0, "tensor_coeffs: bad arguments");
  if (scaling == MMSB_M2_GPU) {  // init_buff, stpm.c:1026-1038
    out3[0] = 1.0;
    out3[1] = -alpha0 / (alpha0 + 2.0);
    out3[2] = 2.0 * alpha0 * alpha0 / ((alpha0 + 1.0) * (alpha0 + 2.0));
  } else {  // The_second_term, CPU Util.cpp:289-298
    out3[0] = (alpha0 + 1.0) * (alpha0 + 2.0) / 2.0;
    out3[1] = -alpha0 * (alpha0 + 1.0) / 2.0;
    out3[2] = alpha0 * alpha0;
  }
  return MMSB_OK;
}

extern "C" int mmsb_stgd_grad_f64(void* stream, int32_t k, int32_t nb, const double* ya, const double* yb, const double* yc,
                                  int32_t ldy, const double* mu_a, const double* mu_b, const double* mu_c, const double* phi,
                                  const double* coeffs, double theta, double* grad, double* loss, void* work) {
  mmsb::clear_error();
  MMSB_CHECK_ARG(coeffs, "grad: null coefficients");
  return mmsb::stgd_grad<double>(static_cast<hipStream_t>(stream), k, nb, ya, yb, yc, ldy, mu_a, mu_b, mu_c, phi, coeffs[0],
                                 coeffs[1], coeffs[2], theta, grad, loss, work);
}

namespace mmsb {
// Scratch of the allocation-free adjoint entry point (mmsb_stgd_grad_f32_noalloc): a device array of
// fixed size, one copy per GPU, held until the process ends. Host code never passes the array's name
// to a kernel (on the host it is only a stand-in): the device address of each GPU's copy comes from
// hipGetSymbolAddress, called once per device with that device current, and is kept per device.
static constexpr size_t kGradScratchBytes = (size_t)32 << 20;
static __device__ __align__(256) unsigned char scratch[kGradScratchBytes];
static constexpr int kMaxScratchDevices = 64;
static std::mutex g_scratch_mu;
static void* g_scratch_dev[kMaxScratchDevices] = {};

static int grad_scratch(void** out) {
  int dev = 0;
  MMSB_HIP(hipGetDevice(&dev));
  MMSB_CHECK_ARG(dev >= 0 && dev < kMaxScratchDevices, "grad_noalloc: device %d beyond the supported %d", dev,
                 kMaxScratchDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_dev[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return set_error(MMSB_ERR_HIP, "grad_noalloc: hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
    g_scratch_dev[dev] = p;
  }
  *out = g_scratch_dev[dev];
  return MMSB_OK;
}
}  // namespace mmsb

extern "C" int mmsb_stgd_grad_f32_noalloc(void* stream, int32_t k, int32_t nb, const float* ya, const float* yb,
                                          const float* yc, int32_t ldy, const double* mu_a, const double* mu_b,
                                          const double* mu_c, const double* phi, const double* coeffs, double theta,
                                          double* grad, double* loss) {
  mmsb::clear_error();
  MMSB_CHECK_ARG(coeffs, "grad: null coefficients");
  MMSB_CHECK_ARG(k >= 1 && nb >= 1, "grad_noalloc: bad shape k=%d nb=%d", k, nb);
  const size_t need = mmsb::grad_workspace_bytes(k, nb);
  MMSB_CHECK_ARG(need <= mmsb::kGradScratchBytes,
                 "grad_noalloc: k=%d, nb=%d needs %zu bytes of scratch, above the fixed %zu (use mmsb_stgd_grad_f32 with a "
                 "workspace)", k, nb, need, mmsb::kGradScratchBytes);
  void* work = nullptr;
  MMSB_TRY(mmsb::grad_scratch(&work));
  // every region of the workspace is written before it is read (no clearing needed)
  return mmsb::stgd_grad<float>(static_cast<hipStream_t>(stream), k, nb, ya, yb, yc, ldy, mu_a, mu_b, mu_c, phi, coeffs[0],
                                coeffs[1], coeffs[2], theta, grad, loss, work);
}

extern "C" int mmsb_stgd_grad_f32(void* stream, int32_t k, int32_t nb, const float* ya, const float* yb, const float* yc,
                                  int32_t ldy, const double* mu_a, const double* mu_b, const double* mu_c, const double* phi,
                                  const double* coeffs, double theta, double* grad, double* loss, void* work) {
  mmsb::clear_error();
  MMSB_CHECK_ARG(coeffs, "grad: null coefficients");
  return mmsb::stgd_grad<float>(static_cast<hipStream_t>(stream), k, nb, ya, yb, yc, ldy, mu_a, mu_b, mu_c, phi, coeffs[0],
                                coeffs[1], coeffs[2], theta, grad, loss, work);
}
