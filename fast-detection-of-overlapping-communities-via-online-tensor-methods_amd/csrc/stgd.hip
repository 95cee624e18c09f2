// STGD step kernels, FP32 and BF16 MFMA (the hot loop of GPU_Task, stpm.c:497-790).
//
// One step over a minibatch X_b of nb nodes (layouts in stgd.h):
//   P1  P_A = Y_A[X_b] Phi, P_B = Y_B[X_b] Phi, with m_A = Phi^T mu_A, m_B = Phi^T mu_B:
//       C_g = c3 P_A o P_B + c1 (P_A o m_B + m_A o P_B) (rows beyond nb zero);
//       per-tile column sums of P_A o P_B;  and  H = (Phi^T Phi) o (Phi^T Phi)
//   P2  Phi~ = Phi - eta theta Phi H + eta [Y_C[X_b]^T C_g / nb + mu_C c_mu^T],
//       c_mu = c0 m_A o m_B + c1 sum_x(P_A o P_B) / nb                       (stpm.c:532-691)
//   NS  G = X^T X; X <- c X (3I - c^2 G) / 2 (degree 3), or Q = -(5/4) c^2 G + (3/8) c^4 G^2 and
//       X <- c X (15/8 I + Q) (degree 5), with c = min(1, sqrt(2 / ||G||_inf)), ns_iters times
//       (polar renormalisation in place of the QR of stpm.c:774-786). The polar factor is
//       scale-invariant; c only acts when sigma_max(X)^2 may exceed 2, where the unscaled
//       iterations (convergent for sigma < sqrt 3, resp. sqrt(7/3)) would diverge -- e.g. after a
//       minibatch that holds very high-degree nodes.
// (c3, c1, c0) are the entries of the 4x4 matrices of init_buff (stpm.c:1026-1038).
//
// Work decomposition: every GEMM output is cut into 32 x 32 blocks, one per workgroup of four
// waves. The waves split the reduction dimension (each wave owns its K range) and load their
// operand blocks with whole-cache-line loads, rearranged into the MFMA layout through a small
// per-wave LDS buffer (the staging section below), through a ring of D fragment sets, so that up to
// D groups of loads are in flight ahead of the MFMAs (in P1's data tiles each wave computes both
// Y_A Phi and Y_B Phi over its K range, loading each Phi^T block once for the two). The partial
// accumulators meet in padded LDS tiles that all 256 threads read back for coalesced epilogue
// stores. At k = 500 a phase launches 256-768 workgroups.
// K order inside a fragment: for v_mfma_f32_32x32x2f32 lane half h holds k = 4h + i of a chunk
// of eight k for instruction i (the order of a sum over k is free as long as A and B agree);
// for v_mfma_f32_32x32x16_bf16 lane half h holds the eight contiguous k = 8h .. 8h + 7.
// Precision: FP32 mode multiplies FP32 on v_mfma_f32_32x32x2f32. BF16 mode multiplies the data
// contractions (Y Phi, Y_C^T C_g) as BF16 on v_mfma_f32_32x32x16_bf16 and the k x k x k products
// as split BF16 (x = hi + lo; hi.hi + hi.lo + lo.hi, about 16 significant bits); all accumulate
// in FP32. In BF16 mode every k x k operand is written by the kernel that produces it both in
// FP32 and as its (hi, lo) BF16 pair, so the MFMA loops load ready operands and convert nothing.
// m_A and m_B of the next step are reduced from the tiles of the new Phi where it is written.
// Y_A, Y_B, Y_C^T either hold all of X (row offset row0) or, for checkpointed runs, only the minibatches of
// the next steps, refilled from CSR by a caller-supplied launch (StgdArgs::y_window).
#include <hip/hip_cooperative_groups.h>

#include <algorithm>
#include <cstring>
#include <type_traits>
#include <vector>

#include "common.h"
#include "devmem.h"
#include "stgd.h"
#include "wave.h"

namespace cg = cooperative_groups;

namespace mmsb {

enum { MM_F32 = 0, MM_BF16 = 1, MM_BF16X3 = 2 };

template <int MODE>
using op_t = typename std::conditional<MODE == MM_F32, float, __bf16>::type;

// A matrix operand of wave_mm: rows of length >= K with leading dimension ld; lo is the low BF16
// half of a split operand (split mode only; equal to hi otherwise).
template <typename T>
struct Opnd {
  const T* hi;
  const T* lo;
  int64_t ld;
};

template <typename T>
__host__ __device__ inline Opnd<T> opnd(const T* hi, const T* lo, int64_t ld) {
  return Opnd<T>{hi, lo ? lo : hi, ld};
}

// Waves per workgroup. Every tile's reduction is split over all of them (kWaves parts of the k or
// minibatch range), which keeps kWaves waves of loads in flight per tile -- with one tile per compute
// unit at k ~ 500, the only source of memory-level parallelism. The epilogues run on the first four
// waves (threads 0..255), which own one element group of four each.
#ifndef MMSB_STGD_WAVES
#define MMSB_STGD_WAVES 4
#endif
constexpr int kWaves = MMSB_STGD_WAVES;
constexpr int kThreads = 64 * kWaves;
static_assert(kWaves == 4 || kWaves == 8, "4 or 8 waves per workgroup");

// ---- operand staging ---------------------------------------------------------------------------
// One reduction group of a wave's MFMA operand is a block of 32 rows x 128 bytes (32 FP32 or 64 BF16
// values per row). Read in the MFMA layout -- lane (r, h) taking row r -- every load instruction
// would touch 32 cache lines and use 32 bytes of each, and with a dozen waves per compute unit
// streaming such blocks the L1 refetches each line for each of its four 32-byte pieces. Instead
// every load instruction reads 8 whole 128-byte row segments (lane 8q + s takes 16-byte segment s of
// row q, plus 8 rows per instruction), and a transpose through the wave's own 4 KiB LDS buffer then
// leaves register c of lane (r, h) with segment 2c + h of row r: k = 8c + 4h .. +3 (FP32) or
// 16c + 8h .. +7 (BF16) of the group, the k order the MFMA sequences below assume for A and B alike
// (the order of a sum over k is free as long as both operands agree). Segment s of row q sits at
// slot s ^ ((q >> 1) & 7) of the buffer row, which keeps both the writes (8 rows x 8 slots per
// instruction) and the reads (32 rows x one segment per lane half) on distinct banks in every group
// of 16 lanes. LDS instructions of one wave execute in order, so the reads see the writes and the next
// block's writes land after the reads; the waves of a workgroup use separate buffers and never wait
// on each other here.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <bool AL, typename T>
__device__ inline u32x4 ld16(const T* p) {
  if constexpr (AL) return *reinterpret_cast<const u32x4*>(p);
  constexpr int E = 16 / sizeof(T);  // rows not 16-byte aligned: element by element
  T e[E];
#pragma unroll
  for (int i = 0; i < E; ++i) e[i] = p[i];
  return __builtin_bit_cast(u32x4, e);
}

// The four coalesced loads of one block; row0 (the block's first row and first k) and ld are
// wave-uniform. Each address is that uniform base plus 8c rows plus one 32-bit per-lane byte offset,
// the form the compiler issues with a scalar base register: one offset VGPR per operand instead of a
// 64-bit address pair per load.
template <bool AL, typename T>
__device__ inline void stage_load(u32x4 v[4], const T* row0, int64_t ld) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t off = ((lane >> 3) * (uint32_t)ld + (lane & 7) * (16 / (uint32_t)sizeof(T))) * (uint32_t)sizeof(T);
  const char* base = reinterpret_cast<const char*>(row0);
#pragma unroll
  for (int c = 0; c < 4; ++c) v[c] = ld16<AL>(reinterpret_cast<const T*>(base + 8 * c * ld * (int64_t)sizeof(T) + off));
}

// The calling wave's index within its workgroup, as a wave-uniform (scalar) value.
__device__ inline int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

__device__ inline u32x4* wave_stage() {
  __shared__ u32x4 buf[kWaves][256];
  return buf[wave_id()];
}

// Rearranges a block loaded by stage_load into the MFMA layout, in place, through the wave's buffer.
__device__ inline void stage_swap(u32x4 v[4], u32x4* buf) {
  const int lane = threadIdx.x & 63;
  const int q = lane >> 3, s = lane & 7, r = lane & 31, h = lane >> 5;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int row = q + 8 * c;
    buf[row * 8 + (s ^ ((row >> 1) & 7))] = v[c];
  }
  asm volatile("" ::: "memory");  // compiler ordering only: the reads follow the writes
#pragma unroll
  for (int c = 0; c < 4; ++c) v[c] = buf[r * 8 + ((2 * c + h) ^ ((r >> 1) & 7))];
  asm volatile("" ::: "memory");  // ... and the next block's writes follow these reads
}

__device__ inline void stage_swap(u32x4 v[4]) { stage_swap(v, wave_stage()); }

__device__ inline floatx4 as_f32(const u32x4& v) { return __builtin_bit_cast(floatx4, v); }
__device__ inline bf16x8 as_bf16(const u32x4& v) { return __builtin_bit_cast(bf16x8, v); }

// Reduction group of one fragment set: 32 k for FP32, 64 k for the BF16 modes (128 bytes per row).
template <int MODE>
constexpr int kgroup() { return MODE == MM_F32 ? 32 : 64; }

// Fragment set of one reduction group for one wave: load() issues the coalesced loads of its blocks
// (A rows from pa, B rows from pb, both at the group's first k), swap() puts them in the MFMA layout
// once they are needed, mma() accumulates.
template <int MODE>
struct Frag;

template <>
struct Frag<MM_F32> {
  u32x4 a[4], b[4];
  template <bool AAL>
  __device__ inline void load(const float* pa, const float*, int64_t lda, const float* pb, const float*, int64_t ldb) {
    stage_load<AAL>(a, pa, lda);
    stage_load<true>(b, pb, ldb);
  }
  __device__ inline void swap() {
    stage_swap(a);
    stage_swap(b);
  }
  __device__ inline void mma(floatx16& acc) const {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const floatx4 x = as_f32(a[c]), y = as_f32(b[c]);
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[0], y[0], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[1], y[1], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[2], y[2], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[3], y[3], acc, 0, 0, 0);
    }
  }
};

template <>
struct Frag<MM_BF16> {
  u32x4 a[4], b[4];
  template <bool AAL>
  __device__ inline void load(const __bf16* pa, const __bf16*, int64_t lda, const __bf16* pb, const __bf16*,
                              int64_t ldb) {
    stage_load<AAL>(a, pa, lda);
    stage_load<true>(b, pb, ldb);
  }
  __device__ inline void swap() {
    stage_swap(a);
    stage_swap(b);
  }
  __device__ inline void mma(floatx16& acc) const {
#pragma unroll
    for (int c = 0; c < 4; ++c) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16(a[c]), as_bf16(b[c]), acc, 0, 0, 0);
  }
};

template <>
struct Frag<MM_BF16X3> {
  u32x4 ah[4], al[4], bh[4], bl[4];
  template <bool AAL>
  __device__ inline void load(const __bf16* pa, const __bf16* pal, int64_t lda, const __bf16* pb, const __bf16* pbl,
                              int64_t ldb) {
    stage_load<AAL>(ah, pa, lda);
    stage_load<AAL>(al, pal, lda);
    stage_load<true>(bh, pb, ldb);
    stage_load<true>(bl, pbl, ldb);
  }
  __device__ inline void swap() {
    stage_swap(ah);
    stage_swap(al);
    stage_swap(bh);
    stage_swap(bl);
  }
  __device__ inline void mma(floatx16& acc) const {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const bf16x8 xh = as_bf16(ah[c]), xl = as_bf16(al[c]), yh = as_bf16(bh[c]), yl = as_bf16(bl[c]);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xh, yh, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xh, yl, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xl, yh, acc, 0, 0, 0);
    }
  }
};

// use(f[..]) of the groups at k = 0, G, .. (< kl) in order, each after load(f[..], k), with the loads ahead of the uses: with
// D = 4 sets and a multiple of four groups the next three groups are in flight, else the next one. No load is under a condition of
// its own: where paths with and without a load meet, the compiler waits for all loads in flight (it counts the newest
// ones it is sure of), and a ring of guarded loads then costs one memory latency per group, 0.5 us (P2 of an FP32 step
// at k = 100, b = 1024: 14.5 us with guards, 10.9 without; BF16 at k = 500: 6.1 and 5.5, Newton-Schulz 22 and 20.5). COMPACT keeps the
// guards for fewer registers (the body twice instead of five times): for reductions of one or two groups, where all
// loads go out first anyway.
template <int G, bool COMPACT = false, int D, typename F, typename L, typename M>
__device__ __forceinline__ void pipelined(F (&f)[D], int64_t kl, L load, M mma) {
  static_assert(D == 2 || D == 4, "two or four sets");
  if (kl <= 0) return;
  auto use = [&](F& x) {
    x.swap();
    mma(x);
  };
  if constexpr (COMPACT) {
    load(f[0], (int64_t)0);
    for (int64_t k = 0; k < kl; k += 2 * G) {
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        const int64_t kk = k + d * G;
        if (kk < kl) {
          const int64_t kn = kk + G;
          if (kn < kl) load(f[1 - d], kn);
          use(f[d]);
        }
      }
    }
    return;
  }
  const int n = (int)(kl / G);  // 32-bit offsets: fewer registers
  if constexpr (D == 4) {
    if (n % 4 == 0) {
#pragma unroll
      for (int d = 0; d < 4; ++d) load(f[d], d * G);
      f[0].swap();  // each group goes through LDS under the MFMAs of the one before
      for (int g = 4; g < n; g += 4) {
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          f[(d + 1) % 4].swap();
          mma(f[d]);
          load(f[d], (g + d) * G);
        }
      }
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        if (d < 3) f[d + 1].swap();
        mma(f[d]);
      }
      return;
    }
  }
  load(f[0], 0);
  int g = 0;
  for (; g + 2 < n; g += 2) {
    load(f[1], (g + 1) * G);
    use(f[0]);
    load(f[0], (g + 2) * G);
    use(f[1]);
  }
  if (g + 1 < n) {
    load(f[1], (g + 1) * G);
    use(f[0]);
    use(f[1]);
  } else {
    use(f[0]);
  }
}

// The part of a reduction of length K (a multiple of the group) that wave `idx` of `parts` owns.
template <int MODE>
__device__ inline void kslice(int64_t K, int parts, int idx, int64_t& k0, int64_t& kl) {
  constexpr int G = kgroup<MODE>();
  const int64_t ng = K / G;
  const int64_t g0 = ng * idx / parts, g1 = ng * (idx + 1) / parts;
  k0 = g0 * G;
  kl = (g1 - g0) * G;
}

// acc += A[r0 + 0..32, k0 .. k0+kl) * B[c0 + 0..32, k0 .. k0+kl)^T for the calling wave.
// kl is a multiple of kgroup<MODE>(); AAL says whether A's rows are 16-byte aligned at k0; D fragment sets (32 VGPRs
// each for FP32 and BF16, 64 for split BF16).
template <int MODE, bool AAL, int D = 2, bool COMPACT = false, typename TA, typename TB>
__device__ inline void wave_mm(floatx16& acc, const Opnd<TA>& A, const Opnd<TB>& B, int64_t r0, int64_t c0, int64_t k0,
                               int64_t kl) {
  constexpr int G = kgroup<MODE>();
  const TA* a = A.hi + r0 * A.ld + k0;
  const TA* al = A.lo + r0 * A.ld + k0;
  const TB* b = B.hi + c0 * B.ld + k0;
  const TB* bl = B.lo + c0 * B.ld + k0;
  Frag<MODE> f[D];
  pipelined<G, COMPACT>(
      f, kl, [&](Frag<MODE>& x, auto k) { x.template load<AAL>(a + k, al + k, A.ld, b + k, bl + k, B.ld); },
      [&](Frag<MODE>& x) { x.mma(acc); });
}

// Two products that share their column operand, acc_a += A1 B^T and acc_b += A2 B^T, for one wave
// over k in [k0, k0 + kl) (FP32 or BF16 modes): the fragment set holds A1, A2 and B, so B is loaded
// once for both.
template <int MODE>
struct FragPair {
  using T = op_t<MODE>;
  u32x4 a1[4], a2[4], b[4];
  __device__ inline void load(const T* p1, const T* p2, int64_t lda, const T* pb, int64_t ldb) {
    stage_load<true>(a1, p1, lda);
    stage_load<true>(a2, p2, lda);
    stage_load<true>(b, pb, ldb);
  }
  __device__ inline void swap() {
    stage_swap(a1);
    stage_swap(a2);
    stage_swap(b);
  }
  __device__ inline void mma(floatx16& acc_a, floatx16& acc_b) const {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if constexpr (MODE == MM_F32) {
        const floatx4 x1 = as_f32(a1[c]), x2 = as_f32(a2[c]), y = as_f32(b[c]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          acc_a = __builtin_amdgcn_mfma_f32_32x32x2f32(x1[e], y[e], acc_a, 0, 0, 0);
          acc_b = __builtin_amdgcn_mfma_f32_32x32x2f32(x2[e], y[e], acc_b, 0, 0, 0);
        }
      } else {
        acc_a = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16(a1[c]), as_bf16(b[c]), acc_a, 0, 0, 0);
        acc_b = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16(a2[c]), as_bf16(b[c]), acc_b, 0, 0, 0);
      }
    }
  }
};

template <int MODE, bool COMPACT = false>
__device__ inline void wave_mm_pair(floatx16& acc_a, floatx16& acc_b, const op_t<MODE>* A1, const op_t<MODE>* A2, int64_t lda,
                                    const op_t<MODE>* B, int64_t ldb, int64_t r0, int64_t c0, int64_t k0, int64_t kl) {
  constexpr int G = kgroup<MODE>();
  const op_t<MODE>* p1 = A1 + r0 * lda + k0;
  const op_t<MODE>* p2 = A2 + r0 * lda + k0;
  const op_t<MODE>* b = B + c0 * ldb + k0;
  FragPair<MODE> f[2];
  pipelined<G, COMPACT>(
      f, kl, [&](FragPair<MODE>& x, auto k) { x.load(p1 + k, p2 + k, lda, b + k, ldb); },
      [&](FragPair<MODE>& x) { x.mma(acc_a, acc_b); });
}

__device__ inline bool epi_thread() { return threadIdx.x < 256; }

// Four 32 x 32 partial accumulators. Register i of lane l holds element
// (8 (i / 4) + 4 (l / 32) + i % 4, l % 32) of the block; rows of 66 words keep the column-wise
// read-back of the epilogues to two-way bank conflicts.
struct Red4 {
  float v[4][16][66];
};

__device__ inline void red_slot_put(Red4& R, int slot, const floatx16& acc) {
  const int l = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < 16; ++i) R.v[slot][i][l] = acc[i];
}

// Leaves the wave partials in the four slots of R: with eight waves, wave w + 4 adds its accumulator
// to wave w's first (fixed order), so slot w holds acc_w + acc_{w+4}. The caller synchronises before
// reading R. Every thread of the block calls it.
__device__ inline void red_put(Red4& R, floatx16 acc) {
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  if constexpr (kWaves == 8) {
    if (w >= 4) red_slot_put(R, w - 4, acc);
    __syncthreads();
    if (w < 4) {
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] += R.v[w][i][l];
    }
  }
  if (w < 4) red_slot_put(R, w, acc);
}

__device__ inline float red_get(const Red4& R, int w, int r, int c) {
  return R.v[w][4 * (r >> 3) + (r & 3)][c + 32 * ((r >> 2) & 1)];
}

__device__ inline float red_sum4(const Red4& R, int r, int c) {
  return (red_get(R, 0, r, c) + red_get(R, 1, r, c)) + (red_get(R, 2, r, c) + red_get(R, 3, r, c));
}

// Four consecutive values at element `off` of a kp x kp matrix: the FP32 copy (if f32) and, with
// SPLIT, the (hi, lo) BF16 pair stored as [hi | lo] blocks of nel elements each (if s16).
template <bool SPLIT>
__device__ inline void put4(float* f32, uint16_t* s16, int64_t nel, int64_t off, const float v[4]) {
#pragma clang fp contract(off)  // lo is of the rounded v, also where v is a product
  if (f32) *reinterpret_cast<float4*>(f32 + off) = make_float4(v[0], v[1], v[2], v[3]);
  if constexpr (SPLIT) {
    if (s16) {
      bf16x4 hi, lo;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        hi[e] = (__bf16)v[e];
        lo[e] = (__bf16)(v[e] - (float)hi[e]);
      }
      __bf16* s = reinterpret_cast<__bf16*>(s16);
      *reinterpret_cast<bf16x4*>(s + off) = hi;
      *reinterpret_cast<bf16x4*>(s + nel + off) = lo;
    }
  }
}

// Inputs of finish_tile that do not depend on the tile's products, loaded before the MFMA loop so
// that their latency overlaps the operand loads: the previous iterate's block values (for the frob
// log) and mu_A, mu_B of the thread's row (for the m partial sums; as loaded -- a conversion before the loop would
// wait for them ahead of the operand loads).
struct TilePre {
  float pv[4];
  double ua, ub;
};

__device__ inline void tile_pre(TilePre& t, int kp, int64_t i0, int64_t j0, const float* prev, const double* mu_a,
                                const double* mu_b) {
  if (!epi_thread()) return;
  const int r = threadIdx.x >> 3, c4 = 4 * (threadIdx.x & 7);
  if (prev) {
    const float4 p = *reinterpret_cast<const float4*>(prev + (i0 + r) * kp + j0 + c4);
    t.pv[0] = p.x;
    t.pv[1] = p.y;
    t.pv[2] = p.z;
    t.pv[3] = p.w;
  }
  if (mu_a) {
    t.ua = mu_a[i0 + r];
    t.ub = mu_b[i0 + r];
  }
}

// Keeps what is computed from a value loaded early behind this point (the compiler would move it up to the load,
// and the wait for it ahead of the operand loads).
template <typename T>
__device__ inline void late(T& v) {
  asm volatile("" : "+v"(v));
}

// Shared memory of the tile epilogue.
struct TileShm {
  float t[32][33];    // the block transposed
  double d[4];        // per-wave ||Out - prev||^2
  float m[4][2][32];  // per-wave partial column sums mu^T Out
};

// Writes block (i0, j0) of a new kp x kp iterate held as v[e] = element (i0 + r, j0 + c4 + e), with
// r = thread / 8 and c4 = 4 (thread % 8): Out row-major (FP32 and, with SPLIT, BF16 pairs), OutT
// transposed (FP32 without SPLIT, BF16 pairs with it: the transposes are only ever MFMA operands, and
// a later FP32 run rebuilds its FP32 transpose in SETUP), *fslot = ||Out - prev||_F^2 over the block when fslot
// is given (prev in pre.pv; the step's log entry is the sum of its tiles' slots, see frob_sum), and, when
// mpart is given, mpart[(ti * 2 + s) * kp + j] = sum over the block's rows i of mu_s[i] Out[i][j]
// (s = A, B; mu in pre.ua, pre.ub). Every thread of the block calls it. The stores go first: what the next
// kernel waits for is their way to memory, under which the sums are taken.
template <bool SPLIT>
__device__ inline void finish_tile(TileShm& S, int kp, int ti, int64_t i0, int64_t j0, const float v[4], float* Out,
                                   uint16_t* Out16, float* OutT, uint16_t* OutT16, TilePre& pre, double* fslot,
                                   float* mpart) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int r = threadIdx.x >> 3, c4 = 4 * (threadIdx.x & 7);
  const int64_t nel = (int64_t)kp * kp;
  const int64_t off = (i0 + r) * kp + j0 + c4;
  const bool act = epi_thread();  // waves 4.. hold no elements; they only meet the barriers
  if (act) {
#pragma unroll
    for (int e = 0; e < 4; ++e) S.t[c4 + e][r] = v[e];
    put4<SPLIT>(Out, Out16, nel, off, v);
  }
  __syncthreads();
  if (act) {
    const int c = threadIdx.x >> 3, r4 = 4 * (threadIdx.x & 7);
    const float t[4] = {S.t[c][r4], S.t[c][r4 + 1], S.t[c][r4 + 2], S.t[c][r4 + 3]};
    put4<SPLIT>(SPLIT ? nullptr : OutT, OutT16, nel, (j0 + c) * kp + i0 + r4, t);
  }
  if (!fslot && !mpart) return;  // uniform over the block
  if (act && fslot) {
    double d = 0.0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const double dd = (double)v[e] - (double)pre.pv[e];
      d = fma(dd, dd, d);
    }
    d = wave_sum(d);
    if (lane == 0) S.d[w] = d;
  }
  if (act && mpart) {
    // lanes with equal lane % 8 hold the same columns: their eight rows are summed over offsets 8, 16, 32, the last
    // two packed (the odd rows of 16 lanes carry s = B, the upper half the columns 2 and 3)
    late(pre.ua);
    late(pre.ub);
    const float ua = (float)pre.ua, ub = (float)pre.ub;
    float q[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float sa = fmaf(ua, v[e], dpp_mov<kDppRor8>(ua * v[e])), sb = fmaf(ub, v[e], dpp_mov<kDppRor8>(ub * v[e]));
      q[e] = swap_add16(sa, sb);
    }
    const float s01 = swap_add32(q[0], q[2]), s23 = swap_add32(q[1], q[3]);
    if ((lane & 15) < 8) {
      const int h = lane >> 5, sx = (lane >> 4) & 1, c = 4 * (lane & 7) + 2 * h;
      S.m[w][sx][c] = s01;
      S.m[w][sx][c + 1] = s23;
    }
  }
  __syncthreads();
  if (fslot && threadIdx.x == 0) *fslot = (S.d[0] + S.d[1]) + (S.d[2] + S.d[3]);
  if (mpart && threadIdx.x < 64) {
    const int s = threadIdx.x >> 5, c = threadIdx.x & 31;
    mpart[((int64_t)ti * 2 + s) * kp + j0 + c] = (S.m[0][s][c] + S.m[1][s][c]) + (S.m[2][s][c] + S.m[3][s][c]);
  }
}

// ---- the element-wise formulas of the phases, with their roundings fixed (every form of a phase gives the same bits)
__device__ inline float cg_value(float c3, float c1, float p, float q, float ab, float mA, float mB) {
  return fmaf(c3, ab, c1 * fmaf(p, mB, mA * q));
}
__device__ inline float cmu_value(float c0, float c1, float mA, float mB, float ssum, int nb) {
  return fmaf(c0 * mA, mB, c1 * ssum / (float)nb);
}
__device__ inline float step_value(float p0, float eta, float theta, float phh, float t, float inv_b, float muc, float cmu) {
  return fmaf(eta, fmaf(t, inv_b, muc * cmu), fmaf(-(eta * theta), phh, p0));
}
__device__ inline float update_value(float cs, bool quintic, float x, float y) {
  const float c1 = (quintic ? 1.875f : 1.5f) * cs, c3 = quintic ? cs : -0.5f * cs * cs * cs;
  return fmaf(c1, x, c3 * y);
}
__device__ inline float qpoly_value(float cs, float g, float gg) {
  const float c2 = cs * cs;
  const float a1 = -1.25f * c2, a2 = 0.375f * c2 * c2;
  return fmaf(a2, gg, a1 * g);
}
__device__ inline float guard_value(float mx) { return mx > 2.f ? sqrtf(2.f / mx) : 1.f; }

template <typename T>
__device__ inline void store4(T* p, const float v[4]) {
  if constexpr (sizeof(T) == 2) {
    bf16x4 x;
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = (__bf16)v[e];
    *reinterpret_cast<bf16x4*>(p) = x;
  } else {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
  }
}

// ---- the phases of one step, as per-tile device functions ----------------------------------------
// A step is the phase sequence P1, P2, then ns_iters x (GRAM, UPDATE) -- (GRAM, QPOLY, UPDATE) for
// degree-5 iterations -- or COPY when the step does not renormalise; SETUP precedes the first step of
// a run and FROB follows its last. In the reference's QR mode a renormalising step is P1, P2, the
// host's QR launches and QRFIN. The kernel that finishes a step leaves one partial of the step's log
// entry per tile; the next step's P1 (or FROB) sums them in a fixed order. The same tile functions
// serve the per-phase launches of one instance (stgd_phase_kernel, blockIdx.x = tile) and the
// persistent launch over many instances (stgd_batch_kernel, tiles from a work queue).
enum StgdPhase { PH_SETUP = 0, PH_P1 = 1, PH_P2 = 2, PH_GRAM = 3, PH_UPDATE = 4, PH_COPY = 5, PH_QPOLY = 6, PH_QRFIN = 7,
                 PH_FROB = 8,
                 PH_P2S = 9 };  // P2 spread wider, for one instance's launches (see p2_spread)

// What one phase of one step reads and writes, resolved on the host: every pointer is the one to use (the Phi
// ping-pong, the Newton-Schulz scratch of the iteration, the minibatch's first row), so that a kernel fetches
// its arguments in one go instead of walking a context. Operands are FP32 or split BF16 ([hi | lo]) by the run's
// mode; the *16 outputs are null in FP32 runs.
struct P1Args {
  const void *ya, *yb;   // the minibatch's first row, leading dimension kp
  const void* phiT;      // operand
  const float* mpart;
  void* cgt;
  float *cs_part, *mab;
  float* h;
  uint16_t* h16;
  double* frob_prev;     // the previous step's log entry within the run (null for the run's first), formed here from
  const double* fpart;   // the previous step's tile partials
  int32_t kp, b, nb;
  float c3, c1;
};
struct P2Args {
  const void *phi_op, *h_op;
  const float* phi;
  const void* yct;       // the minibatch's first column, leading dimension n_pad
  const void* cgt;
  const float *cs_part, *mab;
  const double* mu_c;
  float* out;
  uint16_t* out16;
  float* outT;
  uint16_t* outT16;
  unsigned long long* rowsum;  // cleared for the first Newton-Schulz iteration
  double* fpart;               // null unless the log is taken before the renormalisation
  int64_t n_pad;
  int32_t kp, b, nb, aligned;  // aligned: yct rows start on 16 bytes
  float eta, theta, c0, c1;
};
struct GramArgs {
  const void* xT;
  float* g;
  uint16_t* g16;
  unsigned long long* rowsum;
  int32_t kp;
};
struct QpolyArgs {
  const void* g_op;
  const float* g;
  float* q;
  uint16_t* q16;
  const unsigned long long* rowsum;
  int32_t kp;
};
struct UpdateArgs {
  const void *x_op, *g_op;     // g_op: G (degree 3) or Q (degree 5)
  const float* x;
  float* out;
  uint16_t* out16;
  float* outT;
  uint16_t* outT16;
  const float* prev;           // the last iteration logs ||out - prev||^2 (fpart) and the m partials (mpart); else null
  const double *mu_a, *mu_b;
  double* fpart;
  float* mpart;
  const unsigned long long* rowsum;
  unsigned long long* rowsum_next;
  int32_t kp, quintic;
};
struct CopyArgs {              // COPY, QRFIN and SETUP
  const float* x;
  float* out;                  // null in SETUP
  uint16_t* out16;
  float* outT;
  uint16_t* outT16;
  const float* prev;
  const double *mu_a, *mu_b;
  double* fpart;
  float* mpart;
  double* frob_zero;           // SETUP: the run's log entries, cleared by tile 0
  int64_t nfrob;
  int32_t kp, kmax;            // rows and columns from kmax on become zero
};
struct FrobArgs {
  double* frob;
  const double* fpart;
  int32_t kp;
};
union PhaseArgs {
  P1Args p1;
  P2Args p2;
  GramArgs gram;
  QpolyArgs qpoly;
  UpdateArgs update;
  CopyArgs copy;
  FrobArgs frob;
};

template <int PHASE>
__host__ __device__ inline const auto& phase_args(const PhaseArgs& a) {
  if constexpr (PHASE == PH_P1) return a.p1;
  else if constexpr (PHASE == PH_P2 || PHASE == PH_P2S) return a.p2;
  else if constexpr (PHASE == PH_GRAM) return a.gram;
  else if constexpr (PHASE == PH_QPOLY) return a.qpoly;
  else if constexpr (PHASE == PH_UPDATE) return a.update;
  else if constexpr (PHASE == PH_FROB) return a.frob;
  else return a.copy;
}
template <int PHASE>
struct ArgsOf { using type = CopyArgs; };
template <> struct ArgsOf<PH_P1> { using type = P1Args; };
template <> struct ArgsOf<PH_P2> { using type = P2Args; };
template <> struct ArgsOf<PH_P2S> { using type = P2Args; };
template <> struct ArgsOf<PH_GRAM> { using type = GramArgs; };
template <> struct ArgsOf<PH_QPOLY> { using type = QpolyArgs; };
template <> struct ArgsOf<PH_UPDATE> { using type = UpdateArgs; };
template <> struct ArgsOf<PH_FROB> { using type = FrobArgs; };

// The end test of a step (per-phase launches only).
struct StopArgs {
  StgdStop* stop;
  int64_t st;        // step index within the run
  double thresh;
  int64_t iter_min, iter_max;
};

union StgdSmem {
  struct {
    Red4 red[2];  // data tiles: the four waves' partials of P_A (red[0]) and P_B (red[1])
    float mvec[2][32];
  } p1;
  struct {
    Red4 red;
    TileShm S;
    float cmu[32];
    float cscale;
  } p2;
  TileShm S;
};

// Tiles of a phase. The symmetric products -- H = (Phi^T Phi)^o2 in P1, G = X^T X in GRAM -- are
// computed on the upper triangle of 32 x 32 blocks only, each off-diagonal block written twice.
__host__ __device__ inline int phase_tiles(int phase, int kp, int b) {
  const int ntk = kp / 32, tri = ntk * (ntk + 1) / 2;
  switch (phase) {
    case PH_P1: return (b / 32) * ntk + tri;
    case PH_GRAM: return tri;
    case PH_FROB: return 1;
    default: return ntk * ntk;
  }
}

// Block (ti, tj), ti <= tj, of upper-triangle tile t (row-major over the triangle): the row from the root of its
// first tile's index i (2 ntk + 1 - i) / 2 <= t, corrected by one where the rounded root is off.
__device__ inline void tri_tile(int t, int ntk, int& ti, int& tj) {
  const float n = (float)(2 * ntk + 1);
  int i = (int)((n - sqrtf(fmaxf(n * n - 8.f * (float)t, 0.f))) * 0.5f);
  i = min(max(i, 0), ntk - 1);
  if (i * (2 * ntk + 1 - i) / 2 > t) --i;
  if ((i + 1) * (2 * ntk - i) / 2 <= t) ++i;
  ti = __builtin_amdgcn_readfirstlane(i);
  tj = ti + t - ti * (2 * ntk + 1 - ti) / 2;
}

// The log entry ||Phi_{t+1} - Phi_t||_F^2 of a finished step from its tiles' partials fpart[0 .. n):
// lane-strided sums, then a butterfly -- a fixed order, so that every wave that forms the entry gets
// the same bits. Called by whole waves.
__device__ inline double frob_sum(const double* fpart, int n) {
  const int lane = threadIdx.x & 63;
  double s = 0.0;
#pragma unroll 4
  for (int t = lane; t < n; t += 64) s += fpart[t];
  return wave_sum(s);
}

// A kp x kp operand of one mode: FP32 data, or the BF16 (hi, lo) pair.
template <int MODE>
__device__ inline Opnd<op_t<MODE>> pick(const void* p, int64_t nel, int64_t ld) {
  const op_t<MODE>* q = static_cast<const op_t<MODE>*>(p);
  if constexpr (MODE == MM_F32) return opnd<float>(q, nullptr, ld);
  else return opnd<__bf16>(q, q + nel, ld);
}

// Sums of strided partials, one per output column: out[o] = sum_{t < nt} src[t * stride + off(o)]
// for 64 outputs (P1: m_A, m_B of 32 columns) or 32 (P2: column sums). The loads of all threads
// are issued by part_load before the MFMA loop and reduced by part_reduce after it, so their
// latency overlaps the operand loads instead of forming a chain.
constexpr int kPartRegs = 4;
struct PartSum {
  float v[kPartRegs];
  int extra;  // partials beyond kPartRegs * lanes-per-output, summed late (large k or b)
};

// P1: tile (ti rows of Phi) partials of m_s[j0 + c]: thread -> output o = t / 4 (s = o / 32,
// c = o % 32), lane q = t % 4 takes ti = q, q + 4, ...
__device__ inline void mpart_load(PartSum& ps, const float* mpart, int kp, int ntk, int64_t j0) {
  const int o = threadIdx.x >> 2, q = threadIdx.x & 3;
  const int s = o >> 5, c = o & 31;
#pragma unroll
  for (int u = 0; u < kPartRegs; ++u) {
    const int ti = q + 4 * u;
    ps.v[u] = ti < ntk ? mpart[((int64_t)ti * 2 + s) * kp + j0 + c] : 0.f;
  }
  ps.extra = ntk > 4 * kPartRegs;
}

__device__ inline float mpart_reduce(const PartSum& ps, const float* mpart, int kp, int ntk, int64_t j0) {
  const int o = threadIdx.x >> 2, q = threadIdx.x & 3;
  const int s = o >> 5, c = o & 31;
  float m = (ps.v[0] + ps.v[1]) + (ps.v[2] + ps.v[3]);
  if (ps.extra)
    for (int ti = q + 4 * kPartRegs; ti < ntk; ti += 4) m += mpart[((int64_t)ti * 2 + s) * kp + j0 + c];
  return quad_sum(m);  // valid in every lane of the output's group of four
}

// P2: column sums of the b/32 row-tile partials cs_part[tb][j0 + c]: thread -> c = t / 8,
// lane q = t % 8 takes tb = q, q + 8, ...
__device__ inline void cspart_load(PartSum& ps, const float* cs_part, int kp, int ntb, int64_t j0) {
  const int c = threadIdx.x >> 3, q = threadIdx.x & 7;
#pragma unroll
  for (int u = 0; u < kPartRegs; ++u) {
    const int tb = q + 8 * u;
    ps.v[u] = tb < ntb ? cs_part[(int64_t)tb * kp + j0 + c] : 0.f;
  }
  ps.extra = ntb > 8 * kPartRegs;
}

__device__ inline float cspart_reduce(const PartSum& ps, const float* cs_part, int kp, int ntb, int64_t j0) {
  const int c = threadIdx.x >> 3, q = threadIdx.x & 7;
  float m = (ps.v[0] + ps.v[1]) + (ps.v[2] + ps.v[3]);
  if (ps.extra)
    for (int tb = q + 8 * kPartRegs; tb < ntb; tb += 8) m += cs_part[(int64_t)tb * kp + j0 + c];
  return oct_sum(m);
}

// P1 tiles [0, ntk (ntk + 1) / 2): upper-triangle H tiles; the rest: a 32-row slice of the minibatch x
// 32 columns of C_g. Tile 0 also forms the previous step's log entry (wave 0; the partials' loads go first).
template <int DMODE, int KMODE, typename TY, typename TPH>
__device__ __forceinline__ void p1_tile(const P1Args& a, int tile, StgdSmem& sm, bool log) {
  constexpr bool SPLIT = KMODE == MM_BF16X3;
  // three workgroups per compute unit need at most 168 registers: at k = 500, b = 1024 (2048) P1 takes 7.5 (10.6) us,
  // 8.6 (11.3) with the five bodies and their spills, 7.5 (11.2) with two workgroups
  constexpr bool COMPACT = DMODE == MM_BF16;
  const int kp = a.kp;
  const int ntk = kp / 32;
  const int64_t nel = (int64_t)kp * kp;
  const int w = wave_id();
  const int tri = ntk * (ntk + 1) / 2;
  floatx16 acc = {};
  int64_t k0, kl;
  if (tile >= tri) {  // data tiles follow the H tiles, which then start in the first wave
    tile -= tri;
    const int tb = tile / ntk, tj = tile % ntk;
    const int64_t x0 = (int64_t)tb * 32, j0 = (int64_t)tj * 32;
    PartSum ps;
    if (epi_thread()) mpart_load(ps, a.mpart, kp, ntk, j0);  // m_A, m_B of the block's columns
    // every wave: P_A and P_B over its part of the k reduction, sharing the Phi^T fragments
    floatx16 acc_b = {};
    kslice<DMODE>(kp, kWaves, w, k0, kl);
    wave_mm_pair<DMODE, COMPACT>(acc, acc_b, static_cast<const TY*>(a.ya), static_cast<const TY*>(a.yb), kp,
                        pick<DMODE>(a.phiT, nel, kp).hi, kp, x0, j0, k0, kl);
    if (epi_thread()) {
      const float m = mpart_reduce(ps, a.mpart, kp, ntk, j0);
      const int o = threadIdx.x >> 2;
      if ((threadIdx.x & 3) == 0) sm.p1.mvec[o >> 5][o & 31] = m;
    }
    red_put(sm.p1.red[0], acc);
    red_put(sm.p1.red[1], acc_b);
    __syncthreads();
    if (!epi_thread()) return;
    // C_g^T rows are columns j of the block: thread -> column c, rows r4 .. r4 + 3
    const int c = threadIdx.x >> 3, r4 = 4 * (threadIdx.x & 7);
    const float mA = sm.p1.mvec[0][c], mB = sm.p1.mvec[1][c];
    float cg[4], cs = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = r4 + e;
      const float p = red_sum4(sm.p1.red[0], r, c);
      const float q = red_sum4(sm.p1.red[1], r, c);
      const bool valid = (x0 + r) < a.nb;
      const float ab = p * q;
      cs += valid ? ab : 0.f;
      cg[e] = valid ? cg_value(a.c3, a.c1, p, q, ab, mA, mB) : 0.f;
    }
    store4(static_cast<TPH*>(a.cgt) + (j0 + c) * (int64_t)a.b + x0 + r4, cg);
    cs = oct_sum(cs);
    if ((threadIdx.x & 7) == 0) {
      a.cs_part[(int64_t)tb * kp + j0 + c] = cs;
      if (tb == 0) {
        a.mab[j0 + c] = mA;
        a.mab[kp + j0 + c] = mB;
      }
    }
  } else {
    log = log && tile == 0 && a.frob_prev && w == 0;
    double fs = 0.0;
    if (log) {
#pragma unroll 4
      for (int t = threadIdx.x; t < ntk * ntk; t += 64) fs += a.fpart[t];
    }
    int ti, tj;
    tri_tile(tile, ntk, ti, tj);
    const int64_t i0 = (int64_t)ti * 32, j0 = (int64_t)tj * 32;
    const Opnd<op_t<KMODE>> phiT_k = pick<KMODE>(a.phiT, nel, kp);
    kslice<KMODE>(kp, kWaves, w, k0, kl);
    wave_mm<KMODE, true, 2, COMPACT>(acc, phiT_k, phiT_k, i0, j0, k0, kl);  // G = Phi^T Phi
    if (log) {
      const double f = wave_sum(fs);
      if (threadIdx.x == 0) *a.frob_prev = f;
    }
    Red4& red = sm.p1.red[0];
    red_put(red, acc);
    __syncthreads();
    if (!epi_thread()) return;
    const int r = threadIdx.x >> 3, c4 = 4 * (threadIdx.x & 7);
    float g[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      g[e] = red_sum4(red, r, c4 + e);
      g[e] *= g[e];
    }
    put4<SPLIT>(a.h, a.h16, nel, (i0 + r) * kp + j0 + c4, g);
    if (ti != tj) {  // the mirror block (j, i): thread -> row c of it, columns r4 .. r4 + 3
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        g[e] = red_sum4(red, c4 + e, r);
        g[e] *= g[e];
      }
      put4<SPLIT>(a.h, a.h16, nel, (j0 + r) * kp + i0 + c4, g);
    }
  }
}

template <int DMODE, int KMODE, typename TY, typename TPH>
__device__ __forceinline__ void p2_tile(const P2Args& a, int tile, StgdSmem& sm) {
  constexpr bool SPLIT = KMODE == MM_BF16X3;
  const int kp = a.kp, ntk = kp / 32;
  const int64_t nel = (int64_t)kp * kp;
  const int w = wave_id();
  const int ti = tile / ntk, tj = tile % ntk;
  const int64_t i0 = (int64_t)ti * 32, j0 = (int64_t)tj * 32;
  Red4& red = sm.p2.red;
  floatx16 acc = {};
  int64_t k0, kl;
  PartSum ps;  // column sums of P_A o P_B and m_A, m_B for c_mu, gathered during the MFMA loop
  const bool epi = epi_thread();
  const int r = threadIdx.x >> 3, c4 = 4 * (threadIdx.x & 7);
  float mab_a = 0.f, mab_b = 0.f;
  double muc_d = 0.0;  // converted after the MFMA loop
  float4 ph = make_float4(0.f, 0.f, 0.f, 0.f);
  if (epi) {  // epilogue inputs, loaded ahead of the MFMA loop
    cspart_load(ps, a.cs_part, kp, a.b / 32, j0);
    mab_a = a.mab[j0 + (threadIdx.x >> 3)];
    mab_b = a.mab[kp + j0 + (threadIdx.x >> 3)];
    muc_d = a.mu_c[i0 + r];
    ph = *reinterpret_cast<const float4*>(a.phi + (i0 + r) * kp + j0 + c4);
  }
  // waves with (w & 2) == 0 take Phi H, the others Y_C^T C_g, each over kWaves / 2 parts of its range;
  // after red_put, slots 0, 1 hold Phi H and slots 2, 3 Y_C^T C_g
  const int part = (w & 1) + 2 * (w >> 2);
  if ((w & 2) == 0) {  // Phi H (H symmetric: row j of H is column j)
    kslice<KMODE>(kp, kWaves / 2, part, k0, kl);
    wave_mm<KMODE, true>(acc, pick<KMODE>(a.phi_op, nel, kp), pick<KMODE>(a.h_op, nel, kp), i0, j0, k0, kl);
  } else {             // Y_C^T C_g over parts of the minibatch tile
    kslice<DMODE>(a.b, kWaves / 2, part, k0, kl);
    const Opnd<TY> yc = opnd<TY>(static_cast<const TY*>(a.yct), nullptr, a.n_pad);
    const Opnd<TPH> cg = opnd<TPH>(static_cast<const TPH*>(a.cgt), nullptr, a.b);
    if (a.aligned)
      wave_mm<DMODE, true, 4>(acc, yc, cg, i0, j0, k0, kl);
    else
      wave_mm<DMODE, false, 4>(acc, yc, cg, i0, j0, k0, kl);
  }
  if (epi) {
    const int c = threadIdx.x >> 3;
    const float ssum = cspart_reduce(ps, a.cs_part, kp, a.b / 32, j0);
    if ((threadIdx.x & 7) == 0) sm.p2.cmu[c] = cmu_value(a.c0, a.c1, mab_a, mab_b, ssum, a.nb);
  }
  if (tile == 0)
    for (int t = threadIdx.x; t < kp; t += blockDim.x) a.rowsum[t] = 0ull;
  red_put(red, acc);
  __syncthreads();
  late(muc_d);
  const float inv_b = 1.f / (float)a.nb, muc = (float)muc_d;
  const float p0[4] = {ph.x, ph.y, ph.z, ph.w};
  float v[4] = {0.f, 0.f, 0.f, 0.f};
  if (epi) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int c = c4 + e;
      const float phh = red_get(red, 0, r, c) + red_get(red, 1, r, c);
      const float t = red_get(red, 2, r, c) + red_get(red, 3, r, c);
      v[e] = step_value(p0[e], a.eta, a.theta, phh, t, inv_b, muc, sm.p2.cmu[c]);
    }
  }
  TilePre pre{};  // the reference's log: ||Phi~ - Phi||^2 before the renormalisation
#pragma unroll
  for (int e = 0; e < 4; ++e) pre.pv[e] = p0[e];
  finish_tile<SPLIT>(sm.p2.S, kp, ti, i0, j0, v, a.out, a.out16, a.outT, a.outT16, pre, a.fpart ? a.fpart + tile : nullptr, nullptr);
}

// A block of 16 rows x 128 bytes of an FP32 operand: loaded and put into the layout of the 16 x 16 x 4 MFMA through the
// wave's buffer, in the k order of the 32-row blocks (8 c + e, 8 c + 4 + e for e = 0 .. 3). Both MFMA shapes add one
// product after the other in k order, so the 16-row blocks give the 32-row blocks' bits.
template <bool AL>
__device__ inline void quad_load(u32x4 v[2], const float* row0, int64_t ld) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t off = ((lane >> 3) * (uint32_t)ld + (lane & 7) * 4) * 4;
  const char* base = reinterpret_cast<const char*>(row0);
#pragma unroll
  for (int c = 0; c < 2; ++c) v[c] = ld16<AL>(reinterpret_cast<const float*>(base + 32 * c * ld + off));
}

struct QuadFrag {
  u32x4 a[2], b[2];
  __device__ inline void swap() {
    u32x4* buf = wave_stage();  // A's rows, then B's
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int row = (lane >> 3) + 8 * c, at = row * 8 + ((lane & 7) ^ ((row >> 1) & 7));
      buf[at] = a[c];
      buf[128 + at] = b[c];
    }
    asm volatile("" ::: "memory");
    const uint32_t* p = reinterpret_cast<const uint32_t*>(buf) + (g >> 1);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int at = 4 * (r * 8 + ((2 * c + (g & 1)) ^ ((r >> 1) & 7)));
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        a[c >> 1][2 * (c & 1) + e] = p[at + 2 * e];
        b[c >> 1][2 * (c & 1) + e] = p[512 + at + 2 * e];
      }
    }
    asm volatile("" ::: "memory");
  }
  __device__ inline void mma(floatx4& acc) const {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const floatx4 x = as_f32(a[c]), y = as_f32(b[c]);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], y[e], acc, 0, 0, 0);
    }
  }
};

// wave_mm of one 16 x 16 block in FP32.
template <bool AAL>
__device__ inline void quad_mm(floatx4& acc, const float* a, int64_t lda, const float* b, int64_t ldb, int64_t kl) {
  QuadFrag f[4];
  pipelined<32>(
      f, kl,
      [&](QuadFrag& x, auto k) {
        quad_load<AAL>(x.a, a + k, lda);
        quad_load<true>(x.b, b + k, ldb);
      },
      [&](QuadFrag& x) { x.mma(acc); });
}

// P2 of an FP32 step in 16 x 16 tiles, four times the workgroups: of a 32 x 32 tile the two waves that take Y_C^T C_g
// pass MFMAs in a row for 6.8 us at b = 1024 while most compute units have no tile (16 tiles at k = 100). P2 at k = 100,
// b = 1024 (2048): 4.3 (8.1) us against 10.9 (20.5). Two waves take each of the two products: builds with eight waves per
// workgroup have no such tiles.
__device__ __forceinline__ void p2_quad_tile(const P2Args& a, int tile, StgdSmem& sm) {
  const int kp = a.kp, nq = kp / 16;
  const int w = wave_id(), lane = threadIdx.x & 63;
  const int64_t i0 = (int64_t)(tile / nq) * 16, j0 = (int64_t)(tile % nq) * 16;
  const int r = threadIdx.x >> 4, c = threadIdx.x & 15, pc = threadIdx.x >> 3;  // pc < 16: column of c_mu
  floatx4 acc = {};
  int64_t k0, kl;
  PartSum ps;
  float mab_a = 0.f, mab_b = 0.f;
  double muc_d = a.mu_c[i0 + r];
  float p0 = a.phi[(i0 + r) * kp + j0 + c];
  if (pc < 16) {
    cspart_load(ps, a.cs_part, kp, a.b / 32, j0);
    mab_a = a.mab[j0 + pc];
    mab_b = a.mab[kp + j0 + pc];
  }
  if ((w & 2) == 0) {
    kslice<MM_F32>(kp, 2, w & 1, k0, kl);
    quad_mm<true>(acc, static_cast<const float*>(a.phi_op) + i0 * kp + k0, kp, static_cast<const float*>(a.h_op) + j0 * kp + k0,
                  kp, kl);
  } else {
    kslice<MM_F32>(a.b, 2, w & 1, k0, kl);
    const float* yc = static_cast<const float*>(a.yct) + i0 * a.n_pad + k0;
    const float* cg = static_cast<const float*>(a.cgt) + j0 * a.b + k0;
    if (a.aligned) quad_mm<true>(acc, yc, a.n_pad, cg, a.b, kl);
    else quad_mm<false>(acc, yc, a.n_pad, cg, a.b, kl);
  }
  if (pc < 16) {
    const float ssum = cspart_reduce(ps, a.cs_part, kp, a.b / 32, j0);
    if ((threadIdx.x & 7) == 0) sm.p2.cmu[pc] = cmu_value(a.c0, a.c1, mab_a, mab_b, ssum, a.nb);
  }
  if (tile == 0)
    for (int t = threadIdx.x; t < kp; t += blockDim.x) a.rowsum[t] = 0ull;
  float (*red)[4][66] = reinterpret_cast<float (*)[4][66]>(&sm.p2.red);  // acc[i] of lane l: element (4 (l / 16) + i, l % 16)
#pragma unroll
  for (int i = 0; i < 4; ++i) red[w][i][lane] = acc[i];
  __syncthreads();
  late(muc_d);
  late(p0);
  const int ri = r & 3, rl = 16 * (r >> 2) + c;
  const float phh = red[0][ri][rl] + red[1][ri][rl], t = red[2][ri][rl] + red[3][ri][rl];
  const float v = step_value(p0, a.eta, a.theta, phh, t, 1.f / (float)a.nb, (float)muc_d, sm.p2.cmu[c]);
  a.out[(i0 + r) * kp + j0 + c] = v;
  sm.p2.S.t[c][r] = v;
  __syncthreads();
  a.outT[(j0 + r) * kp + i0 + c] = sm.p2.S.t[r][c];
}

// The Newton-Schulz scale guard c = min(1, sqrt(2 / ||G||_inf)) from the row sums of |G|, computed
// by wave 3 of a block: guard_load issues the loads before the block's MFMA loop, guard_scale
// reduces them after it and leaves c in *cscale (shared memory; read after the next barrier).
// The row sums are accumulated across tiles as fixed-point integers (units of 2^-32): integer
// addition is associative, so the sums -- and the guard they decide -- do not depend on the order in
// which the tiles' atomics land, and Phi is bit-reproducible from run to run. Partial sums are
// clamped at 2^30, far beyond the point where the guard acts. The largest is found among the integers and
// converted once (conversion is monotone): converted one by one under a branch each, eight loads of a wave came
// back one after another, 2.3 us of an UPDATE at kp = 512.
__device__ inline unsigned long long fix32(float s) {
  return (unsigned long long)(long long)llrintf(fminf(s, 1073741824.f) * 4294967296.f);
}

__device__ inline void guard_load(unsigned long long rs[8], const unsigned long long* rowsum, int kp) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int u = 0; u < 8; ++u) rs[u] = rowsum[min(lane + 64 * u, kp - 1)];
}

__device__ inline void guard_scale(unsigned long long rs[8], const unsigned long long* rowsum, int kp, float* cscale) {
  const int lane = threadIdx.x & 63;
  unsigned long long m = 0;
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    late(rs[u]);
    m = rs[u] > m ? rs[u] : m;
  }
  for (int t = lane + 512; t < kp; t += 64) m = rowsum[t] > m ? rowsum[t] : m;
  const float mx = (float)(wave_max((double)m) * 2.3283064365386963e-10);
  if (lane == 0) *cscale = guard_value(mx);
}

// G = X^T X of a Newton-Schulz iteration on upper-triangle tile `tile` (block and mirror), and
// rowsum[i] += sum over the block's columns of |G_ij| for every row i the block and its mirror cover (the atomics
// go out before the stores, whose way to memory is the shorter).
template <int KMODE>
__device__ __forceinline__ void gram_tile(const GramArgs& a, int tile, StgdSmem& sm) {
  constexpr bool SPLIT = KMODE == MM_BF16X3;
  const int kp = a.kp, ntk = kp / 32;
  const int64_t nel = (int64_t)kp * kp;
  const int w = wave_id();
  int ti, tj;
  tri_tile(tile, ntk, ti, tj);
  const int64_t i0 = (int64_t)ti * 32, j0 = (int64_t)tj * 32;
  Red4& red = sm.p2.red;
  floatx16 acc = {};
  int64_t k0, kl;
  const Opnd<op_t<KMODE>> xT = pick<KMODE>(a.xT, nel, kp);
  kslice<KMODE>(kp, kWaves, w, k0, kl);
  wave_mm<KMODE, true>(acc, xT, xT, i0, j0, k0, kl);
  red_put(red, acc);
  __syncthreads();
  if (!epi_thread()) return;
  const int r = threadIdx.x >> 3, c4 = 4 * (threadIdx.x & 7);
  float g[4], t[4], s = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    g[e] = red_sum4(red, r, c4 + e);
    s += fabsf(g[e]);
  }
  s = oct_sum(s);
  if ((threadIdx.x & 7) == 0) atomicAdd(a.rowsum + i0 + r, fix32(s));
  if (ti != tj) {  // the mirror block (j, i): thread -> row r of it, columns c4 .. c4 + 3
    s = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      t[e] = red_sum4(red, c4 + e, r);
      s += fabsf(t[e]);
    }
    s = oct_sum(s);
    if ((threadIdx.x & 7) == 0) atomicAdd(a.rowsum + j0 + r, fix32(s));
  }
  put4<SPLIT>(a.g, a.g16, nel, (i0 + r) * kp + j0 + c4, g);
  if (ti != tj) put4<SPLIT>(a.g, a.g16, nel, (j0 + r) * kp + i0 + c4, t);
}

// Degree-5 iteration, second stage: Q = -(5/4) c^2 G + (3/8) c^4 G^2 (symmetric, as G), so that the
// update is Xout = c X (15/8 I + Q).
template <int KMODE>
__device__ __forceinline__ void qpoly_tile(const QpolyArgs& a, int tile, StgdSmem& sm) {
  constexpr bool SPLIT = KMODE == MM_BF16X3;
  const int kp = a.kp, ntk = kp / 32;
  const int64_t nel = (int64_t)kp * kp;
  const int w = wave_id();
  const int ti = tile / ntk, tj = tile % ntk;
  const int64_t i0 = (int64_t)ti * 32, j0 = (int64_t)tj * 32;
  Red4& red = sm.p2.red;
  floatx16 acc = {};
  int64_t k0, kl;
  kslice<KMODE>(kp, kWaves, w, k0, kl);
  unsigned long long rs[8];
  if (w == 3) guard_load(rs, a.rowsum, kp);
  const int r = threadIdx.x >> 3, c4 = 4 * (threadIdx.x & 7);
  float4 gv = make_float4(0.f, 0.f, 0.f, 0.f);
  if (epi_thread()) gv = *reinterpret_cast<const float4*>(a.g + (i0 + r) * kp + j0 + c4);
  const Opnd<op_t<KMODE>> g = pick<KMODE>(a.g_op, nel, kp);
  wave_mm<KMODE, true>(acc, g, g, i0, j0, k0, kl);  // (G G)_ij = G[i,:] . G[j,:] (G symmetric)
  if (w == 3) guard_scale(rs, a.rowsum, kp, &sm.p2.cscale);
  red_put(red, acc);
  __syncthreads();
  if (!epi_thread()) return;
  const float cs = sm.p2.cscale;
  const float gg[4] = {gv.x, gv.y, gv.z, gv.w};
  float v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = qpoly_value(cs, gg[e], red_sum4(red, r, c4 + e));
  put4<SPLIT>(a.q, a.q16, nel, (i0 + r) * kp + j0 + c4, v);
}

// Degree 3: Xout = c (1.5 X - 0.5 c^2 X G); degree 5: Xout = c (1.875 X + X Q). The outputs are those
// of finish_tile (the last iteration also logs ||Phi_next - Phi||^2 and the partial sums of m_A, m_B).
template <int KMODE>
__device__ __forceinline__ void update_tile(const UpdateArgs& a, int tile, StgdSmem& sm) {
  constexpr bool SPLIT = KMODE == MM_BF16X3;
  const int kp = a.kp, ntk = kp / 32;
  const int64_t nel = (int64_t)kp * kp;
  const int w = wave_id();
  const int ti = tile / ntk, tj = tile % ntk;
  const int64_t i0 = (int64_t)ti * 32, j0 = (int64_t)tj * 32;
  Red4& red = sm.p2.red;
  floatx16 acc = {};
  int64_t k0, kl;
  kslice<KMODE>(kp, kWaves, w, k0, kl);
  unsigned long long rs[8];
  if (w == 3) guard_load(rs, a.rowsum, kp);
  const bool quintic = a.quintic;
  const int r = threadIdx.x >> 3, c4 = 4 * (threadIdx.x & 7);
  float4 xv = make_float4(0.f, 0.f, 0.f, 0.f);
  if (epi_thread()) xv = *reinterpret_cast<const float4*>(a.x + (i0 + r) * kp + j0 + c4);
  TilePre pre;
  tile_pre(pre, kp, i0, j0, a.prev, a.prev ? a.mu_a : nullptr, a.mu_b);
  wave_mm<KMODE, true>(acc, pick<KMODE>(a.x_op, nel, kp), pick<KMODE>(a.g_op, nel, kp), i0, j0, k0, kl);  // X G or X Q (both symmetric)
  if (w == 3) guard_scale(rs, a.rowsum, kp, &sm.p2.cscale);
  if (tile == 0)
    for (int t = threadIdx.x; t < kp; t += blockDim.x) a.rowsum_next[t] = 0ull;
  red_put(red, acc);
  __syncthreads();
  const float cs = sm.p2.cscale;
  const float x[4] = {xv.x, xv.y, xv.z, xv.w};
  float v[4] = {0.f, 0.f, 0.f, 0.f};
  if (epi_thread())
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = update_value(cs, quintic, x[e], red_sum4(red, r, c4 + e));
  finish_tile<SPLIT>(sm.p2.S, kp, ti, i0, j0, v, a.out, a.out16, a.outT, a.outT16, pre, a.fpart ? a.fpart + tile : nullptr,
                     a.mpart);
}

// COPY: Phi_next = Phi~ with the outputs of a last update; QRFIN: Phi_next = the QR factor the host
// launches left in phia (rows and columns from k on set to zero), without a log entry (the step logged
// before its QR). SETUP: the derived copies of the current Phi (split pairs, Phi^T, the m partial
// sums), and tile 0 clears the run's frob entries.
template <bool SPLIT>
__device__ __forceinline__ void copy_tile(const CopyArgs& a, int tile, StgdSmem& sm) {
  const int kp = a.kp, ntk = kp / 32;
  const int ti = tile / ntk, tj = tile % ntk;
  const int64_t i0 = (int64_t)ti * 32, j0 = (int64_t)tj * 32;
  const int r = threadIdx.x >> 3, c4 = 4 * (threadIdx.x & 7);
  float4 xv = make_float4(0.f, 0.f, 0.f, 0.f);
  if (epi_thread()) xv = *reinterpret_cast<const float4*>(a.x + (i0 + r) * kp + j0 + c4);
  float v[4] = {xv.x, xv.y, xv.z, xv.w};
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (i0 + r >= a.kmax || j0 + c4 + e >= a.kmax) v[e] = 0.f;
  if (a.frob_zero && tile == 0)
    for (int64_t t = threadIdx.x; t < a.nfrob; t += blockDim.x) a.frob_zero[t] = 0.0;
  TilePre pre;
  tile_pre(pre, kp, i0, j0, a.prev, a.mu_a, a.mu_b);
  finish_tile<SPLIT>(sm.S, kp, ti, i0, j0, v, a.out, a.out16, a.outT, a.outT16, pre, a.fpart ? a.fpart + tile : nullptr, a.mpart);
}

// FROB: the log entry of a run's last step from its tiles' partials (one wave).
__device__ __forceinline__ void frob_final(const FrobArgs& a) {
  if (threadIdx.x >= 64) return;
  const int ntk = a.kp / 32;
  const double f = frob_sum(a.fpart, ntk * ntk);
  if (threadIdx.x == 0) *a.frob = f;
}

template <int DMODE, int KMODE, typename TY, typename TPH, int PHASE>
__device__ __forceinline__ void phase_tile(const typename ArgsOf<PHASE>::type& a, int tile, StgdSmem& sm, bool log = true) {
  constexpr bool SPLIT = KMODE == MM_BF16X3;
  if constexpr (PHASE == PH_P1) p1_tile<DMODE, KMODE, TY, TPH>(a, tile, sm, log);
  else if constexpr (PHASE == PH_P2) p2_tile<DMODE, KMODE, TY, TPH>(a, tile, sm);
  else if constexpr (PHASE == PH_P2S) {
    static_assert(PHASE == PH_P2S && kWaves == 4, "four waves per tile");
    p2_quad_tile(a, tile, sm);
  }
  else if constexpr (PHASE == PH_GRAM) gram_tile<KMODE>(a, tile, sm);
  else if constexpr (PHASE == PH_QPOLY) qpoly_tile<KMODE>(a, tile, sm);
  else if constexpr (PHASE == PH_UPDATE) update_tile<KMODE>(a, tile, sm);
  else if constexpr (PHASE == PH_FROB) frob_final(a);
  else copy_tile<SPLIT>(a, tile, sm);
}

template <int DMODE, int KMODE, typename TY, typename TPH>
__device__ __forceinline__ void run_tile(const PhaseArgs& a, int phase, int tile, StgdSmem& sm) {
  switch (phase) {
    case PH_P1: phase_tile<DMODE, KMODE, TY, TPH, PH_P1>(a.p1, tile, sm); break;
    case PH_FROB: phase_tile<DMODE, KMODE, TY, TPH, PH_FROB>(a.frob, tile, sm); break;
    case PH_P2: phase_tile<DMODE, KMODE, TY, TPH, PH_P2>(a.p2, tile, sm); break;
    case PH_GRAM: phase_tile<DMODE, KMODE, TY, TPH, PH_GRAM>(a.gram, tile, sm); break;
    case PH_UPDATE: phase_tile<DMODE, KMODE, TY, TPH, PH_UPDATE>(a.update, tile, sm); break;
    case PH_QPOLY: phase_tile<DMODE, KMODE, TY, TPH, PH_QPOLY>(a.qpoly, tile, sm); break;
    default: phase_tile<DMODE, KMODE, TY, TPH, PH_COPY>(a.copy, tile, sm); break;
  }
}

// The end test of the reference's STGD loop after step t (sgd_iter, 0-based) with log value f
// (stpm.c:747-765): converged, or past the cap.
__device__ inline bool stop_test(const StopArgs& a, int64_t t, double f) {
  return (a.iter_min > 0 && f < a.thresh && t > a.iter_min) || (a.iter_max > 0 && t > a.iter_max);
}

// One phase of one step, one kernel per phase (each with its own register allocation):
// blockIdx.x = tile. (An XCD-aware order that gave each XCD a compact group of tiles cut the HBM
// fetches of P1 from 24 to 9 MiB per launch, but the step took 2.6 % longer: the waves of a group
// then request the same lines at the same moment.) At b = 1024 a phase is bound by latency, not by its products:
// with the products taken out, UPDATE kept 6.8 of its 9.2 us at k = 500 (P1 5.6 of 10.4, P2 4.6 of 8.9, GRAM 4.0
// of 6.3) -- argument and guard loads that came back one after another, sums through LDS shuffles ahead of the stores.
// Arguments resolved on the host, independent loads and sums in registers after the stores took a step at k = 500 from
// 55 to 48 us (UPDATE 9.2 -> 6.5) and at k = 100 in FP32 from 45 to 39; loads that stay in flight past the next group's
// MFMAs (pipelined) and P2's smaller FP32 tiles took it on to 44 and 28.
// With the end test on (STOP), every phase of step g = base + st first checks whether the loop
// has ended; P1 of each step but a run's first forms the previous step's log entry in every wave
// (its kernels have finished), workgroup 0 stores it, and every workgroup applies the test to it and
// marks the end -- each reaches the same decision from the same bits, so the whole launch returns
// together. P1 returns early only when an earlier step ended the loop (stop_at < g): stop_at == g
// was set by a sibling workgroup, and workgroup 0 must still store the entry. The skipped kernels
// write nothing, and the host reads stop_at after the run.
template <int DMODE, int KMODE, typename TY, typename TPH, int PHASE, bool STOP>
__global__ __launch_bounds__(kThreads, PHASE == PH_P1 ? 3 : 1) void stgd_phase_kernel(typename ArgsOf<PHASE>::type a, StopArgs s) {
  __shared__ StgdSmem sm;
  if constexpr (STOP && PHASE != PH_SETUP) {
    const int64_t g = s.stop->base + s.st;
    const int64_t sa = s.stop->stop_at;
    if (sa < g || (PHASE != PH_P1 && sa == g)) return;  // an earlier step ended the loop (checked
                                                         // first: the log of a skipped step is never written)
    if constexpr (PHASE == PH_P1) {
      if (a.frob_prev) {
        const int ntk = a.kp / 32;
        const double f = frob_sum(a.fpart, ntk * ntk);
        if (blockIdx.x == 0 && threadIdx.x == 0) *a.frob_prev = f;
        if (stop_test(s, g - 1, f)) {
          if (threadIdx.x == 0) s.stop->stop_at = g;
          return;
        }
      }
    }
  }
  phase_tile<DMODE, KMODE, TY, TPH, PHASE>(a, blockIdx.x, sm, !STOP);
}

// ---- whole runs of a small instance in one workgroup ---------------------------------------------------
// With k <= 32 every k x k matrix is one 32 x 32 block, and a step of the phase kernels is six dependent launches of
// a few workgroups each, 25-30 us of launch and memory latency around about 1 us of work. Here one workgroup of
// eight waves runs all steps of a launch with Phi and the matrices derived from it in LDS and four barriers per
// step; the sums are those of the phase kernels, term by term (MFMA over the same k order, partial sums over the
// same halves of the minibatch, the epilogues' butterflies), so Phi and the log are bit-identical. Products with
// the zero padding beyond k are left out (they add exact zeros).
//   waves 0..3  P_A, P_B and C_g of the minibatch's 32-row tiles (tiles w, w + 4, ..); then, each for eight rows,
//               Phi~ from the summed products
//   wave 4      (Phi^T Phi)^o2 and Phi H; then the Newton-Schulz iterations alone, without barriers
//   waves 5, 6  Y_C^T C_g over the two halves of the minibatch
//   wave 7      c_mu; the log entry of the previous step
// The rows of Y of the next step are loaded during the Newton-Schulz iterations. One compute unit bounds the
// minibatch: at b = 512 a step takes 8.7 us in BF16 and 16.1 in FP32 (k = 32; the phase kernels 23.0 and 24.3), beyond it
// (and beyond the LDS that holds C_g) the phase kernels spread the work. At b = 100: 7.2 us in FP32 (k = 20) and 5.9 in
// BF16 (k = 10), the phase kernels 23.2 and 22.5. FP32 at k <= 16 goes to stgd_small16_kernel.
constexpr int kSmallB = 512;        // largest padded minibatch
constexpr int kSmallThreads = 512;

struct SmallArgs {
  const void *ya, *yb, *yct;        // all rows of X
  const double *mu_a, *mu_b, *mu_c;
  float *phi0, *phi1;               // Phi on entry in phi0; on exit there after an even number of steps, else in phi1
  double* frob;                     // [nsteps]
  StgdSmallCtl* ctl;
  int64_t step0, nsteps, spe, n_x, n_pad;
  int32_t k, kp, b, bl, ns_iters, quintic, renorm_every;
  float c3, c1, c0, eta, theta;
};

// A 32 x 32 operand in LDS: rows along the reduction index, FP32 or a split BF16 pair. The row strides put the 16-byte
// pieces of 16 consecutive rows on distinct banks.
template <int MODE>
struct SmallMat {
  float v[32][36];
};
template <>
struct SmallMat<MM_BF16X3> {
  __bf16 hi[32][40];
  __bf16 lo[32][40];
};

__device__ inline void small_put(SmallMat<MM_F32>& m, int r, int c, float x) { m.v[r][c] = x; }
__device__ inline void small_put(SmallMat<MM_BF16X3>& m, int r, int c, float x) {
#pragma clang fp contract(off)  // lo is of the rounded x, also where x is a product
  const __bf16 hi = (__bf16)x;
  m.hi[r][c] = hi;
  m.lo[r][c] = (__bf16)(x - (float)hi);
}
__device__ inline void small_put4(SmallMat<MM_F32>& m, int r, int c, const float x[4]) {
  *reinterpret_cast<float4*>(&m.v[r][c]) = make_float4(x[0], x[1], x[2], x[3]);
}
__device__ inline void small_put4(SmallMat<MM_BF16X3>& m, int r, int c, const float x[4]) {
#pragma clang fp contract(off)
  bf16x4 hi, lo;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    hi[e] = (__bf16)x[e];
    lo[e] = (__bf16)(x[e] - (float)hi[e]);
  }
  *reinterpret_cast<bf16x4*>(&m.hi[r][c]) = hi;
  *reinterpret_cast<bf16x4*>(&m.lo[r][c]) = lo;
}

// A product of an operand with itself, from accumulator layout, as an operand of its rows. In FP32 it is symmetric to
// the bit, so a lane stores its column as a row, four values at a time; the split form takes hi.lo before lo.hi
// and is not.
template <int MODE>
__device__ inline void small_put_sym(SmallMat<MODE>& m, const float v[16]) {
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if constexpr (MODE == MM_F32) {
      small_put4(m, c, 8 * q + 4 * h, v + 4 * q);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) small_put(m, 8 * q + 4 * h + e, c, v[4 * q + e]);
    }
  }
}

// The fragments of a 32 x 32 operand in MFMA layout: all LDS reads go out before the products that use them.
template <int MODE>
struct SmallFrag;
template <>
struct SmallFrag<MM_F32> {
  floatx4 v[4];
  __device__ inline void load(const SmallMat<MM_F32>& m) {
    const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
#pragma unroll
    for (int c = 0; c < 4; ++c) v[c] = *reinterpret_cast<const floatx4*>(&m.v[r][8 * c + 4 * h]);
  }
};
template <>
struct SmallFrag<MM_BF16X3> {
  bf16x8 hi[2], lo[2];
  __device__ inline void load(const SmallMat<MM_BF16X3>& m) {
    const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      hi[c] = *reinterpret_cast<const bf16x8*>(&m.hi[r][16 * c + 8 * h]);
      lo[c] = *reinterpret_cast<const bf16x8*>(&m.lo[r][16 * c + 8 * h]);
    }
  }
};

// A B^T over the first k columns of two operands; +0 added as the phase kernels' sums over empty parts do.
__device__ inline floatx16 small_mm(const SmallFrag<MM_F32>& A, const SmallFrag<MM_F32>& B, int k) {
  floatx16 acc = {};
#pragma unroll
  for (int c = 0; c < 4; ++c)
    if (8 * c < k) {
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(A.v[c][e], B.v[c][e], acc, 0, 0, 0);
    }
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] += 0.f;
  return acc;
}
__device__ inline floatx16 small_mm(const SmallFrag<MM_BF16X3>& A, const SmallFrag<MM_BF16X3>& B, int k) {
  floatx16 acc = {};
#pragma unroll
  for (int c = 0; c < 2; ++c)
    if (16 * c < k) {
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A.hi[c], B.hi[c], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A.hi[c], B.lo[c], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A.lo[c], B.hi[c], acc, 0, 0, 0);
    }
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] += 0.f;
  return acc;
}

// pa += (a block of 32 data rows in MFMA layout) Phi and pb likewise, over the first k columns.
__device__ inline void small_data_mm(floatx16& pa, floatx16& pb, const u32x4 xa[4], const u32x4 xb[4],
                                     const SmallFrag<MM_F32>& B, int k) {
#pragma unroll
  for (int c = 0; c < 4; ++c)
    if (8 * c < k) {
      const floatx4 x = as_f32(xa[c]), z = as_f32(xb[c]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        pa = __builtin_amdgcn_mfma_f32_32x32x2f32(x[e], B.v[c][e], pa, 0, 0, 0);
        pb = __builtin_amdgcn_mfma_f32_32x32x2f32(z[e], B.v[c][e], pb, 0, 0, 0);
      }
    }
}
__device__ inline void small_data_mm(floatx16& pa, floatx16& pb, const u32x4 xa[4], const u32x4 xb[4],
                                     const SmallFrag<MM_BF16X3>& B, int k) {
#pragma unroll
  for (int c = 0; c < 2; ++c)
    if (16 * c < k) {
      pa = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16(xa[c]), B.hi[c], pa, 0, 0, 0);
      pb = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16(xb[c]), B.hi[c], pb, 0, 0, 0);
    }
}

// acc += (a block of Y_C^T in MFMA layout) C_g over the group's first n columns x (rows of the minibatch; C_g is zero
// beyond them); cg points at the group's first column of C_g^T, row stride ld.
__device__ inline void small_cg_mm(floatx16& acc, const u32x4 a[4], const float* cg, int ld, int n) {
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  floatx4 y[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) y[c] = *reinterpret_cast<const floatx4*>(cg + r * ld + 8 * c + 4 * h);
#pragma unroll
  for (int c = 0; c < 4; ++c)
    if (8 * c < n) {
      const floatx4 x = as_f32(a[c]);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[e], y[c][e], acc, 0, 0, 0);
    }
}
__device__ inline void small_cg_mm(floatx16& acc, const u32x4 a[4], const __bf16* cg, int ld, int n) {
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  bf16x8 y[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) y[c] = *reinterpret_cast<const bf16x8*>(cg + r * ld + 16 * c + 8 * h);
#pragma unroll
  for (int c = 0; c < 4; ++c)
    if (16 * c < n) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16(a[c]), y[c], acc, 0, 0, 0);
}

template <int MODE>
struct SmallShm {
  SmallMat<MODE> phiT, H, xT, g, q;
  SmallMat<MODE> phis, xs;   // split runs: Phi and the Newton-Schulz iterate as operands (FP32 runs use the copies below)
  float phif[2][32][36];     // Phi in FP32, this step's and the next
  float xf[32][36];          // the Newton-Schulz iterate in FP32
  __device__ inline const SmallMat<MODE>& phi_op(int cur) const {
    if constexpr (MODE == MM_F32) return *reinterpret_cast<const SmallMat<MODE>*>(&phif[cur]);
    else return phis;
  }
  __device__ inline const SmallMat<MODE>& x_op() const {
    if constexpr (MODE == MM_F32) return *reinterpret_cast<const SmallMat<MODE>*>(&xf);
    else return xs;
  }
  float slot[3][16][64];     // Phi H and the halves of Y_C^T C_g, in accumulator layout
  float cs[kSmallB / 32][32];
  alignas(16) float mu[2][32];  // mu_A, mu_B
  float mv[2][32];           // m_A, m_B
  float cmu[32];
  int stop;
  alignas(16) u32x4 stage[8][256];       // per-wave transpose buffers
  typedef typename std::conditional<MODE == MM_F32, float, __bf16>::type T;
  alignas(16) T cgt[1];      // [32][b + 16 bytes]
};

template <int MODE>
static size_t small_shm_bytes(int b) {
  typedef typename SmallShm<MODE>::T T;
  return sizeof(SmallShm<MODE>) + sizeof(T) * 32 * (size_t)(b + 16 / sizeof(T));
}

// The new Phi as the wave that holds it in accumulator layout (v[i] = element (8 (i / 4) + 4 h + i % 4, lane % 32)):
// its operands, FP32 copy and the sums m_s = mu_s^T Phi (rows in pairs, fours and eights, then the four groups of
// eight, as finish_tile takes them).
template <int MODE>
__device__ inline void small_new_phi(SmallShm<MODE>& S, int buf, const float v[16]) {
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  float ma[4], mb[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float* x = v + 4 * q;
    small_put4(S.phiT, c, 8 * q + 4 * h, x);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (MODE != MM_F32) small_put(S.phis, 8 * q + 4 * h + e, c, x[e]);
      S.phif[buf][8 * q + 4 * h + e][c] = x[e];
    }
    const floatx4 u = *reinterpret_cast<const floatx4*>(&S.mu[0][8 * q + 4 * h]);
    const floatx4 w = *reinterpret_cast<const floatx4*>(&S.mu[1][8 * q + 4 * h]);
    float sa, sb;
    {
#pragma clang fp contract(off)
      sa = fmaf(u[0], x[0], u[1] * x[1]) + fmaf(u[2], x[2], u[3] * x[3]);
      sb = fmaf(w[0], x[0], w[1] * x[1]) + fmaf(w[2], x[2], w[3] * x[3]);
    }
    ma[q] = swap_add32(sa, sa);
    mb[q] = swap_add32(sb, sb);
  }
  if (h == 0) {
    S.mv[0][c] = (ma[0] + ma[1]) + (ma[2] + ma[3]) + 0.f;
    S.mv[1][c] = (mb[0] + mb[1]) + (mb[2] + mb[3]) + 0.f;
  }
}

// Clears the buffer of the next Phi ([64 x 64]) outside the T x T block that the run writes: the phase kernels and batches
// that go on from it take all of it, and a diverged run may have left anything there. (The current Phi's is clean:
// whatever leaves a Phi writes or has cleared the whole buffer.) Done while the first loads are on their way: 0.2 us
// of a run's 16-21 for one step. As part of the stores at a run's end it cost 1-2 % of every step (registers of the loop).
constexpr int kSmallKp = 64;
template <int T>
__device__ inline void small_clear(const SmallArgs& a) {
  for (int e = threadIdx.x; e < kSmallKp * kSmallKp / 4; e += blockDim.x)
    if (e / (kSmallKp / 4) >= T || e % (kSmallKp / 4) * 4 >= T) reinterpret_cast<float4*>(a.phi1)[e] = make_float4(0.f, 0.f, 0.f, 0.f);
}

template <int MODE, typename TY>
__global__ __launch_bounds__(kSmallThreads, 1) void stgd_small_kernel(SmallArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char small_raw[];
  SmallShm<MODE>& S = *reinterpret_cast<SmallShm<MODE>*>(small_raw);
  typedef typename SmallShm<MODE>::T T;
  constexpr int G = MODE == MM_F32 ? 32 : 64;  // minibatch rows of one Y_C^T group
  constexpr int PF = 4;                        // groups in flight per wave
  const int w = wave_id(), lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  const int kp = a.kp, b = a.b, k = a.k, nt = b / 32, ldc = b + 16 / (int)sizeof(T);
  const TY* ya = static_cast<const TY*>(a.ya);
  const TY* yb = static_cast<const TY*>(a.yb);
  const TY* yct = static_cast<const TY*>(a.yct);
  u32x4* stage = S.stage[w];
  T* cgt = S.cgt;

  int64_t pos = a.step0 % a.spe;               // place of the step in its epoch and in its renormalisation period
  int rn = a.renorm_every > 0 ? (int)(a.step0 % a.renorm_every) : 0;
  u32x4 pre[PF][4];                            // rows ahead: two tiles of Y_A, Y_B (waves 0..3), PF groups of Y_C^T
  u32x4 (&ra)[4] = pre[0], (&rb)[4] = pre[1];
  const int part = w - 5, ng = b / G;          // waves 5, 6: groups [g0, g1)
  const int g0 = w >= 5 ? ng * part / 2 : 0, g1 = w >= 5 ? ng * (part + 1) / 2 : 0;
  auto load_tile = [&](int64_t row0, int tile) {
    stage_load<true>(ra, ya + (row0 + 32 * tile) * kp, kp);
    stage_load<true>(rb, yb + (row0 + 32 * tile) * kp, kp);
  };
  auto load_group = [&](u32x4 (&y)[4], int64_t row0, int g) {
    const TY* p = yct + row0 + (int64_t)g * G;
    if (row0 % (16 / (int64_t)sizeof(TY)) == 0) stage_load<true>(y, p, a.n_pad);
    else stage_load<false>(y, p, a.n_pad);
  };
  auto prefetch = [&](int64_t row0) {
    if (w < 4) {
      if (w < nt) load_tile(row0, w);
    } else if (w == 5 || w == 6) {
#pragma unroll
      for (int u = 0; u < PF; ++u)
        if (g0 + u < g1) load_group(pre[u], row0, g0 + u);
    }
  };

  // log entry of step st: Phi in buffer `now` against the other, summed as the four waves of finish_tile do (rows 8 q ..,
  // four columns per lane)
  auto log_entry = [&](int64_t st, int now) {
    double f[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = 8 * q + (lane >> 3), c4 = 4 * (lane & 7);
      double d = 0.0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const double dd = (double)S.phif[now][r][c4 + e] - (double)S.phif[now ^ 1][r][c4 + e];
        d = fma(dd, dd, d);
      }
      f[q] = wave_sum(d);
    }
    if (lane == 0) a.frob[st] = (f[0] + f[1]) + (f[2] + f[3]);
  };

  float uc[4];                                 // waves 0..3: mu_C of their rows
  if (w < 4)
#pragma unroll
    for (int e = 0; e < 4; ++e) uc[e] = (float)a.mu_c[8 * w + 4 * h + e];
  if (w == 4) {
    S.mu[h][c] = (float)(h ? a.mu_b[c] : a.mu_a[c]);
    asm volatile("" ::: "memory");
    float v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = a.phi0[(8 * (i >> 2) + 4 * h + (i & 3)) * kp + c];
    small_new_phi<MODE>(S, 0, v);
  }
  prefetch(pos * a.bl);
  small_clear<32>(a);
  __syncthreads();

  int cur = 0;
  int64_t st = 0;
  while (true) {
    const int64_t row0 = pos * a.bl;
    const int nb = (int)min((int64_t)a.bl, a.n_x - row0);
    if (++pos == a.spe) pos = 0;
    const bool renorm = a.renorm_every > 0 && ++rn == a.renorm_every;
    if (renorm) rn = 0;
    const bool poll = pos == 0 && st + 1 < a.nsteps;  // an epoch ends here with more to come
    int stop = 0;
    if (poll && w == 7) stop = __hip_atomic_load(&a.ctl->stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    // P_A, P_B, C_g; (Phi^T Phi)^o2; the previous step's log entry
    if (w < 4) {
      const float mA = S.mv[0][c], mB = S.mv[1][c];
      SmallFrag<MODE> phi;
      phi.load(S.phiT);
      for (int tile = w; tile < nt; tile += 4) {
        u32x4 xa[4], xb[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          xa[i] = ra[i];
          xb[i] = rb[i];
        }
        if (tile + 4 < nt) load_tile(row0, tile + 4);
        stage_swap(xa, stage);
        stage_swap(xb, stage);
        floatx16 pa = {}, pb = {};
        small_data_mm(pa, pb, xa, xb, phi, k);
        float t[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float cg[4], cs = 0.f;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int x = 32 * tile + 8 * q + 4 * h + e;
            const float p = pa[4 * q + e] + 0.f, r = pb[4 * q + e] + 0.f;
            const bool valid = x < nb;
            const float ab = p * r;
            {
#pragma clang fp contract(off)
              cs += valid ? ab : 0.f;
            }
            cg[e] = valid ? cg_value(a.c3, a.c1, p, r, ab, mA, mB) : 0.f;
          }
          store4(cgt + c * ldc + 32 * tile + 8 * q + 4 * h, cg);
          t[q] = swap_add32(cs, cs);
        }
        if (h == 0) S.cs[tile][c] = (t[0] + t[1]) + (t[2] + t[3]);
      }
    } else if (w == 4) {
      SmallFrag<MODE> phi;
      phi.load(S.phiT);
      const floatx16 g = small_mm(phi, phi, k);
      float v[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = g[i] * g[i];
      small_put_sym<MODE>(S.H, v);
    } else if (w == 5 || w == 6) {  // Y_C^T into MFMA layout ahead of C_g
#pragma unroll
      for (int u = 0; u < PF; ++u)
        if (g0 + u < g1) stage_swap(pre[u], stage);
    } else if (st > 0) {
      log_entry(st - 1, cur);
    }
    __syncthreads();
    // Phi H, the halves of Y_C^T C_g, c_mu
    if (w == 4) {
      SmallFrag<MODE> phi, hh;
      phi.load(S.phi_op(cur));
      hh.load(S.H);
      const floatx16 v = small_mm(phi, hh, k);
#pragma unroll
      for (int i = 0; i < 16; ++i) S.slot[0][i][lane] = v[i];
    } else if (w == 5 || w == 6) {
      floatx16 acc = {};
      for (int g = g0; g < g1; g += PF) {
#pragma unroll
        for (int u = 0; u < PF; ++u) {
          if (g + u < g1) {
            if (g > g0) stage_swap(pre[u], stage);
            small_cg_mm(acc, pre[u], cgt + (g + u) * G, ldc, nb - (g + u) * G);
            if (g + u + PF < g1) load_group(pre[u], row0, g + u + PF);
          }
        }
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) S.slot[w - 4][i][lane] = acc[i];
    } else if (w == 7) {
      float m[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const float v0 = q < nt ? S.cs[q][c] : 0.f, v1 = q + 8 < nt ? S.cs[q + 8][c] : 0.f;
        m[q] = v0 + v1;
      }
      const float ssum = ((m[0] + m[1]) + (m[2] + m[3])) + ((m[4] + m[5]) + (m[6] + m[7]));
      if (h == 0) S.cmu[c] = cmu_value(a.c0, a.c1, S.mv[0][c], S.mv[1][c], ssum, nb);
    }
    __syncthreads();
    // Phi~
    if (w < 4) {
      const float inv_b = 1.f / (float)nb, cmu = S.cmu[c];
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = 8 * w + 4 * h + e;
        const float phh = S.slot[0][4 * w + e][lane], t = S.slot[1][4 * w + e][lane] + S.slot[2][4 * w + e][lane];
        v[e] = step_value(S.phif[cur][r][c], a.eta, a.theta, phh, t, inv_b, uc[e], cmu);
        if constexpr (MODE != MM_F32) small_put(S.xs, r, c, v[e]);
        S.xf[r][c] = v[e];
      }
      small_put4(S.xT, c, 8 * w + 4 * h, v);
    }
    __syncthreads();
    // the renormalisation (wave 4) under the next step's loads
    if (st + 1 < a.nsteps) prefetch(pos * a.bl);
    if (poll && w == 7 && lane == 0) S.stop = stop;
    if (w == 4) {
      float x[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) x[i] = S.xf[8 * (i >> 2) + 4 * h + (i & 3)][c];
      const int its = renorm ? a.ns_iters : 0;
      for (int it = 0; it < its; ++it) {
        SmallFrag<MODE> fa, fb;
        fa.load(S.xT);
        const floatx16 g = small_mm(fa, fa, k);
        fa.load(S.x_op());
        float gv[16], rs;  // rs: a row sum of |G| (every row on some lane), four columns at a time
#pragma unroll
        for (int i = 0; i < 16; ++i) gv[i] = g[i];
        small_put_sym<MODE>(S.g, gv);
        if constexpr (MODE == MM_F32) {  // lane c's column is row c
          float t[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            float s = 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) s += fabsf(gv[4 * q + e]);
            t[q] = swap_add32(s, s);
          }
          rs = (t[0] + t[1]) + (t[2] + t[3]);
        } else {                         // through LDS: lane 2 r + i takes half a row
#pragma unroll
          for (int i = 0; i < 16; ++i) S.xf[8 * (i >> 2) + 4 * h + (i & 3)][c] = gv[i];
          asm volatile("" ::: "memory");
          float t[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const float4 x = *reinterpret_cast<const float4*>(&S.xf[lane >> 1][16 * (lane & 1) + 4 * q]);
            t[q] = ((fabsf(x.x) + fabsf(x.y)) + fabsf(x.z)) + fabsf(x.w);
          }
          rs = (t[0] + t[1]) + (t[2] + t[3]);
          rs += dpp_mov<kDppXor1>(rs);
        }
        // the largest row sum, clamped as fix32 does; above 2, where the guard acts, its fixed point is exact
        const float cs = guard_value(wave_max(fminf(rs, 1073741824.f)));
        asm volatile("" ::: "memory");
        fb.load(S.g);
        if (a.quintic) {
          const floatx16 gg = small_mm(fb, fb, k);
#pragma unroll
          for (int i = 0; i < 16; ++i) gv[i] = qpoly_value(cs, gv[i], gg[i]);
          small_put_sym<MODE>(S.q, gv);
          asm volatile("" ::: "memory");
          fb.load(S.q);
        }
        const floatx16 y = small_mm(fa, fb, k);
        asm volatile("" ::: "memory");
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] = update_value(cs, a.quintic, x[i], y[i]);
        if (it + 1 < its) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            small_put4(S.xT, c, 8 * q + 4 * h, x + 4 * q);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              if constexpr (MODE != MM_F32) small_put(S.xs, 8 * q + 4 * h + e, c, x[4 * q + e]);
              else S.xf[8 * q + 4 * h + e][c] = x[4 * q + e];
            }
          }
          asm volatile("" ::: "memory");
        }
      }
      small_new_phi<MODE>(S, cur ^ 1, x);
    }
    cur ^= 1;
    ++st;
    __syncthreads();
    if (st == a.nsteps || (poll && S.stop)) break;
  }
  if (w == 7) {
    log_entry(st - 1, cur);
    if (lane == 0) a.ctl->ran = st;
  }
  float* phi_out = cur ? a.phi1 : a.phi0;
  if (w < 4)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = 8 * w + 4 * h + e;
      phi_out[r * kp + c] = S.phif[cur][r][c];
    }
}

// ---- the same for k <= 16 in FP32: one 16 x 16 block -----------------------------------------------------
// Matrices live in registers in accumulator layout (lane l: rows 4 (l / 16) + i, column l % 16, i = 0 .. 3). Read as
// "row l % 16, columns 4 (l / 16) + i" the same registers are the transposed matrix as an MFMA operand, up to the
// exchange of half-waves that gives the k order of the 32 x 32 products (tile_frag). So one wave keeps Phi and Phi^T, each
// product with a symmetric matrix is taken for both (the same products in the same order, so each stays the exact
// transpose of the other), and a Newton-Schulz iteration is three short MFMA chains with nothing through LDS. Y_A, Y_B
// and Y_C^T are loaded in operand layout by the same reading. A step at k = 10, b = 100 takes 3.0 us against 6.5 in the
// 32-wide kernel, whose chains are four times as long and pass every matrix through LDS; what is left is latency, about
// 1000 cycles each of P_A, P_B, of Y_C^T C_g and of an iteration. Twelve waves: eight for P_A, P_B, C_g in units of 16
// rows, one that owns Phi, two for the halves of Y_C^T C_g, one for c_mu and the log (with four, two and the owner, the
// log ahead of the first barrier: 3.3 us).
struct Small16Shm {
  floatx4 phi[64];           // Phi in accumulator layout
  float phif[3][16][20];     // Phi by rows: the previous step's, this one's and the next
  floatx4 t[2][64];          // halves of Y_C^T C_g in accumulator layout
  float tr[2][16][20];       // and by rows
  float cs[kSmallB / 16][16];
  float mv[2][16];           // m_A, m_B
  alignas(16) float cmu[16];
  int stop;
  alignas(16) float cgt[1];  // [16][b + 4]
};

static size_t small16_shm_bytes(int b) { return sizeof(Small16Shm) + sizeof(float) * 16 * (size_t)(b + 4); }

// The operand of four columns per lane group in the k order 0, 4, 1, 5 | 2, 6, 3, 7 | 8, 12, ..: f[0 .. 1] of the first
// eight columns, f[2 .. 3] of the others.
__device__ inline floatx4 tile_frag(const floatx4& v) {
  float a0 = v[0], b0 = v[1], a1 = v[2], b1 = v[3];
  half_swap(a0, b0);
  half_swap(a1, b1);
  return floatx4{a0, a1, b0, b1};
}

__device__ inline void tile_mma(floatx4& acc, const floatx4& a, const floatx4& b) {
#pragma unroll
  for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], acc, 0, 0, 0);
}

__device__ inline floatx4 tile_mm(const floatx4& a, const floatx4& b) {
  floatx4 acc = {};
  tile_mma(acc, a, b);
  return acc + 0.f;
}

constexpr int kSmall16Threads = 768;

__global__ __launch_bounds__(kSmall16Threads, 1) void stgd_small16_kernel(SmallArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char small_raw[];
  Small16Shm& S = *reinterpret_cast<Small16Shm*>(small_raw);
  constexpr int P1W = 8, OWNER = 8, P2A = 9, P2B = 10, AUX = 11;  // roles of the waves
  constexpr int PF = 4;                                          // P2: groups of 32 minibatch rows loaded ahead
  small_clear<16>(a);
  const int w = wave_id(), lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int kp = a.kp, b = a.b, nt = b / 32, nu = b / 16, ldc = b + 4;
  const float* ya = static_cast<const float*>(a.ya);
  const float* yb = static_cast<const float*>(a.yb);
  const float* yct = static_cast<const float*>(a.yct);
  float* cgt = S.cgt;

  int64_t pos = a.step0 % a.spe;
  int rn = a.renorm_every > 0 ? (int)(a.step0 % a.renorm_every) : 0;
  const bool p2w = w == P2A || w == P2B;
  const int g0 = w == P2B ? nt / 2 : 0, ng = nt / 2;  // P2: groups [g0, g0 + ng)
  floatx4 ra, rb;         // P1: the next 16 rows of Y_A, Y_B
  floatx4 yc[PF][2];      // P2: Y_C^T of the groups
  auto load_rows = [&](int64_t row0, int u) {
    const int64_t at = (row0 + 16 * u + c) * kp + 4 * g;
    ra = *reinterpret_cast<const floatx4*>(ya + at);
    rb = *reinterpret_cast<const floatx4*>(yb + at);
  };
  auto load_groups = [&](int64_t row0, int u0) {  // groups u0 .. u0 + PF - 1 of this wave
    const float* p = yct + c * a.n_pad + row0 + 32 * (g0 + u0) + 4 * g;
    auto load = [&](auto aligned) {
#pragma unroll
      for (int u = 0; u < PF; ++u)
        if (u0 + u < ng) {
          yc[u][0] = __builtin_bit_cast(floatx4, ld16<decltype(aligned)::value>(p + 32 * u));
          yc[u][1] = __builtin_bit_cast(floatx4, ld16<decltype(aligned)::value>(p + 32 * u + 16));
        }
    };
    if (row0 % 4 == 0) load(std::true_type());
    else load(std::false_type());
  };
  auto prefetch = [&](int64_t row0) {
    if (w < P1W) {
      if (w < nu) load_rows(row0, w);
    } else if (p2w) {
      load_groups(row0, 0);
    }
  };
  // as in the 32-wide kernel: the rows and columns from 16 on are zero
  auto log_entry = [&](int64_t st, int now, int before) {
    double f[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int r = 8 * q + (lane >> 3), c4 = 4 * (lane & 7);
      double d = 0.0;
      if (c4 < 16)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const double dd = (double)S.phif[now][r][c4 + e] - (double)S.phif[before][r][c4 + e];
          d = fma(dd, dd, d);
        }
      f[q] = wave_sum(d);
    }
    if (lane == 0) a.frob[st] = f[0] + f[1];
  };

  // OWNER: Phi and Phi^T in accumulator layout; mu_A, mu_B, mu_C of the rows 4 g + i and mu_C of row c
  floatx4 x = {}, xt = {}, ua = {}, ub = {}, uc = {};
  float uct = 0.f;
  auto new_phi = [&](int buf) {
    S.phi[lane] = x;
    *reinterpret_cast<floatx4*>(&S.phif[buf][c][4 * g]) = xt;
    float sa, sb;
    {
#pragma clang fp contract(off)
      sa = fmaf(ua[0], x[0], ua[1] * x[1]) + fmaf(ua[2], x[2], ua[3] * x[3]);
      sb = fmaf(ub[0], x[0], ub[1] * x[1]) + fmaf(ub[2], x[2], ub[3] * x[3]);
    }
    const float ma = swap_add16(sa, sa), mb = swap_add16(sb, sb);
    const float m = swap_add32(ma, mb) + 0.f;  // m_A in the lower half, m_B in the upper
    if ((g & 1) == 0) S.mv[g >> 1][c] = m;
  };
  if (w == OWNER) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[i] = a.phi0[(4 * g + i) * kp + c];
      xt[i] = a.phi0[c * kp + 4 * g + i];
      ua[i] = (float)a.mu_a[4 * g + i];
      ub[i] = (float)a.mu_b[4 * g + i];
      uc[i] = (float)a.mu_c[4 * g + i];
    }
    uct = (float)a.mu_c[c];
    new_phi(0);
  }
  prefetch(pos * a.bl);
  __syncthreads();

  int cur = 0;       // S.phif[cur] holds Phi, the buffer before it (of three) the previous one
  int64_t st = 0;
  while (true) {
    const int64_t row0 = pos * a.bl;
    const int nb = (int)min((int64_t)a.bl, a.n_x - row0);
    if (++pos == a.spe) pos = 0;
    const bool renorm = a.renorm_every > 0 && ++rn == a.renorm_every;
    if (renorm) rn = 0;
    const bool poll = pos == 0 && st + 1 < a.nsteps;
    int stop = 0;
    if (poll && w == AUX) stop = __hip_atomic_load(&a.ctl->stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    const float inv_b = 1.f / (float)nb;
    floatx4 ph = {}, pht = {};  // OWNER: Phi H and its transpose
    // P_A, P_B, C_g; Phi H
    if (w < P1W) {
      const float mA = S.mv[0][c], mB = S.mv[1][c];
      const floatx4 phi = tile_frag(S.phi[lane]);
      for (int u = w; u < nu; u += P1W) {
        const floatx4 xa = tile_frag(ra), xb = tile_frag(rb);
        if (u + P1W < nu) load_rows(row0, u + P1W);
        floatx4 pa = {}, pb = {};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          pa = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[e], phi[e], pa, 0, 0, 0);
          pb = __builtin_amdgcn_mfma_f32_16x16x4f32(xb[e], phi[e], pb, 0, 0, 0);
        }
        float cg[4], cs = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float p = pa[e] + 0.f, r = pb[e] + 0.f;
          const bool valid = 16 * u + 4 * g + e < nb;
          const float ab = p * r;
          {
#pragma clang fp contract(off)
            cs += valid ? ab : 0.f;
          }
          cg[e] = valid ? cg_value(a.c3, a.c1, p, r, ab, mA, mB) : 0.f;
        }
        store4(cgt + c * ldc + 16 * u + 4 * g, cg);
        const float t = swap_add16(cs, cs), v = swap_add32(t, t);
        if (g == 0) S.cs[u][c] = v;
      }
    } else if (w == OWNER) {
      const floatx4 f = tile_frag(x), ft = tile_frag(xt);
      const floatx4 gr = tile_mm(f, f);
      const floatx4 fh = tile_frag(gr * gr);
      ph = tile_mm(ft, fh);
      pht = tile_mm(fh, ft);
    } else if (p2w) {
#pragma unroll
      for (int u = 0; u < PF; ++u)
        if (u < ng)
#pragma unroll
          for (int h = 0; h < 2; ++h) yc[u][h] = tile_frag(yc[u][h]);
    }
    __syncthreads();
    // the halves of Y_C^T C_g, c_mu
    if (p2w) {
      floatx4 acc = {};
      const float* p = cgt + c * ldc + 32 * g0 + 4 * g;
      for (int u0 = 0; u0 < ng; u0 += PF) {
        if (u0 > 0) load_groups(row0, u0);
        floatx4 y[PF][2];
#pragma unroll
        for (int u = 0; u < PF; ++u) {
          const float* q = p + 32 * min(u0 + u, ng - 1);
          y[u][0] = *reinterpret_cast<const floatx4*>(q);
          y[u][1] = *reinterpret_cast<const floatx4*>(q + 16);
        }
#pragma unroll
        for (int u = 0; u < PF; ++u)
          if (u0 + u < ng)
#pragma unroll
            for (int h = 0; h < 2; ++h) tile_mma(acc, u0 > 0 ? tile_frag(yc[u][h]) : yc[u][h], tile_frag(y[u][h]));
      }
      S.t[w - P2A][lane] = acc;
#pragma unroll
      for (int i = 0; i < 4; ++i) S.tr[w - P2A][4 * g + i][c] = acc[i];
    } else if (w == AUX) {
      float m[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const float v0 = q < nt ? S.cs[2 * q][c] + S.cs[2 * q + 1][c] : 0.f;
        const float v1 = q + 8 < nt ? S.cs[2 * q + 16][c] + S.cs[2 * q + 17][c] : 0.f;
        m[q] = v0 + v1;
      }
      const float ssum = ((m[0] + m[1]) + (m[2] + m[3])) + ((m[4] + m[5]) + (m[6] + m[7]));
      if (g == 0) S.cmu[c] = cmu_value(a.c0, a.c1, S.mv[0][c], S.mv[1][c], ssum, nb);
    }
    __syncthreads();
    // Phi~ and the renormalisation (OWNER) under the next step's loads and the previous step's log entry
    const int next = cur == 2 ? 0 : cur + 1;
    if (w != OWNER) {
      if (st + 1 < a.nsteps) prefetch(pos * a.bl);
      if (w == AUX) {
        if (poll && lane == 0) S.stop = stop;
        if (st > 0) log_entry(st - 1, cur, cur == 0 ? 2 : cur - 1);
      }
    } else {
      const float cmu = S.cmu[c];
      const floatx4 cmut = *reinterpret_cast<const floatx4*>(&S.cmu[4 * g]);
      const floatx4 t0 = S.t[0][lane], t1 = S.t[1][lane];
      const floatx4 r0 = *reinterpret_cast<const floatx4*>(&S.tr[0][c][4 * g]);
      const floatx4 r1 = *reinterpret_cast<const floatx4*>(&S.tr[1][c][4 * g]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[i] = step_value(x[i], a.eta, a.theta, ph[i], t0[i] + t1[i], inv_b, uc[i], cmu);
        xt[i] = step_value(xt[i], a.eta, a.theta, pht[i], r0[i] + r1[i], inv_b, uct, cmut[i]);
      }
      const int its = renorm ? a.ns_iters : 0;
      for (int it = 0; it < its; ++it) {
        const floatx4 f = tile_frag(x), ft = tile_frag(xt);
        const floatx4 gr = tile_mm(f, f);
        floatx4 fg = tile_frag(gr);
        if (a.quintic) {
          const floatx4 gg = tile_mm(fg, fg);
          float s = 0.f;
#pragma unroll
          for (int e = 0; e < 4; ++e) s += fabsf(gr[e]);
          const float t = swap_add16(s, s);
          const float cs = guard_value(wave_max(fminf(swap_add32(t, t), 1073741824.f)));
          floatx4 q;
#pragma unroll
          for (int i = 0; i < 4; ++i) q[i] = qpoly_value(cs, gr[i], gg[i]);
          fg = tile_frag(q);
          const floatx4 y = tile_mm(ft, fg), yt = tile_mm(fg, ft);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            x[i] = update_value(cs, true, x[i], y[i]);
            xt[i] = update_value(cs, true, xt[i], yt[i]);
          }
        } else {
          const floatx4 y = tile_mm(ft, fg), yt = tile_mm(fg, ft);
          float s = 0.f;
#pragma unroll
          for (int e = 0; e < 4; ++e) s += fabsf(gr[e]);
          const float t = swap_add16(s, s);
          const float cs = guard_value(wave_max(fminf(swap_add32(t, t), 1073741824.f)));
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            x[i] = update_value(cs, false, x[i], y[i]);
            xt[i] = update_value(cs, false, xt[i], yt[i]);
          }
        }
      }
      new_phi(next);
    }
    cur = next;
    ++st;
    __syncthreads();
    if (st == a.nsteps || (poll && S.stop)) break;
  }
  if (w == AUX) {
    log_entry(st - 1, cur, cur == 0 ? 2 : cur - 1);
    if (lane == 0) a.ctl->ran = st;
  }
  float* phi_out = (st & 1) ? a.phi1 : a.phi0;
  if (w == OWNER)
#pragma unroll
    for (int i = 0; i < 4; ++i) phi_out[(4 * g + i) * kp + c] = x[i];
}

// ---- resolving the arguments (host) ------------------------------------------------------------------
// One instance's buffers and settings, as the plan of a run or of a batch holds them.
struct StepPlan {
  StgdArgs a;
  StgdBuffers B;
  const void *YA, *YB, *YCt;
  int32_t ns_iters, ns_degree;
  bool bf16;
  int64_t esz() const { return bf16 ? 2 : 4; }
  const void* op(const float* f32, const uint16_t* s16) const { return bf16 ? (const void*)s16 : (const void*)f32; }
  uint16_t* out16(uint16_t* p) const { return bf16 ? p : nullptr; }
  const void* at(const void* p, int64_t elems) const { return static_cast<const char*>(p) + elems * esz(); }

  // Newton-Schulz iteration `it` reads x, xT and writes dst, dstT: phit -> phia -> phit -> ...; the last
  // iteration writes phi[cur ^ 1] and phiT.
  struct Ns {
    float *x, *xT, *dst, *dstT;
    uint16_t *x16, *xT16, *dst16, *dstT16;
  };
  Ns ns(int cur, int it) const {
    Ns n;
    const bool from_t = (it & 1) == 0, last = it == ns_iters - 1;
    n.x = from_t ? B.phit : B.phia;
    n.xT = from_t ? B.phitT : B.phiaT;
    n.x16 = from_t ? B.phit16 : B.phia16;
    n.xT16 = from_t ? B.phitT16 : B.phiaT16;
    n.dst = last ? B.phi[cur ^ 1] : (from_t ? B.phia : B.phit);
    n.dstT = last ? B.phiT : (from_t ? B.phiaT : B.phitT);
    n.dst16 = last ? B.phi16[cur ^ 1] : (from_t ? B.phia16 : B.phit16);
    n.dstT16 = last ? B.phiT16 : (from_t ? B.phiaT16 : B.phitT16);
    return n;
  }

  // Arguments of `phase` (iteration `it` of a renormalisation) of a step that reads phi[cur] and the minibatch of nb
  // rows at row yrow0 of the Y buffers. log / log_prev: its and the previous step's log entries (log_prev null
  // for a run's first step); log0, nlog: all of the run's (SETUP).
  PhaseArgs resolve(int phase, int it, int cur, int64_t yrow0, int32_t nb, double* log, double* log_prev, double* log0,
                    int64_t nlog) const {
    PhaseArgs out;
    std::memset(static_cast<void*>(&out), 0, sizeof(out));
    const int kp = a.kp;
    switch (phase) {
      case PH_P1: {
        P1Args& p = out.p1;
        p.ya = at(YA, yrow0 * kp);
        p.yb = at(YB, yrow0 * kp);
        p.phiT = op(B.phiT, B.phiT16);
        p.mpart = B.mpart;
        p.cgt = B.cgt;
        p.cs_part = a.cs_part;
        p.mab = a.mab;
        p.h = B.h;
        p.h16 = out16(B.h16);
        p.frob_prev = log_prev;
        p.fpart = B.fpart;
        p.kp = kp;
        p.b = a.b;
        p.nb = nb;
        p.c3 = a.c3;
        p.c1 = a.c1;
        break;
      }
      case PH_P2:
      case PH_P2S: {
        P2Args& p = out.p2;
        p.phi_op = op(B.phi[cur], B.phi16[cur]);
        p.h_op = op(B.h, B.h16);
        p.phi = B.phi[cur];
        p.yct = at(YCt, yrow0);
        p.cgt = B.cgt;
        p.cs_part = a.cs_part;
        p.mab = a.mab;
        p.mu_c = a.mu_c;
        p.out = B.phit;
        p.out16 = out16(B.phit16);
        p.outT = B.phitT;
        p.outT16 = out16(B.phitT16);
        p.rowsum = B.rowsum;
        p.fpart = a.frob_pre ? B.fpart : nullptr;
        p.n_pad = a.n_pad;
        p.kp = kp;
        p.b = a.b;
        p.nb = nb;
        p.aligned = yrow0 % (16 / esz()) == 0;
        p.eta = a.eta;
        p.theta = a.theta;
        p.c0 = a.c0;
        p.c1 = a.c1;
        break;
      }
      case PH_GRAM: {
        const Ns n = ns(cur, it);
        out.gram = GramArgs{op(n.xT, n.xT16), B.gt, out16(B.gt16), B.rowsum + (it & 1) * kp, kp};
        break;
      }
      case PH_QPOLY:
        out.qpoly = QpolyArgs{op(B.gt, B.gt16), B.gt, B.q, out16(B.q16), B.rowsum + (it & 1) * kp, kp};
        break;
      case PH_UPDATE: {
        const Ns n = ns(cur, it);
        const bool last = it == ns_iters - 1, quintic = ns_degree == 5;
        UpdateArgs& p = out.update;
        p.x_op = op(n.x, n.x16);
        p.g_op = quintic ? op(B.q, B.q16) : op(B.gt, B.gt16);
        p.x = n.x;
        p.out = n.dst;
        p.out16 = out16(n.dst16);
        p.outT = n.dstT;
        p.outT16 = out16(n.dstT16);
        p.prev = last ? B.phi[cur] : nullptr;
        p.mu_a = a.mu_a;
        p.mu_b = a.mu_b;
        p.fpart = last ? B.fpart : nullptr;
        p.mpart = last ? B.mpart : nullptr;
        p.rowsum = B.rowsum + (it & 1) * kp;
        p.rowsum_next = B.rowsum + ((it + 1) & 1) * kp;
        p.kp = kp;
        p.quintic = quintic;
        break;
      }
      case PH_FROB:
        out.frob = FrobArgs{log, B.fpart, kp};
        break;
      default: {  // COPY, QRFIN, SETUP
        CopyArgs& p = out.copy;
        const bool setup = phase == PH_SETUP, qrfin = phase == PH_QRFIN;
        p.x = setup ? B.phi[cur] : (qrfin ? B.phia : B.phit);
        p.out = setup ? nullptr : B.phi[cur ^ 1];
        p.out16 = out16(B.phi16[setup ? cur : cur ^ 1]);
        p.outT = B.phiT;
        p.outT16 = out16(B.phiT16);
        p.prev = setup ? nullptr : B.phi[cur];
        p.mu_a = a.mu_a;
        p.mu_b = a.mu_b;
        p.fpart = setup || qrfin || a.frob_pre ? nullptr : B.fpart;
        p.mpart = B.mpart;
        p.frob_zero = setup ? log0 : nullptr;
        p.nfrob = nlog;
        p.kp = kp;
        p.kmax = qrfin ? a.k : kp;
        break;
      }
    }
    return out;
  }
};

// ---- many instances in one persistent launch -------------------------------------------------------
// The host lays the phases of every instance's steps out slot by slot: slot s holds the s-th phase
// segment of every instance that has one, so each segment's inputs were produced in an earlier
// slot. The cooperative grid walks the slots; in each, the workgroups share the slot's tiles
// (tile t of the slot goes to workgroup t mod grid), and a grid barrier separates consecutive
// slots. Every workgroup executes every barrier, and no workgroup waits on another except there.
struct BatchSeg {      // host only: the plan before it is laid out
  int32_t phase;
  int32_t ntiles;
  PhaseArgs args;
};

// The segment of slot segments [s0, s1) that holds slot tile t (the last with first <= t): the lanes compare 64
// segments at a time, one load deep. (A binary search walked its probes one load after another.)
__device__ inline int32_t find_seg(const int32_t* __restrict__ first, int32_t s0, int32_t s1, int32_t t) {
  const int lane = threadIdx.x & 63;
  int32_t n = 0;
  for (int32_t s = s0; s < s1; s += 64) {
    const bool le = first[min(s + lane, s1 - 1)] <= t && s + lane < s1;
    n += __popcll(__ballot(le));
  }
  return __builtin_amdgcn_readfirstlane(s0 + n - 1);
}

// The arguments are resolved on the host with the plan, one PhaseArgs per segment, and read here through
// a uniform reference into global memory, as the per-phase kernels read theirs from the kernel
// arguments: in scalar registers. (A context held in LDS is per-lane data to the compiler, which costs
// the scalar operand bases and doubles the register footprint; one built in registers goes to the
// stack, as it is indexed at run time. The tile functions are forced inline for the same reason: an
// out-of-line call passes the context as a per-lane pointer.)
template <int DMODE, int KMODE, typename TY, typename TPH>
__global__ __launch_bounds__(kThreads) void stgd_batch_kernel(const PhaseArgs* __restrict__ args, const int32_t* __restrict__ first,
                                                         const int32_t* __restrict__ phase, const int32_t* slot_seg,
                                                         const int64_t* slot_tiles, int32_t nslots) {
  cg::grid_group grid = cg::this_grid();
  __shared__ StgdSmem sm;
  for (int32_t sl = 0; sl < nslots; ++sl) {
    const int32_t s0 = slot_seg[sl], s1 = slot_seg[sl + 1];
    const int64_t ntiles = slot_tiles[sl];
    for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
      const int32_t sg = find_seg(first, s0, s1, (int32_t)t);
      run_tile<DMODE, KMODE, TY, TPH>(args[sg], phase[sg], (int)t - first[sg], sm);
      __syncthreads();
    }
    grid.sync();
  }
}

// One phase slot of the plan as its own launch (blockIdx.x = tile of the slot): the grouped
// alternative to the persistent kernel, where the kernel boundary orders consecutive slots.
template <int DMODE, int KMODE, typename TY, typename TPH>
__global__ __launch_bounds__(kThreads) void stgd_slot_kernel(const PhaseArgs* __restrict__ args, const int32_t* __restrict__ first,
                                                        const int32_t* __restrict__ phase, int32_t s0, int32_t s1) {
  __shared__ StgdSmem sm;
  const int32_t sg = find_seg(first, s0, s1, blockIdx.x);
  run_tile<DMODE, KMODE, TY, TPH>(args[sg], phase[sg], (int)blockIdx.x - first[sg], sm);
}

// A slot whose segments are all of one phase, launched with that phase's code only: the generic slot
// kernel holds every phase and gets the register budget of the largest (one wave per SIMD), this one
// that of its phase, as the per-phase kernels of single instances.
template <int DMODE, int KMODE, typename TY, typename TPH, int PHASE>
__global__ __launch_bounds__(kThreads) void stgd_slot_phase_kernel(const PhaseArgs* __restrict__ args, const int32_t* __restrict__ first,
                                                              int32_t s0, int32_t s1) {
  __shared__ StgdSmem sm;
  const int32_t sg = find_seg(first, s0, s1, blockIdx.x);
  phase_tile<DMODE, KMODE, TY, TPH, PHASE>(phase_args<PHASE>(args[sg]), (int)blockIdx.x - first[sg], sm);
}

__global__ void set_i64_kernel(int64_t* p, int64_t v) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *p = v;
}

int stgd_set_i64(hipStream_t s, int64_t* p, int64_t v) {
  hipLaunchKernelGGL(set_i64_kernel, dim3(1), dim3(64), 0, s, p, v);
  MMSB_LAUNCH_CHECK();
  return MMSB_OK;
}

__global__ void f32_to_bf16_kernel(int64_t n, const float* __restrict__ in, __bf16* __restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) out[t] = (__bf16)in[t];
}

int f32_to_bf16(hipStream_t s, int64_t n, const float* in, bf16_bits* out) {
  if (n <= 0) return MMSB_OK;
  hipLaunchKernelGGL(f32_to_bf16_kernel, dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, s, n, in,
                     reinterpret_cast<__bf16*>(out));
  MMSB_LAUNCH_CHECK();
  return MMSB_OK;
}

// ---- host driver -----------------------------------------------------------------------------------
static bool step_renorms(int64_t gstep, int32_t renorm_every, int32_t ns_iters) {
  return renorm_every > 0 && ((gstep + 1) % renorm_every == 0) && ns_iters > 0;
}

// Whether P2 of an FP32 instance takes 16 x 16 tiles (without the log of Phi~, which is by 32 x 32 tiles). They load
// each operand twice as often and win while they leave the chip's load paths idle; at b = 1024, 16 x 16 against
// 32 x 32: 8.4 and 11.2 us at kp = 320, 11.6 and 11.2 at kp = 384, 15.9 and 11.9 at kp = 512.
constexpr int kQuadTiles = 100;  // of 32 x 32: kp <= 320
template <int DMODE>
static bool p2_spread(const StgdArgs& a) {
  return DMODE == MM_F32 && kWaves == 4 && !a.frob_pre && phase_tiles(PH_P2, a.kp, a.b) <= kQuadTiles;
}

bool stgd_small_fits(const StgdArgs& a) {  // the one-workgroup kernels add in the order of four-wave tiles
  return kWaves == 4 && a.k <= 32 && a.kp == kSmallKp && a.b <= kSmallB && !a.y_window && !a.stop && !a.frob_pre;
}

template <int MODE, typename TY>
static int run_small(hipStream_t s, const StgdArgs& args, const void* YA, const void* YB, const void* YCt, int64_t step0,
                     int64_t nsteps, int32_t renorm_every, int32_t ns_iters, int32_t ns_degree, const StgdBuffers& B, int cur,
                     double* frob_log, StgdSmallCtl* ctl) {
  SmallArgs a;
  a.ya = YA;
  a.yb = YB;
  a.yct = YCt;
  a.mu_a = args.mu_a;
  a.mu_b = args.mu_b;
  a.mu_c = args.mu_c;
  a.phi0 = B.phi[cur];
  a.phi1 = B.phi[cur ^ 1];
  a.frob = frob_log;
  a.ctl = ctl;
  a.step0 = step0;
  a.nsteps = nsteps;
  a.spe = ceil_div(args.n_x, args.bl);
  a.n_x = args.n_x;
  a.n_pad = args.n_pad;
  a.k = args.k;
  a.kp = args.kp;
  a.b = args.b;
  a.bl = args.bl;
  a.ns_iters = ns_iters;
  a.quintic = ns_degree == 5;
  a.renorm_every = renorm_every;
  a.c3 = args.c3;
  a.c1 = args.c1;
  a.c0 = args.c0;
  a.eta = args.eta;
  a.theta = args.theta;
  if (MODE == MM_F32 && a.k <= 16) {
    hipLaunchKernelGGL(stgd_small16_kernel, dim3(1), dim3(kSmall16Threads), small16_shm_bytes(a.b), s, a);
  } else {
    const void* fn = reinterpret_cast<const void*>(stgd_small_kernel<MODE, TY>);
    MMSB_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)small_shm_bytes<MODE>(kSmallB)));
    hipLaunchKernelGGL((stgd_small_kernel<MODE, TY>), dim3(1), dim3(kSmallThreads), small_shm_bytes<MODE>(a.b), s, a);
  }
  MMSB_LAUNCH_CHECK();
  return MMSB_OK;
}

int stgd_run_small(hipStream_t s, int32_t precision, const StgdArgs& args, const void* YA, const void* YB, const void* YCt,
                   int64_t step0, int64_t nsteps, int32_t renorm_every, int32_t ns_iters, int32_t ns_degree,
                   const StgdBuffers& bufs, int cur, double* frob_log, StgdSmallCtl* ctl) {
  MMSB_CHECK_ARG(stgd_small_fits(args) && nsteps > 0, "stgd_run_small: instance too large");
  if (precision == MMSB_PREC_BF16)
    return run_small<MM_BF16X3, __bf16>(s, args, YA, YB, YCt, step0, nsteps, renorm_every, ns_iters, ns_degree, bufs, cur,
                                        frob_log, ctl);
  return run_small<MM_F32, float>(s, args, YA, YB, YCt, step0, nsteps, renorm_every, ns_iters, ns_degree, bufs, cur, frob_log,
                                  ctl);
}

template <int DMODE, int KMODE, typename TY, typename TPH>
static int run_steps(hipStream_t s, const StgdArgs& args, const void* YA, const void* YB, const void* YCt, int64_t step0,
                     int64_t nsteps, int32_t renorm_every, int32_t ns_iters, int32_t ns_degree, const StgdBuffers& B,
                     int& cur, double* frob_log, StgdTiming* timing, const StgdFill& fill, const StgdRenorm& renorm) {
  const int kp = args.kp;
  const int64_t spe = ceil_div(args.n_x, args.bl);
  const StepPlan P{args, B, YA, YB, YCt, ns_iters, ns_degree, KMODE == MM_BF16X3};
  StopArgs stop{args.stop, 0, args.thresh, args.iter_min, args.iter_max};
  int64_t yrow0 = 0, win0 = 0, win1 = 0;  // rows [win0, win1) of X in the window
  int32_t nb = 0;
  auto launch = [&](int phase, int it) -> int {
    const dim3 grid(phase_tiles(phase, kp, args.b) * (phase == PH_P2S ? 4 : 1)), block(kThreads);
    const int64_t st = stop.st;
    const PhaseArgs a = P.resolve(phase, it, cur, yrow0, nb, frob_log + st, st > 0 ? frob_log + st - 1 : nullptr, frob_log, nsteps);
#define MMSB_PHASE(PH)                                                                                                      \
  case PH:                                                                                                                  \
    if (stop.stop)                                                                                                          \
      hipLaunchKernelGGL((stgd_phase_kernel<DMODE, KMODE, TY, TPH, PH, true>), grid, block, 0, s, phase_args<PH>(a), stop);   \
    else                                                                                                                    \
      hipLaunchKernelGGL((stgd_phase_kernel<DMODE, KMODE, TY, TPH, PH, false>), grid, block, 0, s, phase_args<PH>(a), stop);  \
    break;
    switch (phase) {
      MMSB_PHASE(PH_SETUP)
      MMSB_PHASE(PH_P1)
      MMSB_PHASE(PH_P2)
      case PH_P2S:
        if constexpr (DMODE == MM_F32 && kWaves == 4) {
          if (stop.stop)
            hipLaunchKernelGGL((stgd_phase_kernel<DMODE, KMODE, TY, TPH, PH_P2S, true>), grid, block, 0, s, a.p2, stop);
          else
            hipLaunchKernelGGL((stgd_phase_kernel<DMODE, KMODE, TY, TPH, PH_P2S, false>), grid, block, 0, s, a.p2, stop);
        }
        break;
      MMSB_PHASE(PH_GRAM)
      MMSB_PHASE(PH_UPDATE)
      MMSB_PHASE(PH_QPOLY)
      MMSB_PHASE(PH_QRFIN)
      MMSB_PHASE(PH_FROB)
      MMSB_PHASE(PH_COPY)
    }
#undef MMSB_PHASE
    MMSB_LAUNCH_CHECK();
    return MMSB_OK;
  };
  MMSB_TRY(launch(PH_SETUP, 0));
  for (int64_t st = 0; st < nsteps; ++st) {
    const int64_t gstep = step0 + st;
    const int64_t row0 = (gstep % spe) * args.bl;
    nb = (int32_t)std::min<int64_t>(args.bl, args.n_x - row0);
    yrow0 = row0 - win0;
    stop.st = st;
    if (timing) MMSB_HIP(hipEventRecord(timing->ev[0], s));
    if (args.y_window && (row0 < win0 || row0 + nb > win1)) {
      const int64_t in_epoch = std::min<int64_t>(spe - gstep % spe, timing ? 1 : nsteps - st);  // timed phases: step by step
      const int64_t steps = std::max<int64_t>(1, std::min<int64_t>(in_epoch, (args.n_pad - args.b) / args.bl + 1));
      win0 = row0;
      win1 = std::min<int64_t>(row0 + steps * args.bl, args.n_x);
      yrow0 = 0;
      MMSB_TRY(fill(win0, (int32_t)(win1 - win0)));
    }
    MMSB_TRY(launch(PH_P1, 0));
    if (timing) MMSB_HIP(hipEventRecord(timing->ev[1], s));
    MMSB_TRY(launch(p2_spread<DMODE>(args) ? PH_P2S : PH_P2, 0));
    if (timing) MMSB_HIP(hipEventRecord(timing->ev[2], s));
    if (renorm && renorm_every > 0 && (gstep + 1) % renorm_every == 0) {
      MMSB_TRY(renorm(B.phit, B.phia));
      MMSB_TRY(launch(PH_QRFIN, 0));
    } else if (!renorm && step_renorms(gstep, renorm_every, ns_iters)) {
      for (int it = 0; it < ns_iters; ++it) {
        MMSB_TRY(launch(PH_GRAM, it));
        if (ns_degree == 5) MMSB_TRY(launch(PH_QPOLY, it));
        MMSB_TRY(launch(PH_UPDATE, it));
      }
    } else {
      MMSB_TRY(launch(PH_COPY, 0));
    }
    if (timing) {
      MMSB_HIP(hipEventRecord(timing->ev[3], s));
      MMSB_HIP(hipEventSynchronize(timing->ev[3]));
      for (int ph = 0; ph < 3; ++ph) {
        float ms = 0.f;
        MMSB_HIP(hipEventElapsedTime(&ms, timing->ev[ph], timing->ev[ph + 1]));
        timing->ms[ph] += ms;
      }
    }
    cur ^= 1;
  }
  return launch(PH_FROB, 0);  // the last step's log entry
}

static int check_args(const StgdArgs& args, int32_t ns_iters, int32_t ns_degree) {
  MMSB_CHECK_ARG(args.kp % 64 == 0 && args.b % 64 == 0 && args.kp >= 64 && args.b >= 64,
                 "stgd: kp and b must be positive multiples of 64 (got %d, %d)", args.kp, args.b);
  MMSB_CHECK_ARG(args.bl >= 1 && args.bl <= args.b, "stgd: logical minibatch %d outside [1, %d]", args.bl, args.b);
  MMSB_CHECK_ARG(args.n_pad % 64 == 0, "stgd: n_pad must be a multiple of 64");
  const int64_t spe = ceil_div(args.n_x, args.bl);
  MMSB_CHECK_ARG(args.n_pad >= (args.y_window ? (int64_t)args.b : (spe - 1) * args.bl + args.b), "stgd: n_pad too small");
  MMSB_CHECK_ARG(ns_iters >= 0, "stgd: negative iteration count");
  MMSB_CHECK_ARG(ns_degree == 3 || ns_degree == 5, "stgd: Newton-Schulz degree must be 3 or 5 (got %d)", ns_degree);
  return MMSB_OK;
}

static int check_split(const StgdBuffers& bufs) {
  MMSB_CHECK_ARG(bufs.phi16[0] && bufs.phi16[1] && bufs.phit16 && bufs.phia16 && bufs.phiT16 && bufs.phitT16 &&
                     bufs.phiaT16 && bufs.gt16 && bufs.h16 && bufs.q16,
                 "stgd: BF16 mode needs the split operand buffers");
  return MMSB_OK;
}

int stgd_run(hipStream_t s, int32_t precision, const StgdArgs& args, const void* YA, const void* YB, const void* YCt,
             int64_t step0, int64_t nsteps, int32_t renorm_every, int32_t ns_iters, int32_t ns_degree,
             const StgdBuffers& bufs, int& cur, double* frob_log, StgdTiming* timing, const StgdFill& fill,
             const StgdRenorm& renorm) {
  MMSB_TRY(check_args(args, ns_iters, ns_degree));
  MMSB_CHECK_ARG(nsteps >= 0, "stgd: negative step count");
  MMSB_CHECK_ARG(!args.y_window || fill, "stgd: a minibatch window needs a fill callback");
  if (nsteps == 0) return MMSB_OK;
  if (precision == MMSB_PREC_BF16) {
    MMSB_TRY(check_split(bufs));
    return run_steps<MM_BF16, MM_BF16X3, __bf16, __bf16>(s, args, YA, YB, YCt, step0, nsteps, renorm_every, ns_iters,
                                                         ns_degree, bufs, cur, frob_log, timing, fill, renorm);
  }
  MMSB_CHECK_ARG(precision == MMSB_PREC_FP32, "stgd: unknown precision %d", precision);
  return run_steps<MM_F32, MM_F32, float, float>(s, args, YA, YB, YCt, step0, nsteps, renorm_every, ns_iters, ns_degree,
                                                 bufs, cur, frob_log, timing, fill, renorm);
}

// ---- batch ------------------------------------------------------------------------------------------
struct StgdBatch {
  int32_t precision = MMSB_PREC_FP32;
  int32_t ninst = 0;
  int32_t nslots = 0;
  int32_t grid = 0;
  int32_t grid_max = 0;
  PhaseArgs* d_args = nullptr;     // [segments]
  int32_t* d_first = nullptr;      // [segments]: index of the segment's first tile within its slot
  int32_t* d_phase = nullptr;      // [segments]
  int32_t* d_slot_seg = nullptr;   // [nslots + 1]: first segment of each slot
  int64_t* d_slot_tiles = nullptr; // [nslots]
  std::vector<int32_t> h_slot_seg;  // host copies for the per-slot launches
  std::vector<int64_t> h_slot_tiles;
  std::vector<int32_t> h_slot_phase;  // the phase of every segment of the slot, or -1 when they differ
};

template <int DMODE, int KMODE, typename TY, typename TPH>
static const void* batch_fn() {
  return reinterpret_cast<const void*>(stgd_batch_kernel<DMODE, KMODE, TY, TPH>);
}

static const void* batch_kernel(int32_t precision) {
  return precision == MMSB_PREC_BF16 ? batch_fn<MM_BF16, MM_BF16X3, __bf16, __bf16>() : batch_fn<MM_F32, MM_F32, float, float>();
}

int stgd_batch_plan(StgdBatch*& out, int32_t precision, const std::vector<StgdBatchMember>& members, int32_t ns_iters,
                    int32_t ns_degree, int32_t renorm_every) {
  out = nullptr;
  MMSB_CHECK_ARG(!members.empty(), "stgd batch: no instances");
  MMSB_CHECK_ARG(precision == MMSB_PREC_FP32 || precision == MMSB_PREC_BF16, "stgd batch: unknown precision %d", precision);
  std::vector<std::vector<BatchSeg>> per(members.size());
  for (size_t i = 0; i < members.size(); ++i) {
    const StgdBatchMember& m = members[i];
    MMSB_TRY(check_args(m.args, ns_iters, ns_degree));
    MMSB_CHECK_ARG(!m.args.y_window, "stgd batch: instance %zu recomputes its minibatches (not supported in a batch)", i);
    MMSB_CHECK_ARG(!m.args.stop && !m.args.frob_pre, "stgd batch: instance %zu uses the per-step end test or QR mode", i);
    if (precision == MMSB_PREC_BF16) MMSB_TRY(check_split(m.bufs));
    MMSB_CHECK_ARG(m.nsteps >= 1, "stgd batch: instance %zu has no steps", i);
    const StepPlan P{m.args, m.bufs, m.YA, m.YB, m.YCt, ns_iters, ns_degree, precision == MMSB_PREC_BF16};
    const int64_t spe = ceil_div(m.args.n_x, m.args.bl);
    auto add = [&](int phase, int it, int64_t st) {
      const int64_t row0 = ((m.step0 + st) % spe) * m.args.bl;
      BatchSeg sg;
      sg.phase = phase;
      sg.ntiles = phase_tiles(phase, m.args.kp, m.args.b);
      sg.args = P.resolve(phase, it, m.cur ^ (int)(st & 1), row0, (int32_t)std::min<int64_t>(m.args.bl, m.args.n_x - row0),
                          m.frob_log + st, st > 0 ? m.frob_log + st - 1 : nullptr, m.frob_log, m.nsteps);
      per[i].push_back(sg);
    };
    add(PH_SETUP, 0, 0);
    for (int64_t st = 0; st < m.nsteps; ++st) {
      add(PH_P1, 0, st);
      add(PH_P2, 0, st);
      if (step_renorms(m.step0 + st, renorm_every, ns_iters)) {
        for (int it = 0; it < ns_iters; ++it) {
          add(PH_GRAM, it, st);
          if (ns_degree == 5) add(PH_QPOLY, it, st);
          add(PH_UPDATE, it, st);
        }
      } else {
        add(PH_COPY, 0, st);
      }
    }
    add(PH_FROB, 0, m.nsteps - 1);
  }
  std::vector<PhaseArgs> args;
  std::vector<int32_t> first, phases;
  std::vector<int32_t> slot_seg;
  std::vector<int64_t> slot_tiles;
  std::vector<int32_t> slot_phase;
  // every member's log entry of its last step is the last segment of its list and goes into one final slot: nothing
  // writes a member's tile partials after its last step, and the other slots keep one phase each
  size_t maxlen = 0;
  for (auto& v : per) maxlen = std::max(maxlen, v.size() - 1);
  for (size_t sl = 0; sl <= maxlen; ++sl) {
    slot_seg.push_back((int32_t)args.size());
    int64_t t = 0;
    int32_t phase = -2;
    for (size_t i = 0; i < per.size(); ++i) {
      const size_t last = per[i].size() - 1;  // the FROB segment
      const size_t at = sl == maxlen ? last : sl;
      if (sl < maxlen && sl >= last) continue;
      const BatchSeg& sg = per[i][at];
      args.push_back(sg.args);
      first.push_back((int32_t)t);
      phases.push_back(sg.phase);
      t += sg.ntiles;
      phase = phase == -2 ? sg.phase : (phase == sg.phase ? phase : -1);
    }
    MMSB_CHECK_ARG(t < INT32_MAX, "stgd batch: too many tiles in a slot");
    slot_tiles.push_back(t);
    slot_phase.push_back(phase < 0 ? -1 : phase);
  }
  slot_seg.push_back((int32_t)args.size());
  MMSB_CHECK_ARG(args.size() < (size_t)INT32_MAX, "stgd batch: too many segments");
  auto* b = new StgdBatch();
  b->precision = precision;
  b->ninst = (int32_t)members.size();
  b->nslots = (int32_t)slot_tiles.size();
  b->h_slot_seg = slot_seg;
  b->h_slot_tiles = slot_tiles;
  b->h_slot_phase = slot_phase;
  auto fail = [&](hipError_t e) {
    stgd_batch_free(b);
    return set_error(MMSB_ERR_HIP, "stgd batch: %s", hipGetErrorString(e));
  };
  hipError_t e;
  auto put = [](auto** dst, const auto& src) -> hipError_t {
    const size_t bytes = sizeof(src[0]) * src.size();
    const hipError_t me = dev_malloc(dst, bytes);
    return me != hipSuccess ? me : hipMemcpy(*dst, src.data(), bytes, hipMemcpyHostToDevice);
  };
  if ((e = put(&b->d_args, args)) != hipSuccess || (e = put(&b->d_first, first)) != hipSuccess ||
      (e = put(&b->d_phase, phases)) != hipSuccess || (e = put(&b->d_slot_seg, slot_seg)) != hipSuccess ||
      (e = put(&b->d_slot_tiles, slot_tiles)) != hipSuccess)
    return fail(e);
  int dev = 0, per_cu = 0, cus = 0;
  if ((e = hipGetDevice(&dev)) != hipSuccess) return fail(e);
  if ((e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, batch_kernel(precision), kThreads, 0)) != hipSuccess) return fail(e);
  if ((e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)) != hipSuccess) return fail(e);
  if (per_cu < 1) {
    stgd_batch_free(b);
    return set_error(MMSB_ERR_HIP, "stgd batch: the persistent kernel does not fit on a compute unit");
  }
  b->grid_max = per_cu * cus;   // cooperative launch: every workgroup resident
  b->grid = cus;
  out = b;
  return MMSB_OK;
}

void stgd_batch_set_grid(StgdBatch* b, int32_t grid) {
  if (b && grid > 0) b->grid = std::min(grid, b->grid_max);
}

int32_t stgd_batch_grid(const StgdBatch* b) { return b ? b->grid : 0; }
int32_t stgd_batch_grid_max(const StgdBatch* b) { return b ? b->grid_max : 0; }

int stgd_batch_launch(hipStream_t s, StgdBatch* b) {
  MMSB_CHECK_ARG(b, "stgd batch: null plan");
  void* args[] = {&b->d_args, &b->d_first, &b->d_phase, &b->d_slot_seg, &b->d_slot_tiles, &b->nslots};
  MMSB_HIP(hipLaunchCooperativeKernel(batch_kernel(b->precision), dim3(b->grid), dim3(kThreads), args, 0, s));
  return MMSB_OK;
}

template <int DMODE, int KMODE, typename TY, typename TPH>
static void launch_slot(hipStream_t s, const StgdBatch* b, int32_t sl) {
  const dim3 grid((unsigned)b->h_slot_tiles[sl]), block(kThreads);
  const int32_t s0 = b->h_slot_seg[sl], s1 = b->h_slot_seg[sl + 1];
  switch (b->h_slot_phase[sl]) {
#define MMSB_SLOT(PH)                                                                                              \
  case PH:                                                                                                         \
    hipLaunchKernelGGL((stgd_slot_phase_kernel<DMODE, KMODE, TY, TPH, PH>), grid, block, 0, s, b->d_args, b->d_first, s0, s1); \
    break;
    MMSB_SLOT(PH_SETUP)
    MMSB_SLOT(PH_P1)
    MMSB_SLOT(PH_P2)
    MMSB_SLOT(PH_GRAM)
    MMSB_SLOT(PH_UPDATE)
    MMSB_SLOT(PH_COPY)
    MMSB_SLOT(PH_QPOLY)
    MMSB_SLOT(PH_FROB)
#undef MMSB_SLOT
    default:  // segments of different phases
      hipLaunchKernelGGL((stgd_slot_kernel<DMODE, KMODE, TY, TPH>), grid, block, 0, s, b->d_args, b->d_first, b->d_phase, s0, s1);
  }
}

int stgd_batch_launch_slots(hipStream_t s, StgdBatch* b) {
  MMSB_CHECK_ARG(b, "stgd batch: null plan");
  for (int32_t sl = 0; sl < b->nslots; ++sl) {
    if (b->precision == MMSB_PREC_BF16) launch_slot<MM_BF16, MM_BF16X3, __bf16, __bf16>(s, b, sl);
    else launch_slot<MM_F32, MM_F32, float, float>(s, b, sl);
    MMSB_LAUNCH_CHECK();
  }
  return MMSB_OK;
}

void stgd_batch_free(StgdBatch* b) {
  if (!b) return;
  (void)hipFree(b->d_args);
  (void)hipFree(b->d_first);
  (void)hipFree(b->d_phase);
  (void)hipFree(b->d_slot_seg);
  (void)hipFree(b->d_slot_tiles);
  delete b;
}

}  // namespace mmsb
