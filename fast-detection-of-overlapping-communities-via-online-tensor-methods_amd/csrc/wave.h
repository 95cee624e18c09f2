// Wave-wide butterfly sums without LDS, added in the order of a shuffle butterfly with offsets 32, 16, 8, 4, 2, 1
// (each exchange adds the same two numbers on both sides, so the bits are those of v += __shfl_xor(v, off)).
// Offsets 32 and 16 are permlane swaps, the others DPP moves inside a row of 16 lanes -- a few cycles each where a
// shuffle goes through the LDS pipe (two ds_bpermute of ~100 cycles per double). Offset 4 rotates the row by 4:
// after the exchange over 8 the values repeat every 8 lanes, so lane (i + 4) % 16 holds what lane i ^ 4 does.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace mmsb {

// kDppHalfMirror reverses each group of 8 lanes: once the values of a quad agree, lane 7 - i holds what lane i ^ 4 does.
enum { kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppRor4 = 0x124, kDppRor8 = 0x128, kDppHalfMirror = 0x141 };

template <int CTRL>
__device__ inline float dpp_mov(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}

__device__ inline uint32_t lo32(double v) { return (uint32_t)__builtin_bit_cast(uint64_t, v); }
__device__ inline uint32_t hi32(double v) { return (uint32_t)(__builtin_bit_cast(uint64_t, v) >> 32); }
__device__ inline double join32(uint32_t lo, uint32_t hi) { return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo); }

template <int CTRL>
__device__ inline double dpp_mov(double v) {
  return join32((uint32_t)__builtin_amdgcn_mov_dpp((int)lo32(v), CTRL, 0xf, 0xf, false),
                (uint32_t)__builtin_amdgcn_mov_dpp((int)hi32(v), CTRL, 0xf, 0xf, false));
}

__device__ inline double read_lane(double v, int lane) {
  return join32((uint32_t)__builtin_amdgcn_readlane((int)lo32(v), lane), (uint32_t)__builtin_amdgcn_readlane((int)hi32(v), lane));
}

// The first exchange of two sums at once: lanes 0..31 get p[l] + p[l + 32], lanes 32..63 q[l - 32] + q[l].
__device__ inline double swap_add32(double p, double q) {
#pragma clang fp contract(off)  // a product that ends in p or q is rounded before it is summed
  const auto l = __builtin_amdgcn_permlane32_swap(lo32(p), lo32(q), false, false);
  const auto h = __builtin_amdgcn_permlane32_swap(hi32(p), hi32(q), false, false);
  return join32(l[0], h[0]) + join32(l[1], h[1]);
}

// The exchange over 16: in each half, the even row gets p's sum of its two rows, the odd row q's.
__device__ inline double swap_add16(double p, double q) {
#pragma clang fp contract(off)
  const auto l = __builtin_amdgcn_permlane16_swap(lo32(p), lo32(q), false, false);
  const auto h = __builtin_amdgcn_permlane16_swap(hi32(p), hi32(q), false, false);
  return join32(l[0], h[0]) + join32(l[1], h[1]);
}

__device__ inline float swap_add32(float p, float q) {
#pragma clang fp contract(off)
  const auto x = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, p), __builtin_bit_cast(uint32_t, q), false, false);
  return __builtin_bit_cast(float, (uint32_t)x[0]) + __builtin_bit_cast(float, (uint32_t)x[1]);
}

__device__ inline float swap_add16(float p, float q) {
#pragma clang fp contract(off)
  const auto x = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, p), __builtin_bit_cast(uint32_t, q), false, false);
  return __builtin_bit_cast(float, (uint32_t)x[0]) + __builtin_bit_cast(float, (uint32_t)x[1]);
}

__device__ inline double row_sum(double v) {  // over the row's 16 lanes
#pragma clang fp contract(off)
  v += dpp_mov<kDppRor8>(v);
  v += dpp_mov<kDppRor4>(v);
  v += dpp_mov<kDppXor2>(v);
  v += dpp_mov<kDppXor1>(v);
  return v;
}

// The sums of a, b and c over the wave, wave-uniform: the first two exchanges leave a's, c's and b's partial sums in
// rows of their own, so that the last four are taken once for the three.
__device__ inline void wave_sum3(double& a, double& b, double& c) {
  const double v = row_sum(swap_add16(swap_add32(a, b), swap_add32(c, c)));
  a = read_lane(v, 0);
  c = read_lane(v, 16);
  b = read_lane(v, 32);
}

__device__ inline double wave_sum(double v) { return row_sum(swap_add16(swap_add32(v, v), swap_add32(v, v))); }

// The largest of the wave's values (not negative).
__device__ inline double wave_max(double v) {
  v = fmax(v, dpp_mov<kDppRor8>(v));
  v = fmax(v, dpp_mov<kDppRor4>(v));
  v = fmax(v, dpp_mov<kDppXor2>(v));
  v = fmax(v, dpp_mov<kDppXor1>(v));
  return fmax(fmax(read_lane(v, 0), read_lane(v, 16)), fmax(read_lane(v, 32), read_lane(v, 48)));
}

__device__ inline float read_lane(float v, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

__device__ inline float wave_max(float v) {
  v = fmaxf(v, dpp_mov<kDppRor8>(v));
  v = fmaxf(v, dpp_mov<kDppRor4>(v));
  v = fmaxf(v, dpp_mov<kDppXor2>(v));
  v = fmaxf(v, dpp_mov<kDppXor1>(v));
  return fmaxf(fmaxf(read_lane(v, 0), read_lane(v, 16)), fmaxf(read_lane(v, 32), read_lane(v, 48)));
}

// Exchanges the upper half of a with the lower half of b.
__device__ inline void half_swap(float& a, float& b) {
  const auto x = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false);
  a = __builtin_bit_cast(float, (uint32_t)x[0]);
  b = __builtin_bit_cast(float, (uint32_t)x[1]);
}

// Sums over the lanes of a quad, and of a group of eight (offsets 1, 2, 4).
__device__ inline float quad_sum(float v) {
#pragma clang fp contract(off)
  v += dpp_mov<kDppXor1>(v);
  v += dpp_mov<kDppXor2>(v);
  return v;
}

__device__ inline float oct_sum(float v) {
#pragma clang fp contract(off)
  v = quad_sum(v);
  v += dpp_mov<kDppHalfMirror>(v);
  return v;
}

}  // namespace mmsb
