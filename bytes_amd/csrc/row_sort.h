// Descending sort of up to 256 (order key, element) pairs per wave, by four or
// eight waves, in registers.
//
// A pair is one fp64 number in [1, 2): the 32-bit order key above the
// complement of the 16-bit element number in the mantissa, so the numbers
// order as (key descending, element ascending) and one v_max_f64 compares and
// exchanges.  Wave w holds values 256 w + 64 r + lane in y[r] (r = 0..3) of a
// bitonic network: strides below 64 exchange lanes (DPP moves within rows of
// 16, the LDS crossbar without memory beyond), strides 64 and 128 exchange
// registers, strides from 256 on go through LDS with a barrier.  A lane that
// has to keep the smaller value holds the pair negated for that stage, so each
// exchange is max(y, -partner) on every lane: four VALU operations a value and
// stage.  (Sorting 64-bit integers with LDS shuffles, one 64-value segment
// after another: 3584 rows of 819 selected from 2867 in 98 us against 27
// without the sort.)
#pragma once
#include "common.h"

namespace bytes_amd {

constexpr int kRowSortMax = 2048;   // eight waves

__device__ __forceinline__ uint64_t row_sort_pair(uint32_t key, int e) {   // e < 65536
  return 0x3FF0000000000000ull | ((uint64_t)key << 16) | (uint64_t)(0xFFFFu - (uint32_t)e);
}
constexpr uint64_t kRowSortPad = 0x3FF0000000000000ull;   // below every pair
__device__ __forceinline__ int row_sort_element(double y) {
  return (int)(0xFFFFu - ((uint32_t)__builtin_bit_cast(uint64_t, y) & 0xFFFFu));
}

template <int STRIDE>
__device__ __forceinline__ int lane_xor(int v) {
  if constexpr (STRIDE == 1) return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, true);        // quad_perm [1,0,3,2]
  else if constexpr (STRIDE == 2) return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, true);   // quad_perm [2,3,0,1]
  else if constexpr (STRIDE == 4) return __builtin_amdgcn_ds_swizzle(v, 0x101F);              // lane ^ 4
  else if constexpr (STRIDE == 8) return __builtin_amdgcn_mov_dpp(v, 0x128, 0xF, 0xF, true);  // row_ror:8
  else if constexpr (STRIDE == 16) return __builtin_amdgcn_ds_swizzle(v, 0x401F);             // lane ^ 16
  else return __shfl_xor(v, 32, 64);
}

__device__ __forceinline__ void flip_sign(double& y, uint32_t m) {   // m: 0 or the sign bit
  const uint64_t b = __builtin_bit_cast(uint64_t, y) ^ ((uint64_t)m << 32);
  y = __builtin_bit_cast(double, b);
}

// Exchange over lanes at STRIDE; z: the sign bit where this wave's register r
// belongs to an ascending block.
template <int STRIDE>
__device__ __forceinline__ void sort_lanes(double (&y)[4], const uint32_t (&z)[4]) {
  const uint32_t m = (threadIdx.x & STRIDE) ? 0x80000000u : 0u;
  double p[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    flip_sign(y[r], m ^ z[r]);
    const uint64_t b = __builtin_bit_cast(uint64_t, y[r]);
    const uint32_t lo = (uint32_t)lane_xor<STRIDE>((int)(uint32_t)b), hi = (uint32_t)lane_xor<STRIDE>((int)(uint32_t)(b >> 32));
    p[r] = __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
  }
  // (a DPP read of a VALU result needs two wait states: the s_nop covers the
  // moves that may follow)
  asm("v_max_f64 %0, %0, -%4\n\tv_max_f64 %1, %1, -%5\n\tv_max_f64 %2, %2, -%6\n\tv_max_f64 %3, %3, -%7\n\ts_nop 1"
      : "+v"(y[0]), "+v"(y[1]), "+v"(y[2]), "+v"(y[3])
      : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]));
#pragma unroll
  for (int r = 0; r < 4; ++r) flip_sign(y[r], m ^ z[r]);
}

// Exchange of two registers: the larger (of the negated values in an ascending
// block) goes to a.
__device__ __forceinline__ void sort_pair(double& a, double& b, uint32_t z) {
  flip_sign(a, z);
  flip_sign(b, z);
  double hi, lo;
  asm("v_max_f64 %0, %2, %3\n\tv_min_f64 %1, %2, %3\n\ts_nop 1" : "=&v"(hi), "=&v"(lo) : "v"(a), "v"(b));
  a = hi;
  b = lo;
  flip_sign(a, z);
  flip_sign(b, z);
}

// The stages of blocks of SIZE.
template <int SIZE, int NW>
__device__ __forceinline__ void sort_size(double (&y)[4], uint64_t* sb) {
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  uint32_t z[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = 256 * w + 64 * r + lane;
    z[r] = (i & SIZE) ? 0x80000000u : 0u;
  }
#pragma unroll
  for (int stride = SIZE / 2; stride >= 256; stride >>= 1) {
    __syncthreads();
    if (w < NW)
#pragma unroll
      for (int r = 0; r < 4; ++r) sb[256 * w + 64 * r + lane] = __builtin_bit_cast(uint64_t, y[r]);
    __syncthreads();
    if (w < NW)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 256 * w + 64 * r + lane;
        const uint64_t a = __builtin_bit_cast(uint64_t, y[r]), p = sb[i ^ stride];
        const bool larger = ((i & stride) == 0) == (z[r] == 0u);   // (pairs are positive: bits order as values)
        y[r] = __builtin_bit_cast(double, larger == (a > p) ? a : p);
      }
  }
  if (SIZE > 128) {
    sort_pair(y[0], y[2], z[0]);
    sort_pair(y[1], y[3], z[0]);
  }
  if (SIZE > 64) {
    sort_pair(y[0], y[1], z[0]);
    sort_pair(y[2], y[3], z[2]);
  }
  if (SIZE > 32) sort_lanes<32>(y, z);
  if (SIZE > 16) sort_lanes<16>(y, z);
  if (SIZE > 8) sort_lanes<8>(y, z);
  if (SIZE > 4) sort_lanes<4>(y, z);
  if (SIZE > 2) sort_lanes<2>(y, z);
  sort_lanes<1>(y, z);
}

// Sorts the n <= 256 NW pairs of sb (LDS, 256 NW entries) into y: value i of
// the descending order is y[r] of wave w, lane l with i = 256 w + 64 r + l.
// Every thread of the workgroup (at least NW waves) calls it; waves from NW on
// only meet the barriers.  Begins with a barrier.
template <int NW>
__device__ __forceinline__ void row_sort_desc(uint64_t* sb, int n, double (&y)[4]) {
  static_assert(NW == 4 || NW == 8, "256 pairs a wave");
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = 256 * w + 64 * r + lane;
    y[r] = __builtin_bit_cast(double, i < n ? sb[i] : kRowSortPad);
  }
  sort_size<2, NW>(y, sb);
  sort_size<4, NW>(y, sb);
  sort_size<8, NW>(y, sb);
  sort_size<16, NW>(y, sb);
  sort_size<32, NW>(y, sb);
  sort_size<64, NW>(y, sb);
  if (n > 64) sort_size<128, NW>(y, sb);
  if (n > 128) sort_size<256, NW>(y, sb);
  if (n > 256) sort_size<512, NW>(y, sb);
  if (n > 512) sort_size<1024, NW>(y, sb);
  if constexpr (NW == 8)
    if (n > 1024) sort_size<2048, NW>(y, sb);
}

}  // namespace bytes_amd
