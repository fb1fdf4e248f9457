// Running sums and maxima over the lanes of a wave with lane moves inside the vector unit (DPP), transpose reads, and a workgroup's barrier.
//
// A permute through the LDS pipe (__shfl_up and the like) costs a kernel that has a wave or two per
// SIMD, and so nothing to hide a latency behind, some 70 cycles each: six dependent ones per scan.
// These take a handful of vector instructions.  All 64 lanes of the wave must be active.
#ifndef SSPMM_AMD_LANE_OPS_H
#define SSPMM_AMD_LANE_OPS_H

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sspmm {

// CTRL: 0x110 + n = the value of the lane n below in the same row of 16 lanes; 0x142 = of lane 15 of the row
// below; 0x143 = of lane 31; delivered to the rows ROW_MASK names.  Lanes without a source, and rows not
// named, get 0.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t lanes_below(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROW_MASK, 0xf, true);
}
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ unsigned long long lanes_below(unsigned long long v) {
  const uint32_t lo = lanes_below<CTRL, ROW_MASK>((uint32_t)v);
  const uint32_t hi = lanes_below<CTRL, ROW_MASK>((uint32_t)(v >> 32));
  return ((unsigned long long)hi << 32) | lo;
}

// Sum of v over lanes 0 .. own lane.  T: uint32_t or unsigned long long.
template <typename T>
__device__ __forceinline__ T wave_inclusive_sum(T v) {
  v += lanes_below<0x111, 0xf>(v);
  v += lanes_below<0x112, 0xf>(v);
  v += lanes_below<0x114, 0xf>(v);
  v += lanes_below<0x118, 0xf>(v);
  v += lanes_below<0x142, 0xa>(v);  // rows 1 and 3 take the sum of the row below
  v += lanes_below<0x143, 0xc>(v);  // rows 2 and 3 take the sum of rows 0 and 1
  return v;
}

// Maximum of v over lanes 0 .. own lane.
__device__ __forceinline__ uint32_t wave_inclusive_max(uint32_t v) {
  v = max(v, lanes_below<0x111, 0xf>(v));
  v = max(v, lanes_below<0x112, 0xf>(v));
  v = max(v, lanes_below<0x114, 0xf>(v));
  v = max(v, lanes_below<0x118, 0xf>(v));
  v = max(v, lanes_below<0x142, 0xa>(v));
  v = max(v, lanes_below<0x143, 0xc>(v));
  return v;
}

// The same moves for floats, with what a lane without a source (or a row not named) gets instead given by the caller.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float lanes_below_or(float v, float otherwise) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(otherwise), __float_as_int(v), CTRL, ROW_MASK, 0xf, false));
}
// Maximum / sum of x over all 64 lanes, in every lane (the running value reaches lane 63, which is then read out).
__device__ __forceinline__ float wave_max_all(float x) {
  x = fmaxf(x, lanes_below_or<0x111, 0xf>(x, x));
  x = fmaxf(x, lanes_below_or<0x112, 0xf>(x, x));
  x = fmaxf(x, lanes_below_or<0x114, 0xf>(x, x));
  x = fmaxf(x, lanes_below_or<0x118, 0xf>(x, x));
  x = fmaxf(x, lanes_below_or<0x142, 0xa>(x, x));
  x = fmaxf(x, lanes_below_or<0x143, 0xc>(x, x));
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}
__device__ __forceinline__ float wave_sum_all(float x) {
  x += lanes_below_or<0x111, 0xf>(x, 0.f);
  x += lanes_below_or<0x112, 0xf>(x, 0.f);
  x += lanes_below_or<0x114, 0xf>(x, 0.f);
  x += lanes_below_or<0x118, 0xf>(x, 0.f);
  x += lanes_below_or<0x142, 0xa>(x, 0.f);
  x += lanes_below_or<0x143, 0xc>(x, 0.f);
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}

// The value lane 63 holds, in every lane.
__device__ __forceinline__ uint32_t from_last_lane(uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane((int)v, 63); }

// Four consecutive fp16 values of a row of which `left` exist.  RAGGED: the row begins at any element, and what lies behind its
// end is neither read nor written.
typedef _Float16 four_halfs __attribute__((ext_vector_type(4)));
typedef _Float16 four_halfs_any __attribute__((ext_vector_type(4), aligned(2)));
template <bool RAGGED, bool NT = false>
__device__ __forceinline__ four_halfs load_four(const _Float16 *p, int left) {
  if constexpr (RAGGED) {
    if (left >= 4) return *reinterpret_cast<const four_halfs_any *>(p);
    four_halfs v = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 3; ++i)
      if (i < left) v[i] = p[i];
    return v;
  } else if constexpr (NT) {
    return __builtin_nontemporal_load(reinterpret_cast<const four_halfs *>(p));
  } else {
    return *reinterpret_cast<const four_halfs *>(p);
  }
}
template <bool RAGGED>
__device__ __forceinline__ void store_four(_Float16 *p, four_halfs v, int left) {
  if constexpr (RAGGED) {
    if (left >= 4) {
      *reinterpret_cast<four_halfs_any *>(p) = v;
      return;
    }
#pragma unroll
    for (int i = 0; i < 3; ++i)
      if (i < left) p[i] = v[i];
  } else {
    *reinterpret_cast<four_halfs *>(p) = v;
  }
}

// Maximum, and below the sum, of v over the lanes of the wave with the same lane % 16, in each of them.
__device__ __forceinline__ float max_over_rows(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float sum_over_rows(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Sum of v over the lanes of the wave with the same lane % 4, in each of them.
__device__ __forceinline__ float sum_over_quads(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, false));  // rotated by 8 in each 16
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xf, 0xf, false));  // and by 4
  return sum_over_rows(v);
}

// Transpose read of 16-bit elements from LDS: within 16 lanes, lane n receives element n of the four 32-byte runs addressed by lanes 0-3,
// 4-7, 8-11, 12-15.
typedef uint32_t two_words __attribute__((ext_vector_type(2)));
__device__ __forceinline__ two_words lds_read_tr(const unsigned char *p) {
  typedef short four_shorts __attribute__((ext_vector_type(4)));
  return __builtin_bit_cast(two_words, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) four_shorts *)p));
}

// Workgroup barrier that orders LDS only: global loads in flight stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

}  // namespace sspmm
#endif
