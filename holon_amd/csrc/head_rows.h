// A head's values eight neighbouring ones a lane: 16 bytes a load in bfloat16, LANES = size / 8 lanes a head (sizes of 64, 128 and 256),
// 64 / LANES heads a wave. For kernels that take a wave a head and a value a lane at a time in general; the sums here are bit for bit theirs.
#pragma once
#include "common.h"

namespace head_rows {
template <typename T>
__device__ __forceinline__ void load8(const T* p, float (&v)[8]) {
  if constexpr (sizeof(T) == 2) {
    const uint4 raw = *reinterpret_cast<const uint4*>(p);
    const T* e = reinterpret_cast<const T*>(&raw);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = Elem<T>::load(e[j]);
  } else {
    *reinterpret_cast<float4*>(v) = *reinterpret_cast<const float4*>(p);
    *reinterpret_cast<float4*>(v + 4) = *reinterpret_cast<const float4*>(p + 4);
  }
}
template <typename T>
__device__ __forceinline__ void store8(T* p, const float (&v)[8]) {
  if constexpr (sizeof(T) == 2) {
    uint4 raw;
    T* e = reinterpret_cast<T*>(&raw);
#pragma unroll
    for (int j = 0; j < 8; ++j) e[j] = Elem<T>::store(v[j]);
    *reinterpret_cast<uint4*>(p) = raw;
  } else {
    *reinterpret_cast<float4*>(p) = *reinterpret_cast<const float4*>(v);
    *reinterpret_cast<float4*>(p + 4) = *reinterpret_cast<const float4*>(v + 4);
  }
}

// The sum of a head's squares, for every lane of the head: the bits that a wave gives whose lane l adds up values l, l + 64, .. with
// multiply-adds, then over its lanes by 32, 16, .. 1. Value 8 i + j lies in register j of the head's lane i: what those lanes 64 apart hold
// lies 8 lanes apart here (added in order), a distance of 32, 16 or 8 is one of 4, 2 or 1 lanes, and one of 4, 2 or 1 is between registers.
template <int LANES>
__device__ __forceinline__ float sum_of_squares(const float (&v)[8], int lane) {
  static_assert(LANES == 8 || LANES == 16 || LANES == 32, "heads of 64, 128 and 256");
  float s[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    if constexpr (LANES == 8) {
      s[j] = xor_sum<4>(fmaf(v[j], v[j], 0.f));                // (a product that no addition may take in)
    } else {
      float a = v[j], b = lane_xor<8>(a);
      if (lane & 8) { const float x = a; a = b; b = x; }
      if constexpr (LANES == 32) {
        float c = lane_xor<16>(a), d = lane_xor<16>(b);
        if (lane & 16) { float x = a; a = c; c = x; x = b; b = d; d = x; }
        s[j] = fmaf(d, d, fmaf(c, c, fmaf(b, b, a * a)));
      } else {
        s[j] = fmaf(b, b, a * a);
      }
      s[j] += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(s[j]), 0x124, 0xf, 0xf, true));      // row_ror:4 (lanes 8 apart hold the same)
    }
    s[j] = xor_sum<1>(xor_sum<2>(s[j]));
  }
  return ((s[0] + s[4]) + (s[2] + s[6])) + ((s[1] + s[5]) + (s[3] + s[7]));
}

inline bool on16(const void* p) { return (uintptr_t)p % 16 == 0; }      // (nullptr too)
}  // namespace head_rows
