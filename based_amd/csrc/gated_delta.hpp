// What the kernels of the gated delta rule share (gated_delta.hip, gated_delta_chunk.hip).
#pragma once

#include "stream_common.hpp"

namespace based {

constexpr float kUnitEps = 1e-6f;

template <typename T> __device__ __forceinline__ float log_decay_of(float a, const void* a_log, const void* dt_bias, int h) {
  const float dt = softplus_f(a + to_f32(static_cast<const T*>(dt_bias)[h]));
  return -expf(to_f32(static_cast<const T*>(a_log)[h])) * dt;
}

// 4 consecutive channels of a row of d as they lie in memory.  Fetched without a condition (channels
// past the end come from the row's start) and cleared where they are used: a load in a branch or
// in front of a select is waited for on the spot.  LAY: 0 element by element, 1 whole aligned groups, 2 whole
// groups of rows that fill the tile (nothing to clear).
template <typename T, int LAY> struct Four {
  typedef __attribute__((ext_vector_type(4))) T t4;
  t4 r;
  __device__ __forceinline__ void load(const T* row, int e, int d) {
    if constexpr (LAY == 2) {
      r = *reinterpret_cast<const t4*>(row + e);
    } else if constexpr (LAY == 1) {
      r = *reinterpret_cast<const t4*>(row + (e < d ? e : 0));
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) r[i] = row[e + i < d ? e + i : 0];
    }
  }
  __device__ __forceinline__ f32x4 get(int e, int d) const {
    f32x4 x;
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = LAY == 2 || e + i < d ? to_f32(r[i]) : 0.f;
    return x;
  }
};

}  // namespace based
