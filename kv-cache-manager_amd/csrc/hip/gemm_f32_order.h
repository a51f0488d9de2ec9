// What the 32-bit products share (gemm_f32.hip, gemm_f32_few.hip): how K is cut, which is a function of K alone, and how pieces of rows are read.
#pragma once
#include "common.h"

namespace kvcm {

using f32x4 = __attribute__((__vector_size__(4 * sizeof(float)))) float;

constexpr int kUnit = 32, kSegments = 8;      // k of a unit; most segments

// Units of 32 k per segment: up to 8 segments of equal length.
__host__ __device__ __forceinline__ int segment_units(int K) {
  const int units = (K + kUnit - 1) / kUnit;
  return (units + kSegments - 1) / kSegments;
}

// Four consecutive k of one row, zero from K on.  Rows may begin at any float: the hardware takes 16-byte loads there.  FULL: no
// piece lies outside.  FOURS: K is a multiple of 4, so a piece lies wholly inside or outside; the load is unconditional (from
// k = 0 where it would be outside) and masked afterwards.
typedef float any_four __attribute__((ext_vector_type(4), aligned(4)));
template <bool FOURS, bool FULL = false>
__device__ __forceinline__ f32x4 load4(const float* __restrict__ row, int k, int K) {
  f32x4 v;
  if constexpr (FULL) {
    const any_four x = *reinterpret_cast<const any_four*>(row + k);
    v = f32x4{x.x, x.y, x.z, x.w};
  } else if constexpr (FOURS) {
    const any_four x = *reinterpret_cast<const any_four*>(row + (k < K ? k : 0));
    v = f32x4{x.x, x.y, x.z, x.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = k < K ? v[e] : 0.f;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x = row[k + e < K ? k + e : 0];
      v[e] = k + e < K ? x : 0.f;
    }
  }
  return v;
}

// K up to 256 (models of small width, low-rank factors): these launches are bound by their latency, so they are not cut.
constexpr int kShortK = 256;

}  // namespace kvcm
