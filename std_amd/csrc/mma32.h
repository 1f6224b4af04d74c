// 32x32x16 MFMA tiles of 16-bit elements, shared by the prompt attention and the
// selection: types, the product, the LDS row swizzle and the scheduler's classes.
#pragma once

#include "common.h"

namespace stdhip {

typedef float f32x16 __attribute__((ext_vector_type(16)));

// c += a b on a 32x32 tile: lane (n = l % 32, h = l / 32) holds A[n][8 h, +8), B[8 h,
// +8)[n] and, as element i, C[8 (i / 4) + 4 h + i % 4][n].
template <typename T> struct Mma32;
template <> struct Mma32<bf16_t> {
  typedef __bf16 v8 __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ f32x16 mma(v8 a, v8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct Mma32<f16_t> {
  typedef _Float16 v8 __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ f32x16 mma(v8 a, v8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

// LDS position of a row's 16-byte chunks: chunk c of row r lives at c ^ row_swz(r). 16
// consecutive rows map one chunk to 16 positions (operand reads, a row per lane), and
// four consecutive rows map a run of four chunks to 16 positions (transposed reads, 4
// rows x 32 columns per half wave).
__device__ __forceinline__ int row_swz(int row) { return ((row & 3) << 2) | ((row >> 2) & 3); }

constexpr int kSchedMfma = 0x008, kSchedDsRead = 0x100;   // sched_group_barrier classes

}  // namespace stdhip
