// Rows of a 64-token block in registers and the V^T store, shared by the pooling pass and the
// new-KV tables.
#pragma once

#include "icsa_common.h"

// Raw storage of 8 consecutive elements of one row (one thread's share of a 64-token row).
template <typename T> struct Raw8;
template <> struct Raw8<bf16> {
  bf16x8 v;
  __device__ __forceinline__ void load(const bf16* p) { v = *reinterpret_cast<const bf16x8*>(p); }
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (bf16)0.f;
  }
  __device__ __forceinline__ void to_f32(float o[8]) const {
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = (float)v[e];
  }
};
template <> struct Raw8<float> {
  floatx4 a, b;
  __device__ __forceinline__ void load(const float* p) {
    a = *reinterpret_cast<const floatx4*>(p);
    b = *reinterpret_cast<const floatx4*>(p + 4);
  }
  __device__ __forceinline__ void zero() { a = floatx4{0.f, 0.f, 0.f, 0.f}; b = a; }
  __device__ __forceinline__ void to_f32(float o[8]) const {
#pragma unroll
    for (int e = 0; e < 4; ++e) { o[e] = a[e]; o[4 + e] = b[e]; }
  }
};

// V^T of one block from its staged rows vtile[token][d] to the 64 columns at `dst` (row d at
// dst + d * row_stride): thread -> (d, half), 32 consecutive slots, in kv_slot order
__device__ __forceinline__ void vt_store(bf16* dst, int64_t row_stride, const bf16 (*vtile)[ICSA_D + 8]) {
  const int d = threadIdx.x >> 1, half = threadIdx.x & 1;
  dst += (int64_t)d * row_stride + 32 * half;
#pragma unroll
  for (int q4 = 0; q4 < 4; ++q4) {
    bf16x8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int slot = 32 * half + 8 * q4 + e;
      o[e] = vtile[kv_slot(slot)][d];
    }
    *reinterpret_cast<bf16x8*>(dst + 8 * q4) = o;
  }
}
