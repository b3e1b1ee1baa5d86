// Stage 1: BLOCK_M = 64 block pooling of Q/K/V (HBM streaming).
//
// Reference: editing_sparse_attention.py:89-111 (pad + block mean, compress_seq :37-55) and
// the block-sum kernels tilelang_kernels.py:33-120 / triton_kernels.py:16-119.
//
// One workgroup per (b*h, 64-token block), heads fastest.  Each input is read exactly once:
//   * fp32 block sums        -> sums[i]  [B, H, NB, D]   (means = sums / block size)
//   * bf16 block sums        -> sb[i]    [B, H, NBp, D]  (what the sparse kernels read as KC / VC;
//     written here instead of by a pass over the fp32 sums: 4 heads, 2,048 tokens, forward and
//     backward 213 -> 198 us with the launches this saves)
//   * optional bf16 copy     -> xb[i]    same strides as a contiguous [B, S, H, D]
//   * optional V transposed  -> vt       [B, H, D, Sp] bf16, kv_slot() order, zero padded;
//     with vt_limit only blocks n < vt_nblk (the pipeline's target blocks; newkv.hip
//     transposes the selected source blocks once the selection is known)
// Token rows at or beyond S read as zeros, so the partial last block sums only real tokens
// and the transposed copy is zero for padding tokens.
#include <algorithm>

#include "icsa_kernels.h"
#include "pool_rows.h"

// Thread t covers chunk c = t % 16 (8 of the 128 dims) of rows g + 16 j, g = t / 16.
template <typename T>
__device__ __forceinline__ void pool_load(const PoolParams& p, int i, int n, int b, int h, Raw8<T> (&r)[4]) {
  const int t = threadIdx.x;
  const int c = t & 15, g = t >> 4;
  const T* base = reinterpret_cast<const T*>(p.x[i].p) + (int64_t)b * p.x[i].sb + (int64_t)h * p.x[i].sh;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int tok = n * ICSA_BLOCK + g + 16 * j;
    if (tok < p.S[i]) r[j].load(base + (int64_t)tok * p.x[i].ss + 8 * c);
    else r[j].zero();
  }
}

template <typename T>
__device__ __forceinline__ void pool_one(const PoolParams& p, int i, int n, int b, int h, const Raw8<T> (&rows)[4],
                                         float (*red)[ICSA_D + 4], bf16 (*vtile)[ICSA_D + 8]) {
  const int t = threadIdx.x;
  const int c = t & 15;          // 16 chunks of 8 elements across D = 128
  const int g = t >> 4;          // 16 row groups, 4 rows each
  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.f;
  const bool want_copy = p.xb[i] != nullptr;
  const bool want_vt = (p.vt != nullptr) && (i == p.vt_src) && !(p.vt_limit && n >= p.vt_nblk);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int r = g + 16 * j;
    const int tok = n * ICSA_BLOCK + r;
    float v[8];
    rows[j].to_f32(v);           // rows past S were loaded as zeros
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] += v[e];
    if (want_copy && tok < p.S[i]) {
      bf16* dst = p.xb[i] + (int64_t)b * p.xb_sb + (int64_t)tok * p.xb_ss + (int64_t)h * p.xb_sh + 8 * c;
      *reinterpret_cast<bf16x8*>(dst) = pack8_bf16(v);
    }
    if (want_vt) {
      *reinterpret_cast<bf16x8*>(&vtile[r][8 * c]) = pack8_bf16(v);
    }
  }
  const bool want_sums = p.sums[i] != nullptr || p.sb[i] != nullptr;
  if (want_sums) {
#pragma unroll
    for (int e = 0; e < 8; ++e) red[g][8 * c + e] = acc[e];
  }
  __syncthreads();
  if (want_sums && t < ICSA_D) {
    float s = 0.f;
#pragma unroll
    for (int gg = 0; gg < 16; ++gg) s += red[gg][t];      // fixed order: deterministic
    const int64_t bh = (int64_t)b * p.H + h;
    if (p.sums[i] != nullptr) p.sums[i][(bh * p.NB[i] + n) * ICSA_D + t] = s;
    if (p.sb[i] != nullptr) p.sb[i][(bh * p.NBp[i] + n) * ICSA_D + t] = f2bf(s);
  }
  if (want_vt)
    vt_store(p.vt + (int64_t)b * p.vt_sb + (int64_t)h * p.vt_sh + (int64_t)n * ICSA_BLOCK, p.vt_sd, vtile);
  __syncthreads();
}

template <typename T0, typename T1, typename T2>
__global__ void __launch_bounds__(256) icsa_pool_kernel(PoolParams p) {
  __shared__ float red[16][ICSA_D + 4];
  __shared__ bf16 vtile[ICSA_BLOCK][ICSA_D + 8];
  const int bh = blockIdx.x;          // heads fastest: neighbouring workgroups read adjacent
  const int n = blockIdx.y;           // 256-byte head rows of the same tokens
  const int b = bh / p.H, h = bh % p.H;
  // every present input's rows are requested before any is reduced
  Raw8<T0> r0[4];
  Raw8<T1> r1[4];
  Raw8<T2> r2[4];
  const bool on0 = p.x[0].p && n < p.NB[0], on1 = p.x[1].p && n < p.NB[1], on2 = p.x[2].p && n < p.NB[2];
  if (on0) pool_load<T0>(p, 0, n, b, h, r0);
  if (on1) pool_load<T1>(p, 1, n, b, h, r1);
  if (on2) pool_load<T2>(p, 2, n, b, h, r2);
  if (on0) pool_one<T0>(p, 0, n, b, h, r0, red, vtile);
  if (on1) pool_one<T1>(p, 1, n, b, h, r1, red, vtile);
  if (on2) pool_one<T2>(p, 2, n, b, h, r2, red, vtile);
#pragma unroll
  for (int i = 0; i < 3; ++i)                              // the padding rows of the bf16 sums
    if (p.sb[i] != nullptr && n >= p.NB[i] && n < p.NBp[i] && threadIdx.x < ICSA_D)
      p.sb[i][((int64_t)bh * p.NBp[i] + n) * ICSA_D + threadIdx.x] = (bf16)0.f;
}

// Host launcher: dtypes select the instantiation (bf16 / fp32 per input).
hipError_t launch_pool(const PoolParams& p, hipStream_t stream) {
  int rows = 0;
  for (int i = 0; i < 3; ++i)
    if (p.x[i].p) rows = std::max(rows, p.sb[i] ? p.NBp[i] : p.NB[i]);
  if (rows == 0) return hipSuccess;
  dim3 grid(p.B * p.H, rows);
  dim3 block(256);
  const int d0 = p.x[0].p ? p.x[0].dtype : ICSA_DT_BF16;
  const int d1 = p.x[1].p ? p.x[1].dtype : ICSA_DT_BF16;
  const int d2 = p.x[2].p ? p.x[2].dtype : ICSA_DT_BF16;
  const int code = d0 * 4 + d1 * 2 + d2;
  switch (code) {
#define ICSA_POOL_CASE(C, A, B_, C_) \
    case C: hipLaunchKernelGGL((icsa_pool_kernel<A, B_, C_>), grid, block, 0, stream, p); break;
    ICSA_POOL_CASE(0, bf16, bf16, bf16)
    ICSA_POOL_CASE(1, bf16, bf16, float)
    ICSA_POOL_CASE(2, bf16, float, bf16)
    ICSA_POOL_CASE(3, bf16, float, float)
    ICSA_POOL_CASE(4, float, bf16, bf16)
    ICSA_POOL_CASE(5, float, bf16, float)
    ICSA_POOL_CASE(6, float, float, bf16)
    ICSA_POOL_CASE(7, float, float, float)
#undef ICSA_POOL_CASE
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
