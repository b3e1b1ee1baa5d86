// The new KV's tables, built in one launch once the source blocks are selected:
//   * V^T of the selected source blocks, in the columns behind the target blocks';
//   * block sums of the new KV (tilelang_host.py:163-168), copied from the pooled sums: fp32 for
//     the level-3 scores, bf16 rows / transposed for the sparse kernel;
//   * with t % 64 != 0, the sums of the straddling blocks from their token rows
//     (editing_sparse_attention.py:138-159, the new KV's blocks from n_t on).
// Each is a few us of latency: as launches of their own they took 5, 6 and 7-9 us (2 heads, 8,192
// tokens), as one 8.5 us; with the value means and the interval bound also taken out of launches
// of their own the layer went from 117 to 107 us (40 heads, 3,120 tokens: 185 -> 171 us).  With every
// load made unconditionally, from a clamped place, and the value selected afterwards: 5.0 us
// (layer 102 -> 98; 5 heads, 65,536 tokens 11.7 -> 8.2, 40 heads 38 -> 32 us).
// Workgroups of 256 threads along y: the selected blocks, then 32 new-KV blocks each, then two
// straddling blocks each.
#include "icsa_kernels.h"
#include "pool_rows.h"

// V^T of selected block r (an entry outside the sequence stores a zero block, so no column
// keeps stale workspace data).  Thread t: chunk t % 16 (8 dims) of rows t / 16 + 16 j.
template <typename T>
__device__ __forceinline__ void newkv_vt(const NewKvParams& p, int bh, int r, bf16 (*vtile)[ICSA_D + 8]) {
  const int b = bh / p.H, h = bh % p.H;
  const int n = p.sel_base + p.sel[(int64_t)bh * p.sel_stride + r];
  const int NB = (p.S + ICSA_BLOCK - 1) / ICSA_BLOCK;
  const bool real = n >= 0 && n < NB;                  // uniform for the workgroup
  const int c = threadIdx.x & 15, g = threadIdx.x >> 4;
  const T* base = reinterpret_cast<const T*>(p.v.p) + (int64_t)b * p.v.sb + (int64_t)h * p.v.sh + 8 * c;
  Raw8<T> rows[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int tok = n * ICSA_BLOCK + g + 16 * j;
    rows[j].load(base + (int64_t)(real ? min(tok, p.S - 1) : 0) * p.v.ss);
    if (!real || tok >= p.S) rows[j].zero();
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float v[8];
    rows[j].to_f32(v);
    *reinterpret_cast<bf16x8*>(&vtile[g + 16 * j][8 * c]) = pack8_bf16(v);
  }
  __syncthreads();
  vt_store(p.vt + (int64_t)b * p.vt_sb + (int64_t)h * p.vt_sh + (int64_t)(p.vt_dst0 + r) * ICSA_BLOCK, p.vt_sd, vtile);
}

// Sums of 16 consecutive new-KV blocks from j0, thread d (of 128): dim d of each (the 32 source
// sums of a thread are requested together).  The 16 blocks' V sums of dim d are one 16-slot
// group of V^T row d, written as 32 contiguous bytes in kv_slot() order (kv_slot swaps two
// index bits, so it is its own inverse).
__device__ __forceinline__ void newkv_sums(const NewKvParams& p, int bh, int j0, int d) {
  if (j0 >= p.NKVp) return;
  // every load is made (blocks without a source: of block 0) and the sum selected afterwards: a
  // condition around the loads made 16 branches of them, each waiting for the one before
  int src[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) src[i] = p.kvmap[(int64_t)bh * p.NKV + min(j0 + i, p.NKV - 1)];
  float ks[16], vs[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int64_t at = ((int64_t)bh * p.Nsrc + max(src[i], 0)) * ICSA_D + d;
    ks[i] = p.ksum[at];
    vs[i] = p.vsum[at];
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const bool real = j0 + i < p.NKV && src[i] >= 0;
    ks[i] = real ? ks[i] : 0.f;
    vs[i] = real ? vs[i] : 0.f;
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int j = j0 + i;
    if (p.seg_a > 0 && j >= p.seg_from && j < p.NKV) continue;   // newkv_straddle
    if (j < p.NKV) p.kc32[((int64_t)bh * p.NKV + j) * ICSA_D + d] = ks[i];
    p.kc[((int64_t)bh * p.NKVp + j) * ICSA_D + d] = f2bf(ks[i]);
    if (p.vc) p.vc[((int64_t)bh * p.NKVp + j) * ICSA_D + d] = f2bf(vs[i]);
  }
  if (p.vct) {                    // no straddling blocks where V^T sums are wanted (seg_a == 0)
    bf16x8 a, b;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      a[s] = f2bf(vs[kv_slot(s)]);
      b[s] = f2bf(vs[kv_slot(s + 8)]);
    }
    bf16* dst = p.vct + ((int64_t)bh * ICSA_D + d) * p.NKVp + j0;
    *reinterpret_cast<bf16x8*>(dst) = a;
    *reinterpret_cast<bf16x8*>(dst + 8) = b;
  }
}

// Straddling new-KV block j: rows r < a from tokens segA + r, rows r >= a from 64 kvmap[j] +
// r - a, summed straight from the token rows by 128 threads.  Thread t: 8 dims 8 (t % 16) .. +
// 7 of rows t / 16 + 8 m; the 8 row groups are added in fixed order.
template <typename TK, typename TV>
__device__ __forceinline__ void newkv_straddle(const NewKvParams& p, int bh, int j, int t,
                                               float (*red)[8][ICSA_D + 4]) {
  const int b = bh / p.H, h = bh % p.H;
  const int c = t & 15, g = t >> 4;
  const int a = p.seg_a;
  const bool on = j < p.NKV;                           // the last workgroup's second block
  float ks[8], vs[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) { ks[e] = 0.f; vs[e] = 0.f; }
  if (on) {
    const int* map = p.kvmap + (int64_t)bh * p.NKV;
    int tokA = -1;
    if (j == p.seg_from) tokA = ICSA_BLOCK * p.seg_from;
    else if (map[j - 1] >= 0) tokA = ICSA_BLOCK * map[j - 1] + ICSA_BLOCK - a;
    const int tokB = map[j] >= 0 ? ICSA_BLOCK * map[j] - a : -1;    // token of row r >= a: tokB + r
    const TK* kb = reinterpret_cast<const TK*>(p.k.p) + (int64_t)b * p.k.sb + (int64_t)h * p.k.sh;
    const TV* vb = reinterpret_cast<const TV*>(p.v.p) + (int64_t)b * p.v.sb + (int64_t)h * p.v.sh;
    Raw8<TK> kr[8];
    Raw8<TV> vr[8];
    auto token = [&](int m) -> int {
      const int r = g + 8 * m;
      const int tok = r < a ? (tokA < 0 ? -1 : tokA + r) : (tokB < 0 ? -1 : tokB + r);
      return tok < p.S ? tok : -1;
    };
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const int tok = max(token(m), 0);
      kr[m].load(kb + (int64_t)tok * p.k.ss + 8 * c);
      vr[m].load(vb + (int64_t)tok * p.v.ss + 8 * c);
    }
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const bool real = token(m) >= 0;
      float x[8];
      kr[m].to_f32(x);
#pragma unroll
      for (int e = 0; e < 8; ++e) ks[e] += real ? x[e] : 0.f;
      vr[m].to_f32(x);
#pragma unroll
      for (int e = 0; e < 8; ++e) vs[e] += real ? x[e] : 0.f;
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) { red[0][g][8 * c + e] = ks[e]; red[1][g][8 * c + e] = vs[e]; }
  __syncthreads();
  if (!on) return;
  const int d = t;
  float k_sum = 0.f, v_sum = 0.f;
#pragma unroll
  for (int gg = 0; gg < 8; ++gg) { k_sum += red[0][gg][d]; v_sum += red[1][gg][d]; }
  p.kc32[((int64_t)bh * p.NKV + j) * ICSA_D + d] = k_sum;
  p.kc[((int64_t)bh * p.NKVp + j) * ICSA_D + d] = f2bf(k_sum);
  if (p.vc) p.vc[((int64_t)bh * p.NKVp + j) * ICSA_D + d] = f2bf(v_sum);
}

template <typename TK, typename TV>
__global__ void __launch_bounds__(256) icsa_newkv_kernel(NewKvParams p) {
  // the rows of a V^T block, or two straddling blocks' row-group sums
  constexpr int kVtile = ICSA_BLOCK * (ICSA_D + 8) * 2, kRed = 2 * 2 * 8 * (ICSA_D + 4) * 4;
  __shared__ __attribute__((aligned(16))) unsigned char lds[kVtile > kRed ? kVtile : kRed];
  const int bh = blockIdx.x, half = threadIdx.x >> 7, t = threadIdx.x & 127;
  int y = blockIdx.y;
  if (y < p.n_sel) {
    newkv_vt<TV>(p, bh, y, reinterpret_cast<bf16 (*)[ICSA_D + 8]>(lds));
    return;
  }
  y -= p.n_sel;
  const int n_sums = (p.NKVp + 31) / 32;
  if (y < n_sums) {
    newkv_sums(p, bh, 32 * y + 16 * half, t);
    return;
  }
  newkv_straddle<TK, TV>(p, bh, p.seg_from + 2 * (y - n_sums) + half, t,
                         reinterpret_cast<float (*)[8][ICSA_D + 4]>(lds) + 2 * half);
}

hipError_t launch_newkv(const NewKvParams& p, hipStream_t stream) {
  if (p.NKVp % 16 != 0 || (p.vct && p.seg_a > 0) || !p.kvmap || !p.k.p || !p.v.p || (p.n_sel > 0 && !p.vt))
    return hipErrorInvalidValue;
  const bool sums = p.kc32 != nullptr;
  const int n_str = sums && p.seg_a > 0 && p.seg_from < p.NKV ? (p.NKV - p.seg_from + 1) / 2 : 0;
  const int rows = p.n_sel + (sums ? (p.NKVp + 31) / 32 + n_str : 0);
  if (rows == 0 || p.BH == 0) return hipSuccess;
  const dim3 grid(p.BH, rows);
  const bool kf = p.k.dtype == ICSA_DT_F32, vf = p.v.dtype == ICSA_DT_F32;
  if (kf && vf) hipLaunchKernelGGL((icsa_newkv_kernel<float, float>), grid, dim3(256), 0, stream, p);
  else if (kf) hipLaunchKernelGGL((icsa_newkv_kernel<float, bf16>), grid, dim3(256), 0, stream, p);
  else if (vf) hipLaunchKernelGGL((icsa_newkv_kernel<bf16, float>), grid, dim3(256), 0, stream, p);
  else hipLaunchKernelGGL((icsa_newkv_kernel<bf16, bf16>), grid, dim3(256), 0, stream, p);
  return hipGetLastError();
}
