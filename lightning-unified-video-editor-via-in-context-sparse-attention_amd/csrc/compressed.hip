// Stage 2: compressed (block-level) attention, per-head source retrieval, sharpness split,
// new-KV block sums and per-query-block (level-3) top-k selection.
//
// Reference:
//   editing_sparse_attention.py:58-64, 113-123  compressed attention + out_c residual
//   editing_sparse_attention.py:125-136          per-head source top-k (column mass)
//   editing_sparse_attention.py:161-172          sharpness split (peaked / diffuse halves)
//   tilelang_host.py:163-173                     new-KV block sums, top_k per query block
//
// Every ranked decision uses the rule "larger value first, lower index first on ties".
// All score arithmetic is fp32 with fixed reduction orders, so repeated runs are bitwise
// identical and no float atomics are used.
#include <algorithm>

#include "attn_tile.h"
#include "icsa_kernels.h"

#define ICSA_MAX_NB 4096     // longest P row held in registers by the strip kernel
#define ICSA_MAX_SORT 4096   // longest list ranked by the select kernel
#define ICSA_MAX_NKV 2048    // longest level-3 score row held in registers

__device__ __forceinline__ float block_size_f(int blk, int NB, int S) {
  return blk < NB - 1 ? (float)ICSA_BLOCK : (float)(S - (NB - 1) * ICSA_BLOCK);
}

// ---------------------------------------------------------------------------------------
// (a) logits L = (Qs/size) (Ks/size)^T / sqrt(D) at fp32 accuracy on the bf16 matrix pipe.
//     Every fp32 operand x is split exactly into three bf16 parts, x = xh + xm + xl + r with
//     |r| <= 2^-27 |x| (xh = bf16(x), xm = bf16(x - xh), xl = bf16(x - xh - xm)), and each
//     product is formed from the six part products down to 2^-18 of its size
//     (al bh + am bm + ah bl + am bh + ah bm + ah bh, small terms first); the dropped
//     ones are below 2^-25 of it, and every part product is exact in the fp32
//     accumulator.  So the logits carry fp32-level rounding while the matrix work takes
//     6 bf16 MFMAs (32x32x16, 32 cycles) per 16 dims instead of 8 fp32 ones (32x32x2, 64).
//     Workgroup = 4 waves = 128 query rows (wave w: rows 32 w .. 32 w + 31) against one of
//     lg_split() column ranges.  A wave's split A operands stay in registers for the whole
//     range (lane (li, hl) holds row li's dims 16 s + 8 hl .. + 7, s = 0 .. 7); 32-column K
//     tiles pass through a double-buffered LDS ring of split tiles, the next tile prefetched
//     into registers while the current one is multiplied.  A fixed order of MFMAs, so
//     repeated runs are bitwise identical.
// ---------------------------------------------------------------------------------------
#define LG_ROWS 128
#define LG_COLS 32
#define LG_MIN_WG 256
#define LG_KST 136            // bf16 row stride of a split K tile (272 B: conflict-free reads)

__device__ __forceinline__ void split3_bf16(float x, bf16& h, bf16& m, bf16& l) {
  h = f2bf(x);
  const float r1 = x - bf2f(h);
  m = f2bf(r1);
  l = f2bf(r1 - bf2f(m));
}

// The same fp32-accurate product for the logits and for the level-3 block scores:
// C[r][c] = (A_r / sa) . (B_c / sb) / div over D = 128, with A's rows optionally gathered
// through a list, and sa, sb the block sizes (logits) or 1 (level-3 scores: raw sums).
struct Split3Gemm {
  const float* A;           // [BH, a_rows, D]
  const int* rows;          // output row r reads A row rows[bh * rows_stride + rows_offset + r]
  int rows_stride, rows_offset, a_rows;
  int n_rows;               // output rows per head
  const float* B;           // [BH, n_cols, D]
  int n_cols;
  float* C;                 // [BH, n_rows, n_cols]
  int NB, S;                // block sizes (block_mean)
  float div;
  int n_split;              // column ranges
};

// Column ranges per 128 rows: three (each range splits the rows' operands again; two and four
// were slower at 40 heads, 1,024 blocks), more where that leaves CUs without a workgroup, down
// to one 32-column tile a range: 5 heads, 1,024 blocks, logits 42 -> 32 us and level-3 scores
// 20 -> 12 us with 7 and 13 ranges; 2 heads, 128 blocks, 12.9 -> 10.5 us with 4.
static int lg_split(int n_rows, int n_cols, int BH) {
  const int64_t row_wg = (int64_t)BH * ((n_rows + LG_ROWS - 1) / LG_ROWS);
  const int n_ct = (n_cols + LG_COLS - 1) / LG_COLS;
  return std::max(1, std::min<int>(n_ct, (int)std::max<int64_t>(3, (LG_MIN_WG + row_wg - 1) / row_wg)));
}

// The value means for the strip pass (c), by workgroups of the logits' launch past its n_rt row
// tiles (they need nothing of the logits; as a launch of its own this cost 4-5 us).
struct VmeanParams {
  const float* vsum;        // [BH, NB, D]
  bf16* vmt;                // CompressedParams::vmt
  int NB, NBp, S, n_rt;
};

// Vm = Vsum / block size, transposed and split in two bf16 parts, for keys k0 .. k0 + 63:
// vmt[((bh * 2 + part) * D + d) * NBp + key], zero for keys >= NB.
__device__ __forceinline__ void vmean_split(const VmeanParams& p, int bh, int k0, float (*tile)[ICSA_D + 4]) {
  const int NB = p.NB, NBp = p.NBp, t = threadIdx.x;
  const float* V = p.vsum + (int64_t)bh * NB * ICSA_D;
  floatx4 v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {                 // float4 f = t + 256 j: key f / 32, dims 4 (f % 32)
    const int f = t + 256 * j, key = k0 + (f >> 5);
    v[j] = key < NB ? *reinterpret_cast<const floatx4*>(V + (int64_t)key * ICSA_D + 4 * (f & 31))
                    : floatx4{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int f = t + 256 * j, key = k0 + (f >> 5);
    if (key < NB) {
      const float inv = 1.f / block_size_f(key, NB, p.S);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[j][e] *= inv;
    }
    *reinterpret_cast<floatx4*>(&tile[f >> 5][4 * (f & 31)]) = v[j];
  }
  __syncthreads();
  const int d = t >> 1, kh = t & 1;             // dim d, keys 32 kh .. + 31
  bf16* dst = p.vmt + ((int64_t)bh * 2 * ICSA_D + d) * NBp + k0 + 32 * kh;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    bf16x8 hi, lo;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float x = tile[32 * kh + 8 * g + i][d];
      const bf16 h = f2bf(x);
      hi[i] = h;
      lo[i] = f2bf(x - bf2f(h));
    }
    *reinterpret_cast<bf16x8*>(dst + 8 * g) = hi;
    *reinterpret_cast<bf16x8*>(dst + (int64_t)ICSA_D * NBp + 8 * g) = lo;
  }
}

template <bool BLOCK_MEAN>
__global__ void __launch_bounds__(256) icsa_split3_gemm_kernel(Split3Gemm g, VmeanParams vm) {
  __shared__ __attribute__((aligned(16))) bf16 ks[2][3][LG_COLS][LG_KST];
  const int rt = blockIdx.x, cs = blockIdx.y, bh = blockIdx.z;
  if (BLOCK_MEAN && rt >= vm.n_rt) {
    static_assert(sizeof(ks) >= 64 * (ICSA_D + 4) * sizeof(float), "the value tile shares the K tiles' LDS");
    const int k0 = ((rt - vm.n_rt) * (int)gridDim.y + cs) * 64;
    if (k0 < vm.NBp) vmean_split(vm, bh, k0, reinterpret_cast<float (*)[ICSA_D + 4]>(&ks[0][0][0][0]));
    return;
  }
  const int NC = g.n_cols;
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63;
  const int li = l & 31, hl = l >> 5;
  const float* qbase = g.A + (int64_t)bh * g.a_rows * ICSA_D;
  const float* kbase = g.B + (int64_t)bh * NC * ICSA_D;

  // A operands: this lane's row (divided by its block size for the logits), split in three
  bf16x8 ah[8], am[8], al[8];
  {
    const int r = rt * LG_ROWS + 32 * w + li;
    const bool ok = r < g.n_rows;
    const int row = !ok ? 0 : (g.rows ? g.rows[(int64_t)bh * g.rows_stride + g.rows_offset + r] : r);
    const float sz = (BLOCK_MEAN && ok) ? block_size_f(row, g.NB, g.S) : 1.f;
    const float* src = qbase + (int64_t)row * ICSA_D + 8 * hl;
#pragma unroll
    for (int st = 0; st < 8; ++st) {
      floatx4 v0 = {0.f, 0.f, 0.f, 0.f}, v1 = v0;
      if (ok) {
        v0 = *reinterpret_cast<const floatx4*>(src + 16 * st);
        v1 = *reinterpret_cast<const floatx4*>(src + 16 * st + 4);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        bf16 h, m, lo;
        const float x = e < 4 ? v0[e] : v1[e - 4];
        split3_bf16(BLOCK_MEAN ? x / sz : x, h, m, lo);
        ah[st][e] = h;
        am[st][e] = m;
        al[st][e] = lo;
      }
    }
  }

  const int n_ct = (NC + LG_COLS - 1) / LG_COLS;
  const int per = (n_ct + g.n_split - 1) / g.n_split;
  const int t0 = cs * per, t1 = min(n_ct, t0 + per);
  if (t0 >= t1) return;                                // uniform for the workgroup

  // K tile staging: thread -> (column tid / 8, 16 dims from 16 (tid % 8))
  const int kc = tid >> 3, kd = 16 * (tid & 7);
  floatx4 pre[4];
  auto load_tile = [&](int t) {
    const int col = t * LG_COLS + kc;
    if (col < NC) {
      const float sz = BLOCK_MEAN ? block_size_f(col, g.NB, g.S) : 1.f;
      const float* src = kbase + (int64_t)col * ICSA_D + kd;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        pre[q] = *reinterpret_cast<const floatx4*>(src + 4 * q);
        if (BLOCK_MEAN) {
#pragma unroll
          for (int e = 0; e < 4; ++e) pre[q][e] = pre[q][e] / sz;
        }
      }
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) pre[q] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
  };
  auto store_tile = [&](int buf) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      bf16x8 h, m, lo;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        bf16 a, b, c;
        split3_bf16(pre[2 * half + (e >> 2)][e & 3], a, b, c);
        h[e] = a;
        m[e] = b;
        lo[e] = c;
      }
      *reinterpret_cast<bf16x8*>(&ks[buf][0][kc][kd + 8 * half]) = h;
      *reinterpret_cast<bf16x8*>(&ks[buf][1][kc][kd + 8 * half]) = m;
      *reinterpret_cast<bf16x8*>(&ks[buf][2][kc][kd + 8 * half]) = lo;
    }
  };

  float* out = g.C + (int64_t)bh * g.n_rows * NC;
  load_tile(t0);
  store_tile(0);
  __syncthreads();
  for (int t = t0; t < t1; ++t) {
    const int buf = (t - t0) & 1;
    const bool more = t + 1 < t1;
    if (more) load_tile(t + 1);
    floatx16 acc = {};
#pragma unroll
    for (int st = 0; st < 8; ++st) {
      const bf16x8 bh = *reinterpret_cast<const bf16x8*>(&ks[buf][0][li][16 * st + 8 * hl]);
      const bf16x8 bm = *reinterpret_cast<const bf16x8*>(&ks[buf][1][li][16 * st + 8 * hl]);
      const bf16x8 bl = *reinterpret_cast<const bf16x8*>(&ks[buf][2][li][16 * st + 8 * hl]);
      acc = mfma32x32x16(al[st], bh, acc);
      acc = mfma32x32x16(am[st], bm, acc);
      acc = mfma32x32x16(ah[st], bl, acc);
      acc = mfma32x32x16(am[st], bh, acc);
      acc = mfma32x32x16(ah[st], bm, acc);
      acc = mfma32x32x16(ah[st], bh, acc);
    }
    const int col = t * LG_COLS + li;
    if (col < NC) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int row = rt * LG_ROWS + 32 * w + acc_row(i, l);
        if (row < g.n_rows) out[(int64_t)row * NC + col] = acc[i] / g.div;
      }
    }
    if (more) store_tile(buf ^ 1);                     // that buffer was read in step t - 1
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------------------
// (b) row statistics, one wave per row of logits (held in registers, VPL per lane): row
//     max m, 1 / sum exp(L - m), and the sharpness = sum of the k_sparsity largest
//     P[i, :n_t].  exp is monotonic, so the k-th largest target probability is
//     exp(tau - m) / z for the k-th largest target logit tau, found by bisection over the
//     order-preserving float keys with ballot counts.
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ int wave_count(bool pred) { return __popcll(__ballot(pred)); }

// Whole-wave reductions over DPP lane moves (no LDS round trip): quad swaps, half-row and
// row mirrors leave every lane of a 16-lane row holding the row's result; two row
// broadcasts fold rows 0+1 and 2+3 and then the pairs into lane 63, which is read back as
// a wave-uniform value.  A fixed combination order, so sums are bitwise reproducible.
// Every lane of the wave must be active.
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_mov(uint32_t old, uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)x, CTRL, ROWS, 0xf, false);
}
template <typename F>
__device__ __forceinline__ uint32_t wave_reduce(uint32_t x, uint32_t ident, F op) {
  x = op(x, dpp_mov<0xb1, 0xf>(ident, x));     // quad_perm [1, 0, 3, 2]
  x = op(x, dpp_mov<0x4e, 0xf>(ident, x));     // quad_perm [2, 3, 0, 1]
  x = op(x, dpp_mov<0x141, 0xf>(ident, x));    // row_half_mirror
  x = op(x, dpp_mov<0x140, 0xf>(ident, x));    // row_mirror
  x = op(x, dpp_mov<0x142, 0xa>(ident, x));    // row_bcast:15 into rows 1 and 3
  x = op(x, dpp_mov<0x143, 0xc>(ident, x));    // row_bcast:31 into rows 2 and 3
  return (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
}
__device__ __forceinline__ float wave_max_dpp(float x) {
  return __uint_as_float(wave_reduce(__float_as_uint(x), __float_as_uint(-INFINITY), [](uint32_t a, uint32_t b) {
    return __float_as_uint(fmaxf(__uint_as_float(a), __uint_as_float(b)));
  }));
}
__device__ __forceinline__ float wave_sum_dpp(float x) {
  return __uint_as_float(wave_reduce(__float_as_uint(x), 0u, [](uint32_t a, uint32_t b) {
    return __float_as_uint(__uint_as_float(a) + __uint_as_float(b));
  }));
}
__device__ __forceinline__ uint32_t wave_min_u32(uint32_t x) {
  return wave_reduce(x, 0xffffffffu, [](uint32_t a, uint32_t b) { return a < b ? a : b; });
}
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t x) {
  return wave_reduce(x, 0u, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
}

// Largest key lo with count(key >= lo) >= k over the wave's keys (keys 0 = absent; requires
// at least k nonzero keys): the key of the k-th largest.  Only registers u < nu can hold
// nonzero keys; they are visited in groups of four (one uniform branch per group, the
// zero keys of a partly used group never count).  Bisection over the key range; as soon
// as a midpoint has exactly k keys at or above it, the answer is the smallest of those
// keys (one wave minimum), which for spread-out values ends the search long before the
// 32nd step.  The search starts from a bracket that the keys themselves give: every lane's
// largest key is at or above the smallest of the 64 lane maxima, so for k <= 64 that
// minimum has at least k keys at or above it, and no key lies above the wave's largest.
// The answer is the same key from any valid bracket; the narrower one saves steps.
template <int VPL>
__device__ __forceinline__ uint32_t kth_largest_key(const uint32_t (&key)[VPL], int k, int nu) {
  static_assert(VPL % 4 == 0, "registers are visited in groups of four");
  uint32_t lmax = 0u;
#pragma unroll
  for (int g = 0; g < VPL; g += 4)
    if (g < nu) {
#pragma unroll
      for (int u = g; u < g + 4; ++u) lmax = key[u] > lmax ? key[u] : lmax;
    }
  const uint32_t kmax = wave_max_u32(lmax);
  uint32_t lo = k <= 64 ? wave_min_u32(lmax) : 0u;
  uint32_t hi = kmax == 0xffffffffu ? kmax : kmax + 1u;
  while (hi - lo > 1u) {
    const uint32_t mid = lo + ((hi - lo) >> 1);
    int c = 0;
#pragma unroll
    for (int g = 0; g < VPL; g += 4)
      if (g < nu) {
#pragma unroll
        for (int u = g; u < g + 4; ++u) c += wave_count(key[u] >= mid);
      }
    if (c == k) {
      uint32_t mn = 0xffffffffu;
#pragma unroll
      for (int g = 0; g < VPL; g += 4)
        if (g < nu) {
#pragma unroll
          for (int u = g; u < g + 4; ++u)
            if (key[u] >= mid && key[u] < mn) mn = key[u];
        }
      return wave_min_u32(mn);
    }
    if (c > k) lo = mid; else hi = mid;
  }
  return lo;
}

template <int VPL>   // logits per lane: NB <= 64 * VPL
__global__ void __launch_bounds__(256) icsa_compressed_stats_kernel(CompressedParams p) {
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + w;          // over BH * NB rows
  if (row >= (int64_t)p.BH * p.NB) return;
  const int NB = p.NB, n_t = p.n_t;
  const float* L = p.L + row * NB;
  float v[VPL];
  uint32_t key[VPL];                              // order keys of the target logits (0: none)
  float m = -INFINITY;
#pragma unroll
  for (int u = 0; u < VPL; ++u) {
    const int j = lane + 64 * u;
    v[u] = j < NB ? L[j] : -INFINITY;
    key[u] = j < n_t ? f2key(v[u]) : 0u;
    m = fmaxf(m, v[u]);
  }
  m = wave_max_dpp(m);
  float z = 0.f;
#pragma unroll
  for (int u = 0; u < VPL; ++u) {
    v[u] = expf(v[u] - m);                        // v now holds exp(L - m)
    z += v[u];
  }
  z = wave_sum_dpp(z);
  float sharp = 0.f;
  if (n_t > 0) {
    const int k = p.k_sparsity;
    const int nu = (n_t + 63) / 64;
    const uint32_t lo = kth_largest_key<VPL>(key, k, nu);
    int cgt = 0;
    float sa = 0.f;
#pragma unroll
    for (int g = 0; g < VPL; g += 4)
      if (g < nu) {
#pragma unroll
        for (int u = g; u < g + 4; ++u) {
          const bool in = key[u] > lo;
          cgt += wave_count(in);
          sa += in ? v[u] : 0.f;
        }
      }
    sa = wave_sum_dpp(sa);
    sharp = (sa + (float)(k - cgt) * expf(key2f(lo) - m)) / z;
  }
  if (lane == 0) {
    p.rstat[2 * row] = m;
    p.rstat[2 * row + 1] = 1.f / z;
    p.sharp[row] = sharp;
  }
}

// ---------------------------------------------------------------------------------------
// (c) one 64-row strip of P per workgroup of 8 waves, in 32-key chunks: out_c = P Vm with
//     P = exp(L - m) / z, on the bf16 matrix pipe from split operands.  Per chunk:
//       * the chunk's logits (64 x 32 fp32) and its split, transposed value means (two bf16
//         planes of 128 dims x 32 keys, vmean_split) arrive by LDS DMA, double
//         buffered: chunk c + 1 is in flight while chunk c is computed, and two workgroups
//         share each CU (65 KB of LDS each);
//       * P is formed once in fp32 and kept as its two bf16 parts P = Ph + Pl (to 2^-17 of
//         P), and, for strips holding target rows, also in fp32 for the column sums of the
//         source columns over those rows (rows in order: the strip's partial, summed across
//         strips by the select kernel);
//       * wave w adds Pl Vh + Ph Vl + Ph Vh over the chunk's two 16-key steps into output
//         rows 32 (w % 2) .. + 31, columns 32 (w / 2) .. + 31 (the dropped Pl Vl is below
//         2^-16 of each product).
//     Fixed orders throughout, so repeated runs are bitwise identical.
// ---------------------------------------------------------------------------------------
#define RW_PB_LD 36                             // floats per P row in LDS (16-byte skew)

__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4)))
icsa_compressed_rows_kernel(CompressedParams p, int NBp) {
  // two stages of the chunk operands as separate objects; 65 KB in all, two workgroups per CU
  __shared__ __attribute__((aligned(16))) float lc0[64 * 32], lc1[64 * 32];          // logits
  __shared__ __attribute__((aligned(16))) bf16 vc0[2 * ICSA_D * 32], vc1[2 * ICSA_D * 32];  // Vm^T planes
  __shared__ __attribute__((aligned(16))) float pb[64 * RW_PB_LD];   // P as [Ph x 8 | Pl x 8] per 8 keys
  __shared__ __attribute__((aligned(16))) float pf[64 * 32];         // fp32 P (target strips)
  __shared__ float row_m[64], row_iz[64];
  const int strip = blockIdx.x, bh = blockIdx.y;
  const int NB = p.NB, n_t = p.n_t;
  const int r_base = strip * 64;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  if (tid < 64) {
    const int row = r_base + tid;
    row_m[tid] = row < NB ? p.rstat[2 * ((int64_t)bh * NB + row)] : 0.f;
    row_iz[tid] = row < NB ? p.rstat[2 * ((int64_t)bh * NB + row) + 1] : 0.f;
  }
  const int n_ts = (n_t + ICSA_BLOCK - 1) / ICSA_BLOCK;
  const int tgt_rows = min(64, n_t - r_base);          // > 0 only for target strips
  const int nch = NBp / 32;                            // even

  // DMA sources: the strip's logit rows (rows past NB and keys past the last row are
  // outside the resource: no load, and P is zero there) and the head's value planes
  const float* Lbh = p.L + (int64_t)bh * NB * NB;
  const u32x4 rs_l = dma_rsrc(Lbh + (int64_t)r_base * NB, (int64_t)max(0, min(64, NB - r_base)) * NB * 4);
  const u32x4 rs_v = dma_rsrc(p.vmt + (int64_t)bh * 2 * ICSA_D * NBp, (int64_t)2 * ICSA_D * NBp * 2);
  // logits: wave w moves rows 8 w .. + 7 (128 bytes each), 16 bytes per lane
  const int l_off = ((8 * w + (lane >> 3)) * NB + 4 * (lane & 7)) * 4;
  // value planes: instruction j (0, 1) of wave w moves rows R = 16 (2 w + j) .. + 15 of the
  // 256 (plane R / 128, dim R % 128), 64 bytes each; physical 16-byte unit lane % 4 of row R
  // holds logical unit (lane % 4) ^ (R % 4)
  int v_off[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int R = 16 * (2 * w + j) + (lane >> 2);
    v_off[j] = ((R >> 7) * ICSA_D + (R & 127)) * NBp * 2 + 16 * ((lane & 3) ^ (R & 3));
  }
  auto issue = [&](int c, float* lc, bf16* vc) {
    lds_dma16(lds_u32(lc + 256 * w), l_off + 128 * c, rs_l);
#pragma unroll
    for (int j = 0; j < 2; ++j) lds_dma16(lds_u32(vc + 512 * (2 * w + j)), v_off[j] + 64 * c, rs_v);
  };

  const int li = lane & 31, hl = lane >> 5;
  const int rh = w & 1, dc = 32 * (w >> 1);
  floatx16 acc = {};
  // one chunk of 32 keys: P from lc (thread: row t / 8, keys 4 (t % 8) .. + 3), then the
  // MFMAs on vc
  auto chunk = [&](int c, const float* lc, const bf16* vc) {
    const int k0 = 32 * c;
    const bool want_cs = tgt_rows > 0 && k0 + 32 > n_t;   // uniform
    {
      const int r = tid >> 3, q = tid & 7, row = r_base + r;
      const floatx4 a = *reinterpret_cast<const floatx4*>(lc + r * 32 + 4 * q);
      const float m = row_m[r], iz = row_iz[r];
      float pv[4];
      bf16x4 hi, lo;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int col = k0 + 4 * q + i;
        pv[i] = (row < NB && col < NB) ? expf(a[i] - m) * iz : 0.f;
        const bf16 h = f2bf(pv[i]);
        hi[i] = h;
        lo[i] = f2bf(pv[i] - bf2f(h));
      }
      // 8-key group q / 2, half q % 2: Ph at floats 8 (q / 2) + 2 (q % 2), Pl 4 floats on
      float* dst = pb + r * RW_PB_LD + 8 * (q >> 1) + 2 * (q & 1);
      *reinterpret_cast<bf16x4*>(dst) = hi;
      *reinterpret_cast<bf16x4*>(dst + 4) = lo;
      if (want_cs) *reinterpret_cast<floatx4*>(pf + r * 32 + 4 * q) = floatx4{pv[0], pv[1], pv[2], pv[3]};
    }
    ATT_BARRIER();                                   // P of the chunk ready
    if (want_cs && tid < 32) {
      const int col = k0 + tid;
      if (col >= n_t && col < NB) {
        float cs = 0.f;
        for (int r = 0; r < tgt_rows; ++r) cs += pf[r * 32 + tid];
        p.colpart[((int64_t)bh * n_ts + strip) * p.n_s + (col - n_t)] = cs;
      }
    }
    const float* prow = pb + (32 * rh + li) * RW_PB_LD;
    const int d = dc + li;
    const bf16* vh = vc + d * 32;
    const bf16* vl = vc + (ICSA_D + d) * 32;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int u = 2 * s + hl;                      // logical 16-byte unit: keys 8 u .. + 7
      const bf16x8 ah = *reinterpret_cast<const bf16x8*>(prow + 8 * u);
      const bf16x8 al = *reinterpret_cast<const bf16x8*>(prow + 8 * u + 4);
      const int pu = (u ^ (d & 3)) * 8;
      const bf16x8 bh_ = *reinterpret_cast<const bf16x8*>(vh + pu);
      const bf16x8 bl_ = *reinterpret_cast<const bf16x8*>(vl + pu);
      acc = mfma32x32x16(al, bh_, acc);
      acc = mfma32x32x16(ah, bl_, acc);
      acc = mfma32x32x16(ah, bh_, acc);
    }
  };

  __syncthreads();                                   // row statistics in LDS
  issue(0, lc0, vc0);
  for (int c = 0; c < nch; c += 2) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // chunk c (and this wave's older stores)
    ATT_BARRIER();                                   // chunk c in LDS; chunk c - 1 consumed
    issue(c + 1, lc1, vc1);                          // nch is even
    chunk(c, lc0, vc0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    ATT_BARRIER();
    if (c + 2 < nch) issue(c + 2, lc0, vc0);
    chunk(c + 1, lc1, vc1);
  }
  float* out = p.out_c + (int64_t)bh * NB * ICSA_D;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int row = r_base + 32 * rh + acc_row(i, lane);
    if (row < NB) out[(int64_t)row * ICSA_D + dc + li] = acc[i];
  }
}

hipError_t launch_compressed(const CompressedParams& p, hipStream_t stream) {
  if (p.NB > ICSA_MAX_NB || p.vmt == nullptr) return hipErrorInvalidValue;
  const int nt = (p.NB + 63) / 64;
  Split3Gemm g;
  g.A = p.qsum; g.rows = nullptr; g.rows_stride = 0; g.rows_offset = 0; g.a_rows = p.NB;
  g.n_rows = p.NB; g.B = p.ksum; g.n_cols = p.NB; g.C = p.L; g.NB = p.NB; g.S = p.S;
  g.div = sqrtf((float)ICSA_D);
  g.n_split = lg_split(p.NB, p.NB, p.BH);
  const int NBp = compressed_nbp(p.NB), n_rt = (p.NB + LG_ROWS - 1) / LG_ROWS;
  const VmeanParams vm{p.vsum, p.vmt, p.NB, NBp, p.S, n_rt};
  const int n_vm = (NBp / 64 + g.n_split - 1) / g.n_split;
  hipLaunchKernelGGL(icsa_split3_gemm_kernel<true>, dim3(n_rt + n_vm, g.n_split, p.BH), dim3(256), 0, stream, g, vm);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int64_t rows = (int64_t)p.BH * p.NB;
  const dim3 sgrid((unsigned)((rows + 3) / 4));
  if (p.NB <= 256)
    hipLaunchKernelGGL(icsa_compressed_stats_kernel<4>, sgrid, dim3(256), 0, stream, p);
  else if (p.NB <= 512)
    hipLaunchKernelGGL(icsa_compressed_stats_kernel<8>, sgrid, dim3(256), 0, stream, p);
  else if (p.NB <= 1024)
    hipLaunchKernelGGL(icsa_compressed_stats_kernel<16>, sgrid, dim3(256), 0, stream, p);
  else if (p.NB <= 2048)
    hipLaunchKernelGGL(icsa_compressed_stats_kernel<32>, sgrid, dim3(256), 0, stream, p);
  else if (p.NB <= 2560)                             // configuration 5: NB = 2363
    hipLaunchKernelGGL(icsa_compressed_stats_kernel<40>, sgrid, dim3(256), 0, stream, p);
  else
    hipLaunchKernelGGL(icsa_compressed_stats_kernel<64>, sgrid, dim3(256), 0, stream, p);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(icsa_compressed_rows_kernel, dim3(nt, p.BH), dim3(512), 0, stream, p, NBp);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------------------
// (d) per-head selection: source column mass -> top-topK, sharpness ranking, new-KV map
//
// Both rankings by counting: an element's place in the descending order is the number of larger
// keys (the keys hold the index, so no two are equal).  Workgroup = 64 elements, all keys of the
// list in LDS, a wave per quarter of the list (every lane reads the same key: LDS broadcasts),
// so a list of any length is ranked by as many workgroups as it has 64 elements.  A bitonic
// sort in one workgroup per list took a barrier per step, 55 of them at 1,024 blocks: 18.5 us at
// 5 heads, now 7.2; 2 heads, 128 blocks 7.8 -> 3.1 us (layer 107 -> 102 us).
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ unsigned long long rank_key(float v, int idx) {
  return ((unsigned long long)f2key(v) << 32) | (unsigned long long)(0xffffffffu - (uint32_t)idx);
}

#define SEL_ELEMS 64

// Place of element e0 + threadIdx.x % 64 among the n keys (threads below 64; e0 + thread < n).
__device__ __forceinline__ int rank_of(const unsigned long long* keys, int n, int e0, int (*cnt)[SEL_ELEMS]) {
  const int l = threadIdx.x & 63, quarter = threadIdx.x >> 6;
  const int per = (n + 3) / 4, i1 = min(n, (quarter + 1) * per);
  const unsigned long long mine = e0 + l < n ? keys[e0 + l] : ~0ull;
  int larger = 0;
#pragma unroll 8
  for (int i = quarter * per; i < i1; ++i) larger += keys[i] > mine ? 1 : 0;
  cnt[quarter][l] = larger;
  __syncthreads();
  return cnt[0][l] + cnt[1][l] + cnt[2][l] + cnt[3][l];
}

// blockIdx.y < n_src_wg: 64 source blocks (and, in the first, the new-KV map but for the
// selected blocks); the rest: 64 query blocks by sharpness.
__global__ void __launch_bounds__(256) icsa_select_kernel(SelectParams p, int n_src_wg) {
  __shared__ unsigned long long keys[ICSA_MAX_SORT];
  __shared__ int cnt[4][SEL_ELEMS];
  const int bh = blockIdx.x, tid = threadIdx.x;
  const int NB = p.NB, n_t = p.n_t, n_s = p.n_s;
  if ((int)blockIdx.y >= n_src_wg) {                       // uniform for the workgroup
    const int e0 = SEL_ELEMS * (blockIdx.y - n_src_wg);
    for (int i = tid; i < NB; i += 256) keys[i] = rank_key(p.sharp[(int64_t)bh * NB + i], i);
    __syncthreads();
    const int r = rank_of(keys, NB, e0, cnt);
    if (tid < SEL_ELEMS && e0 + tid < NB) p.order[(int64_t)bh * NB + r] = e0 + tid;
    return;
  }
  const int e0 = SEL_ELEMS * blockIdx.y;
  int* kvmap = p.kvmap + (int64_t)bh * p.NKV;
  // new-KV block j -> source block: target blocks, then the selected source blocks in
  // ranked order, then zero padding (-1).  With t % 64 != 0 the blocks from n_t on straddle
  // two of these (the kernels take the first t % 64 rows from the block before).
  if (blockIdx.y == 0)
    for (int j = tid; j < p.NKV; j += 256) {
      const int r = j - n_t;
      if (r < 0) kvmap[j] = j;
      else if (r >= p.topK) kvmap[j] = -1;
      else if (p.inject_sel) kvmap[j] = n_t + p.sel[(int64_t)bh * p.topK + r];
    }
  // column mass of source key blocks over target query blocks: the per-strip partial
  // sums of the strip kernel, added in strip order
  const int n_ts = (n_t + ICSA_BLOCK - 1) / ICSA_BLOCK;
  const float* part = p.colpart + (int64_t)bh * n_ts * n_s;
  for (int j = tid; j < n_s; j += 256) {
    float s = 0.f;
#pragma unroll 8
    for (int st = 0; st < n_ts; ++st) s += part[(int64_t)st * n_s + j];
    if (j - e0 >= 0 && j - e0 < SEL_ELEMS) p.src_score[(int64_t)bh * n_s + j] = s;
    keys[j] = rank_key(s, j);
  }
  if (p.inject_sel) return;
  __syncthreads();
  const int r = rank_of(keys, n_s, e0, cnt);
  if (tid < SEL_ELEMS && e0 + tid < n_s && r < p.topK) {
    p.sel[(int64_t)bh * p.topK + r] = e0 + tid;
    if (n_t + r < p.NKV) kvmap[n_t + r] = n_t + e0 + tid;
  }
}

hipError_t launch_select(const SelectParams& p, hipStream_t stream) {
  if (p.n_s > ICSA_MAX_SORT || p.NB > ICSA_MAX_SORT) return hipErrorInvalidValue;
  const int n_src_wg = std::max(1, (p.n_s + SEL_ELEMS - 1) / SEL_ELEMS);
  const int n_q_wg = p.inject_order ? 0 : (p.NB + SEL_ELEMS - 1) / SEL_ELEMS;
  hipLaunchKernelGGL(icsa_select_kernel, dim3(p.BH, n_src_wg + n_q_wg), dim3(256), 0, stream, p, n_src_wg);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------------------
// (e) level-3: per query block, top_k new-KV blocks by QCsum . KCsum (fp32), ascending list.
//     Scores: the fp32-accurate split-bf16 product of (a) on the raw sums (128 query blocks
//     of the list per workgroup, a range of the new-KV blocks), written to a scratch row
//     per query block.  Selection: one wave per query block, bisection over the float keys
//     (ballot counts), then compaction in ascending block order.  The interval bound of the
//     sparse kernel (largest |KC_j| of each head) takes the launch's last workgroups: as a
//     launch of its own it cost 4-5 us.
// ---------------------------------------------------------------------------------------
// Workgroup y of G per head: rows j = 16 (y + G i) + r, r = 0 .. 15 (i = 0, 1, ...); 16 lanes
// per row, one 16-byte chunk each, the squared norm summed over the 16 lanes with lane
// shuffles; the workgroup maximum goes through an LDS atomic (non-negative floats order like
// their bit patterns).
__device__ __forceinline__ void kc_bound(const Level3Params& p, int bh, int y, int G) {
  __shared__ unsigned mx;
  const int r = threadIdx.x >> 4, ch = threadIdx.x & 15;
  if (threadIdx.x == 0) mx = 0u;
  __syncthreads();
  float best = 0.f;
  for (int j0 = 16 * y; j0 < p.NKV; j0 += 16 * G) {
    const int j = j0 + r;
    float n2 = 0.f;
    if (j < p.NKV) {
      const bf16x8 v = *reinterpret_cast<const bf16x8*>(p.kc + ((int64_t)bh * p.NKVp + j) * ICSA_D + 8 * ch);
#pragma unroll
      for (int e = 0; e < 8; ++e) n2 = fmaf(bf2f(v[e]), bf2f(v[e]), n2);
    }
#pragma unroll
    for (int w = 1; w < 16; w <<= 1) n2 += __shfl_xor(n2, w);
    best = fmaxf(best, n2);
  }
  atomicMax(&mx, __float_as_uint(best));
  __syncthreads();
  if (threadIdx.x == 0) p.bound[(int64_t)bh * G + y] = sqrtf(__uint_as_float(mx));
}

template <int VPL>   // scores per lane: NKV <= 64 * VPL
__global__ void __launch_bounds__(256) icsa_level3_select_kernel(Level3Params p, int n_sel_wg) {
  if ((int)blockIdx.x >= n_sel_wg) {
    const int G = kc_bound_groups(p.NKV), u = blockIdx.x - n_sel_wg;
    kc_bound(p, u / G, u % G, G);
    return;
  }
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + w;          // over BH * n_rows
  if (row >= (int64_t)p.BH * p.n_rows) return;
  const int NKV = p.NKV, k = p.top_k;
  const float* srow = p.scores + row * NKV;
  // unconditional loads from a clamped place: a condition around each made VPL branches, each
  // waiting for the load before it (5 heads, 1,024 blocks 13.5 -> 11.5 us, 40 heads 34.4 -> 31.3)
  float score[VPL];
#pragma unroll
  for (int u = 0; u < VPL; ++u) score[u] = srow[min(lane + 64 * u, NKV - 1)];
  uint32_t key[VPL];
#pragma unroll
  for (int u = 0; u < VPL; ++u) key[u] = lane + 64 * u < NKV ? f2key(score[u]) : 0u;   // 0 is below every real key
  const int nu = (NKV + 63) / 64;
  const uint32_t lo = kth_largest_key<VPL>(key, k, nu);
  int cgt = 0;
#pragma unroll
  for (int g = 0; g < VPL; g += 4)
    if (g < nu) {
#pragma unroll
      for (int u = g; u < g + 4; ++u) cgt += wave_count(key[u] > lo);
    }
  const int need_eq = k - cgt;
  const unsigned long long lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  int seen_eq = 0, taken = 0;
  int* out = p.idx + row * k;
#pragma unroll
  for (int g = 0; g < VPL; g += 4)
    if (g < nu) {
#pragma unroll
      for (int u = g; u < g + 4; ++u) {
        const int j = lane + 64 * u;
        const bool gt = key[u] > lo;
        const bool eq = key[u] == lo && j < NKV;
        const unsigned long long eqm = __ballot(eq);
        const int eq_before = seen_eq + __popcll(eqm & lt_mask);
        const bool take = gt || (eq && eq_before < need_eq);
        const unsigned long long tm = __ballot(take);
        const int pos = taken + __popcll(tm & lt_mask);
        if (take && pos < k) out[pos] = j;
        seen_eq += __popcll(eqm);
        taken += __popcll(tm);
      }
    }
}

hipError_t launch_level3(const Level3Params& p, hipStream_t stream) {
  if (!p.given && (p.NKV > ICSA_MAX_NKV || p.top_k > p.NKV || p.top_k < 1)) return hipErrorInvalidValue;
  if (p.n_rows <= 0) return hipSuccess;
  if (!p.given) {
    Split3Gemm g;
    g.A = p.qsum; g.rows = p.rows; g.rows_stride = p.rows_stride; g.rows_offset = p.rows_offset;
    g.a_rows = p.NQsrc; g.n_rows = p.n_rows; g.B = p.kc32; g.n_cols = p.NKV; g.C = p.scores;
    g.NB = 0; g.S = 0; g.div = 1.f; g.n_split = lg_split(p.n_rows, p.NKV, p.BH);
    hipLaunchKernelGGL(icsa_split3_gemm_kernel<false>, dim3((p.n_rows + LG_ROWS - 1) / LG_ROWS, g.n_split, p.BH),
                       dim3(256), 0, stream, g, VmeanParams{});
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  const int n_sel_wg = p.given ? 0 : (int)(((int64_t)p.BH * p.n_rows + 3) / 4);
  const int n_wg = n_sel_wg + (p.bound ? p.BH * kc_bound_groups(p.NKV) : 0);
  if (n_wg == 0) return hipSuccess;
  const dim3 grid((unsigned)n_wg);
  if (p.NKV <= 256)
    hipLaunchKernelGGL(icsa_level3_select_kernel<4>, grid, dim3(256), 0, stream, p, n_sel_wg);
  else if (p.NKV <= 512)
    hipLaunchKernelGGL(icsa_level3_select_kernel<8>, grid, dim3(256), 0, stream, p, n_sel_wg);
  else if (p.NKV <= 1024)
    hipLaunchKernelGGL(icsa_level3_select_kernel<16>, grid, dim3(256), 0, stream, p, n_sel_wg);
  else
    hipLaunchKernelGGL(icsa_level3_select_kernel<32>, grid, dim3(256), 0, stream, p, n_sel_wg);
  return hipGetLastError();
}
