// Backward of the sparse piecewise attention with the first-order interval approximation.
//
// Reference: sparse_piecewise_attn_1st_intervals_bwd_kernel (triton_kernels.py:265-486) and
// SparsePiecewiseAttn1stIntervalsFunction.backward (:541-598).  With D = rowsum(dO * O)
// and P = exp2(s - lse) (scores in log2-scaled units, lse saved by the forward):
//   exact blocks (the top_k selected per query block):
//     dS = P (dO V^T - D);  dq += dS K scale;  dk += dS^T q scale;  dv += P^T dO
//   interval blocks (every unselected block c < NKV, block sums KC / VC):
//     s = q KC^T scale / 64;  dS = P (dO VC^T - 64 D);  dq += dS KC scale / 64;
//     each key row of block c gets dKC_c / 64 = (dS^T q)_c scale / 64 and dVC_c = (P^T dO)_c.
//
// The reference adds dk / dv (and dq) with fp32 atomics, so its sums depend on timing.  Here
// every gradient is a fixed-order sum:
//   * bw_dq: one workgroup per query block (dq rows are owned);
//   * bw_dkv<true>: one workgroup per (chunk of 64 compressed blocks,
//     range of query blocks) -> interval partials dKC / dVC, summed later in split order;
//   * bw_dkv<false>: one workgroup per key block; it walks the query
//     blocks that selected it in ascending order (from the selection bitmap) and adds the
//     interval partials in its epilogue.
//
// MFMA orientation (v_mfma_f32_32x32x16_bf16, the tile toolkit of the forward):
//   dq kernel: S^T = K Q^T and dP^T = V dO^T with the K / V rows in LDS and Q, dO of the
//     wave's 32 queries in registers; dQ^T += K^T dS^T with K^T (kv_slot order) in LDS.
//   dk / dv kernel, the roles swapped: S = Q K^T and dP = dO V^T with the Q / dO rows in
//     LDS and K, V of the wave's 32 keys in registers; dV^T += dO^T P and dK^T += Q^T dS
//     with the transposed Q / dO tiles in LDS.
// Ragged lengths (the Triton host): NQ = cdiv(TQ, 64), NKV = cdiv(TKV, 64).  Rows past TQ
// and TKV read as zero (q, dO, lse, D, k, v: the tensor descriptors' zero fill), keys past
// TKV are masked out of the exact part (triton_kernels.py:348), and gradient rows past TQ /
// TKV are not stored.
// P and dS are rounded to bf16 for the MFMA (the reference rounds P for dv and uses fp32
// dots for dq / dk).
//
// Workgroup = 4 waves on one 64 x 64 pair of blocks at a time: wave w computes the quadrant of
// S and dP of 32 keys (or queries) it keeps in registers, w % 2, by 32 rows of the tile in LDS,
// w / 2, and adds the products over its own quadrant.  At 228-256 registers two such
// workgroups (at most 76 KB of LDS each) share a CU, so one wave's elementwise work and LDS
// reads run beside another's MFMAs; with two waves per workgroup, 64 rows each and 308-412
// registers, every SIMD held a single wave.  Measured at 40 heads, 7,800 tokens, 12 of 122
// blocks, against that: dq 375 -> 298 us, dk / dv exact 500 -> 355 us, interval 90 -> 61 us
// (4 heads, 2,048 tokens: 14.6 -> 11.7, 28 -> 21, 22 -> 10 us).  A step of the exact part then
// takes 3,700 cycles with two workgroups on the CU, 55 % of them MFMA; about a third of a
// workgroup's time is its start (first tiles, K and V) and its end (sums of the halves,
// output), which is what bounds it at 12 steps.  Copies: all tiles from L2 5 % faster, no
// tiles at all 17 %; no elementwise masks: the same.
// Waits: the tile DMA is inline assembly (lds_dma16); behind the builtin the compiler waited
// for the next step's tiles (vmcnt(0)) before every step's transposing reads; settle_frags keeps its
// waits for the register operands out of the loop (interval 70 -> 61 us).
#include "attn_tile.h"
#include "icsa_kernels.h"

#define BW_THREADS 256
#define BW_MAX_TOPK 512
#define BW_MAX_CHUNKS 32                 // NKV <= 2048
#define BW_MAX_NQ 4096
#define BW_STAGE_BYTES (32 * O_LDS_STRIDE * 4)   // one wave's fp32 staging rows

// ------------------------------------------------------------------------------------------
// prep: D = rowsum(dO * O) per query row and the selection bitmap of each query block
// ------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) icsa_sparse_bwd_rows_kernel(SparseBwdParams p) {
  __shared__ unsigned long long sel[BW_MAX_CHUNKS];
  const int i = blockIdx.x, bh = blockIdx.y;
  const int b = bh / p.H, h = bh % p.H;
  const int t = threadIdx.x;
  if (t < p.nc) sel[t] = 0ull;
  __syncthreads();
  const int* row = p.idx + ((int64_t)bh * p.NQ + i) * p.top_k;
  for (int u = t; u < p.top_k; u += 256) {
    const int j = row[u];
    if (j >= 0 && j < p.NKV) atomicOr(&sel[j >> 6], 1ull << (j & 63));
  }
  const int r = t >> 2, qq = t & 3;               // row, quarter of D (32 elements)
  const int tok = i * ICSA_BLOCK + r;
  float acc = 0.f;
  if (tok < p.TQ) {                               // rows past TQ: D = 0
  const bf16* dor = p.dout + (int64_t)b * p.do_sb + (int64_t)h * p.do_sh + (int64_t)tok * p.do_st + 32 * qq;
  const bf16* orr = p.out + (int64_t)b * p.o_sb + (int64_t)h * p.o_sh + (int64_t)tok * p.o_st + 32 * qq;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const bf16x8 a = *reinterpret_cast<const bf16x8*>(dor + 8 * c);
    const bf16x8 o = *reinterpret_cast<const bf16x8*>(orr + 8 * c);
#pragma unroll
    for (int e = 0; e < 8; ++e) acc = fmaf((float)a[e], (float)o[e], acc);
  }
  }
  acc += __shfl_xor(acc, 1, 64);
  acc += __shfl_xor(acc, 2, 64);
  if (qq == 0) p.dvec[(int64_t)bh * p.NQ * ICSA_BLOCK + tok] = acc;   // D rows padded to NQ * 64
  __syncthreads();
  if (t < p.nc) p.selbits[((int64_t)bh * p.NQ + i) * p.nc + t] = sel[t];
}

// The selection bitmap by key block, for 64 key blocks (ch) of one head: the exact dk / dv
// workgroups walk their query blocks with scalar loads and bit scans alone, instead of listing
// them in LDS between two barriers.  64 x 64 bits at a time: lane l holds query block 64 w +
// l's word, then key block 64 ch + l's.
__device__ __forceinline__ void bw_transpose_bits(const SparseBwdParams& p, int bh, int ch) {
  const int t = threadIdx.x, lane = t & 63, n_qw = (p.NQ + 63) / 64;
  for (int w = t >> 6; w < n_qw; w += 4) {
    const int i = 64 * w + lane;
    const unsigned long long word = i < p.NQ ? p.selbits[((int64_t)bh * p.NQ + i) * p.nc + ch] : 0ull;
    unsigned long long mine = 0ull;
#pragma unroll 8
    for (int j = 0; j < 64; ++j) {
      const unsigned long long b = __ballot((word >> j) & 1ull);
      if (lane == j) mine = b;
    }
    const int key = ch * ICSA_BLOCK + lane;
    if (key < p.NKV) p.seltr[((int64_t)bh * p.NKV + key) * n_qw + w] = mine;
  }
}

// ------------------------------------------------------------------------------------------
// Tile DMA.  A 16 KB row tile (64 rows x 128 dims, swizzled by rt_swz) is 16 LDS-DMA
// instructions, 4 for each of the four waves; each lands 1 KB at consecutive LDS addresses (lane
// l at +16 l), so the XOR swizzle is applied on the global side.  A step's tiles are the only
// loads in flight when a kernel waits for them (vmcnt(0)): the next step's tiles are issued
// after the workgroup barrier that follows, which also tells that all four waves are done with
// the buffer they overwrite (two buffers, one barrier per step).
// ------------------------------------------------------------------------------------------
#define BW_WAIT(n) asm volatile("s_waitcnt vmcnt(" #n ")" ::: "memory")

// A wave-uniform word that an earlier kernel wrote, through the scalar cache.
template <typename T>
__device__ __forceinline__ T uniform_word(const T* p) {
  return *(const __attribute__((address_space(4))) T*)(unsigned long long)p;
}

// Row tiles use the shared layout of attn_tile.h (rt_swz / rt_off).
#define BW_PF 3                 // MFMA operand read-ahead (steps)

// Byte offset of this lane's 16-byte chunk hl of tile row `row`; chunk 2 kk + hl is at that
// offset ^ (kk << 5) (the swizzle only flips chunk bits).
__device__ __forceinline__ int bw_row_off(int row, int hl) { return rt_off(row, hl) * 2; }

// Row tiles of one tensor of a head: block j's 64 rows.  What a tile needs is kept to a product
// and an add, and one select for the partial last block (rows past it lie outside the buffer
// range and land nothing: bw_fill_rows zeroes them once the tile's loads have completed): with the
// byte count worked out for each tile and generic LDS pointers, a step's two tiles took 145
// instructions and about 800 of its 3,400 cycles; now 91 (40 heads, 7,800 tokens: query-major launch
// 352 -> 341 us, exact key-major 368 -> 358 us at the best clock, forward and backward 993 -> 982).
struct BwSrc {
  unsigned long long base;
  long long block_bytes;
  int row_bytes, partial, n_partial;     // partial: index of the last block if it is not whole
  __device__ __forceinline__ BwSrc(const bf16* head, int64_t stride, int rows)
      : base((unsigned long long)head), block_bytes(stride * 2 * ICSA_BLOCK), row_bytes((int)(stride * 2)),
        partial(rows % ICSA_BLOCK ? rows / ICSA_BLOCK : -1) {
    const int64_t n = ((int64_t)(rows % ICSA_BLOCK - 1) * stride + ICSA_D) * 2;
    n_partial = n > 0x7fffffffLL ? 0x7fffffff : (int)n;
  }
  // one wave's quarter of block j's tile (rows 16 w .. 16 w + 15) to LDS address `tile`
  __device__ __forceinline__ void load(unsigned tile, int j, int wave, int lane) const {
    const unsigned long long a = base + (unsigned long long)(unsigned)j * (unsigned long long)block_bytes;
    u32x4 rs;
    rs[0] = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)a);
    rs[1] = (unsigned)__builtin_amdgcn_readfirstlane((int)((unsigned)(a >> 32) & 0xffffu));
    rs[2] = (unsigned)__builtin_amdgcn_readfirstlane(j == partial ? n_partial : 0x7fffffff);
    rs[3] = 0x00020000u;
    const unsigned dst = tile + 4096u * wave;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 16 * wave + 4 * i + (lane >> 4);
      lds_dma16(dst + 1024 * i, r * row_bytes + (((lane & 15) ^ rt_swz(r)) << 4), rs);
    }
  }
};

// Zero this wave's rows >= valid of a row tile (the bytes its DMA lanes would have landed).
__device__ __forceinline__ void bw_fill_rows(unsigned char* tile, int valid, int wave, int lane) {
  if (valid >= ICSA_BLOCK) return;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 16 * wave + 4 * i + (lane >> 4);
    if (r >= valid) *reinterpret_cast<u32x4*>(tile + r * ICSA_D * 2 + (lane & 15) * 16) = u32x4{0u, 0u, 0u, 0u};
  }
}

// s = X Bx, d = Y By over 128 dims for 32 rows of the tiles x and y (this lane's row at byte
// offset `ro`): 16 MFMAs, alternating, operands read BW_PF steps ahead.
__device__ __forceinline__ void bw_scores(floatx16& s, floatx16& d, const unsigned char* x, const unsigned char* y,
                                          int ro, const bf16x8 bx[8], const bf16x8 by[8]) {
  auto ld = [&](int t) -> bf16x8 {
    return *reinterpret_cast<const bf16x8*>(((t & 1) ? y : x) + (ro ^ ((t >> 1) << 5)));
  };
  bf16x8 a[16];
#pragma unroll
  for (int t = 0; t < BW_PF; ++t) a[t] = ld(t);
  __builtin_amdgcn_sched_barrier(0);
  s = d = floatx16{};
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    if (t + BW_PF < 16) a[t + BW_PF] = ld(t + BW_PF);
    if (t & 1) d = mfma32x32x16(a[t], by[t >> 1], d);
    else s = mfma32x32x16(a[t], bx[t >> 1], s);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// o[ND d-subtiles] += X^T P over NM 16-row steps from m0 of row tile X (p[m]: the bf16 B
// operand of step m0 + m, straight from the score accumulators).  tro: the transposing read's
// offset for the first d-subtile; the next 32 dims are 4 chunks on, byte bit 6 of the swizzled
// offset flipped (64 dims: bit 7).
template <int ND, int NM>
__device__ __forceinline__ void bw_accum(floatx16* o, const unsigned char* tile, int tro, int m0,
                                         const bf16x8* p) {
  constexpr int N = ND * NM;
  const unsigned char* base = tile + m0 * 16 * ICSA_D * 2;
  auto ld = [&](int t) -> bf16x8 {
    const int off = tro ^ ((t % ND) << 6);
    const int st = (t / ND) * 16 * ICSA_D * 2;
    const rt_v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((rt_lds_v4s)(base + off + st));
    const rt_v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((rt_lds_v4s)(base + rt_tr_hi<false>(off) + st));
    const short __attribute__((ext_vector_type(8))) a8 = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(bf16x8, a8);
  };
  bf16x8 a[N];
#pragma unroll
  for (int t = 0; t < BW_PF; ++t) a[t] = ld(t);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int t = 0; t < N; ++t) {
    if (t + BW_PF < N) a[t + BW_PF] = ld(t + BW_PF);
    o[t % ND] = mfma32x32x16(a[t], p[t / ND], o[t % ND]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Adds the accumulators of a wave pair (same rows / keys, the two halves of the summed
// dimension) through LDS and leaves mul * sum as rows for store_rows: each wave hands over the
// d-subtiles that the other one adds up.
__device__ __forceinline__ void bw_reduce_stage(float* o_lds, const floatx16 o[4], int half, float mul) {
  const int lane = threadIdx.x & 63, li = lane & 31;
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i)
      o_lds[li * O_LDS_STRIDE + 32 * (2 * (half ^ 1) + d) + acc_row(i, lane)] = half ? o[d][i] : o[2 + d][i];
  __syncthreads();
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float* x = &o_lds[li * O_LDS_STRIDE + 32 * (2 * half + d) + acc_row(i, lane)];
      *x = ((half ? o[2 + d][i] : o[d][i]) + *x) * mul;
    }
  __syncthreads();
}

// ------------------------------------------------------------------------------------------
// dq: one workgroup per query block.  Steps t = 0 .. n_ex + nc - 1: the valid selected
// blocks, then the interval chunks.  Per step the K and V rows (8 DMA per wave) land in
// one of two buffers while the other step's S^T = K Q^T, dP^T = V dO^T and
// dQ^T += K^T dS^T (K^T read transposed from the K rows) run.  Wave w: queries
// 32 (w % 2) .. + 31 in registers, keys 32 (w / 2) .. + 31 of each step.
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ void bw_dq(const SparseBwdParams& p, unsigned char* smem_q, int work) {
  const int bh = work / p.NQ, qb = work % p.NQ;
  const int b = bh / p.H, h = bh % p.H;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int li = lane & 31, hl = lane >> 5;
  const int qh = wave & 1, kh = wave >> 1;
  const int qtok0 = qb * ICSA_BLOCK + 32 * qh;

  const bf16* kb = p.k + (int64_t)b * p.k_sb + (int64_t)h * p.k_sh;
  const bf16* vb = p.v + (int64_t)b * p.v_sb + (int64_t)h * p.v_sh;
  const bf16* kcb = p.kcb + (int64_t)bh * p.NKVp * ICSA_D;
  const bf16* vcb = p.vcb + (int64_t)bh * p.NKVp * ICSA_D;
  // Steps: the listed blocks in list order (out-of-range entries are zero blocks without a
  // gradient: skipped), then chunk ch as block -1 - ch.  Looked up one step ahead.
  const int* row = p.idx + ((int64_t)bh * p.NQ + qb) * p.top_k;
  const unsigned long long* selw = p.selbits + ((int64_t)bh * p.NQ + qb) * p.nc;
  int at = 0;
  auto next = [&]() -> int {
    while (at < p.top_k) {
      const int j = uniform_word(row + at++);
      if (j >= 0 && j < p.NKV) return j;
    }
    return p.top_k - 1 - at++;                         // -1 - chunk
  };
  const int done = -1 - p.nc;
  // real key rows of an exact step (the last block of a ragged TKV is partial)
  auto key_rows = [&](int j) -> int { return j < 0 ? ICSA_BLOCK : min(ICSA_BLOCK, p.TKV - j * ICSA_BLOCK); };
  const BwSrc k_src(kb, p.k_st, p.TKV), v_src(vb, p.v_st, p.TKV);
  const BwSrc kc_src(kcb, ICSA_D, p.NKVp), vc_src(vcb, ICSA_D, p.NKVp);
  const unsigned lds = lds_u32(smem_q);
  // buffer u: K rows at 2 u tiles, V rows at 2 u + 1
  auto issue = [&](int t, int j) {
    const unsigned kt = lds + (t & 1) * 2 * K_TILE_BYTES;
    if (j >= 0) {
      k_src.load(kt, j, wave, lane);
      v_src.load(kt + K_TILE_BYTES, j, wave, lane);
    } else {
      kc_src.load(kt, -1 - j, wave, lane);
      vc_src.load(kt + K_TILE_BYTES, -1 - j, wave, lane);
    }
  };
  int j = next();                                      // at least one chunk
  issue(0, j);
  const int q_valid = max(0, min(32, p.TQ - qtok0));  // this wave's real query rows
  bf16x8 qf[8], dof[8];
  load_q_frags(qf, p.q + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh + (int64_t)qtok0 * p.q_st, p.q_st, q_valid);
  load_q_frags(dof, p.dout + (int64_t)b * p.do_sb + (int64_t)h * p.do_sh + (int64_t)qtok0 * p.do_st, p.do_st,
               q_valid);
  float lse = li < q_valid ? p.lse[(int64_t)bh * p.TQ + qtok0 + li] : 0.f;
  float dd = p.dvec[(int64_t)bh * p.NQ * ICSA_BLOCK + qtok0 + li];
  int tro[4];
  rt_tr_offsets<false>(tro, lane);
  const int ro = bw_row_off(32 * kh + li, hl);

  settle_frags(qf);
  settle_frags(dof);
  asm volatile("" : "+v"(lse), "+v"(dd));

  floatx16 dq[4] = {};
  floatx16 s, dp;
  bf16x8 dsf[2];
  const float c64 = p.scale_log2 * (1.0f / 64.0f);
  for (int t = 0; j != done; ++t) {
    const int kvalid = key_rows(j), jn = next();
    BW_WAIT(0);                                        // step t's tiles, the only loads in flight
    if (kvalid < ICSA_BLOCK) {                         // zero key / value rows past TKV
      bw_fill_rows(smem_q + (t & 1) * 2 * K_TILE_BYTES, kvalid, wave, lane);
      bw_fill_rows(smem_q + (t & 1) * 2 * K_TILE_BYTES + K_TILE_BYTES, kvalid, wave, lane);
    }
    ATT_BARRIER();                                     // step t complete; step t - 1's buffer read by all waves
    if (jn != done) issue(t + 1, jn);                  // into that buffer
    const unsigned char* ks = smem_q + (t & 1) * 2 * K_TILE_BYTES;
    bw_scores(s, dp, ks, ks + K_TILE_BYTES, ro, qf, dof);              // S^T[key][query], dP^T
    // masked keys (past TKV; a chunk's selected blocks and blocks >= NKV) as one word: element
    // e is bit 8 (e / 4) + e % 4 of the word's bits from 4 hl + 32 kh on
    unsigned long long mb;
    float c, dmul, dsmul;
    if (j >= 0) {
      mb = kvalid < ICSA_BLOCK ? ~0ull << kvalid : 0ull;
      c = p.scale_log2; dmul = 1.f; dsmul = 1.f;
    } else {                                           // unselected block sums: score / 64, dS / 64
      const int ch = -1 - j;
      mb = uniform_word(selw + ch);
      const int n_real = p.NKV - ch * ICSA_BLOCK;
      if (n_real < ICSA_BLOCK) mb |= ~0ull << n_real;
      c = c64; dmul = 64.f; dsmul = 1.0f / 64.0f;
    }
    if (mb == 0ull && j >= 0) {                      // the common case: a whole exact block
#pragma unroll
      for (int e = 0; e < 16; ++e)
        dsf[e >> 3][e & 7] = (bf16)(__builtin_amdgcn_exp2f(fmaf(s[e], c, -lse)) * (dp[e] - dd));
    } else {
      const unsigned wd = (unsigned)(mb >> (4 * hl + 32 * kh));
      const float ddm = dmul * dd;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const unsigned keep = ~(unsigned)((int)(wd << (31 - 8 * (e >> 2) - (e & 3))) >> 31);
        const float x = __builtin_amdgcn_exp2f(fmaf(s[e], c, -lse));
        const float pr = __uint_as_float(__float_as_uint(x) & keep);
        dsf[e >> 3][e & 7] = (bf16)(pr * (dp[e] - ddm) * dsmul);
      }
    }
    bw_accum<4, 2>(dq, ks, tro[0], 2 * kh, dsf);          // dQ^T += K^T dS^T
    j = jn;
  }

  // ---- epilogue: dq = scale * (sum over both key halves) ----
  __syncthreads();
  float* o_lds = reinterpret_cast<float*>(smem_q + qh * BW_STAGE_BYTES);
  bw_reduce_stage(o_lds, dq, kh, p.scale);
  if (kh == 1) return;
  AlphaView none;
  none.p = nullptr; none.scalar = 0.f; none.sb = none.ss = none.sh = none.sd = 0; none.dtype = ICSA_DT_F32;
  store_rows(o_lds, p.dq, b, h, qtok0, q_valid, nullptr, none);
}

// ------------------------------------------------------------------------------------------
// dk / dv: kInterval = true -> interval partials per (chunk, query range);
//          kInterval = false -> exact part per key block + the summed partials.
// Per visited query block: its Q and dO rows plus lse (wave 0) / D (wave 1) land in one of two
// buffers while the previous block's S = Q K^T, dP = dO V^T, dV^T += dO^T P and
// dK^T += Q^T dS run (Q^T, dO^T read transposed from the rows).  Wave w: keys
// 32 (w % 2) .. + 31 in registers, rows 32 (w / 2) .. + 31 of each query block.  dK sums the
// wave's own rows over all 128 dims (the two row halves are added at the end); dV takes all
// 64 rows for dims 64 (w / 2) .. + 63, with the other half's P read from LDS: keeping both
// over all dims would need more than 256 registers.
// ------------------------------------------------------------------------------------------
#define BWKV_BUF_BYTES (2 * K_TILE_BYTES + 2 * 64 * 4)      // Q rows, dO rows, lse, D
#define BWKV_P_BYTES (4 * 2 * 1024)                         // each wave's P: two 16-row operands
#define BW_LDS_BYTES (2 * BWKV_BUF_BYTES + BWKV_P_BYTES + 2 * ICSA_D * 4)
#define BWKV_SUM_AHEAD 16                                   // interval partials requested together

template <bool kInterval>
__device__ __forceinline__ void bw_dkv(const SparseBwdParams& p, unsigned char* smem_dyn, int work) {
  unsigned char* pbuf = smem_dyn + 2 * BWKV_BUF_BYTES;
  float* ivec = reinterpret_cast<float*>(pbuf + BWKV_P_BYTES);    // [2][128] interval sums

  int bh, blk, split = 0;
  if (kInterval) {
    bh = work / (p.nc * p.nsplit);
    const int rem = work % (p.nc * p.nsplit);
    split = rem / p.nc;                                // neighbours read the same query blocks
    blk = rem % p.nc;                                  // chunk of 64 compressed blocks
  } else {
    bh = work / p.NKV;
    blk = work % p.NKV;                                // key block
  }
  const int b = bh / p.H, h = bh % p.H;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int li = lane & 31, hl = lane >> 5;
  const int kh = wave & 1, rh = wave >> 1;
  const int key0 = blk * ICSA_BLOCK + 32 * kh;         // this wave's first key (or compressed block)

  int tro[4];
  rt_tr_offsets<false>(tro, lane);
  const int ro = bw_row_off(32 * rh + li, hl);

  const int ckey = key0 + li;                          // interval: this lane's compressed block
  const float cexp = kInterval ? p.scale_log2 * (1.0f / 64.0f) : p.scale_log2;
  const float dmul = kInterval ? 64.0f : 1.0f;

  const bf16* qb0 = p.q + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh;
  const bf16* dob0 = p.dout + (int64_t)b * p.do_sb + (int64_t)h * p.do_sh;
  const float* rowvec = wave == 0 ? p.lse + (int64_t)bh * p.TQ : p.dvec + (int64_t)bh * p.NQ * ICSA_BLOCK;
  // Query blocks to visit, ascending, looked up one ahead: the interval's range (with the
  // chunk's selection word of each), or the set bits of the key block's row of the bitmap.
  const int i_end = kInterval ? min(p.NQ, (split + 1) * p.qb_per_split) : p.NQ;
  const int n_qw = (p.NQ + 63) / 64;
  const unsigned long long* bits = kInterval ? p.selbits + (int64_t)bh * p.NQ * p.nc + blk
                                             : p.seltr + ((int64_t)bh * p.NKV + blk) * n_qw;
  int at = kInterval ? split * p.qb_per_split : 0;     // next query block / current word
  unsigned long long cur = kInterval ? 0ull : uniform_word(bits);
  auto next = [&]() -> int {
    if (kInterval) {
      if (at >= i_end) return -1;
      cur = uniform_word(bits + (int64_t)at * p.nc);
      return at++;
    }
    while (cur == 0ull) {
      if (++at >= n_qw) return -1;
      cur = uniform_word(bits + at);
    }
    const int i = 64 * at + __builtin_ctzll(cur);
    cur &= cur - 1ull;
    return i;
  };
  const BwSrc q_src(qb0, p.q_st, p.TQ), do_src(dob0, p.do_st, p.TQ);
  const unsigned lds = lds_u32(smem_dyn);
  auto issue = [&](int n, int i) {
    const unsigned buf = lds + (n & 1) * BWKV_BUF_BYTES;
    q_src.load(buf, i, wave, lane);
    do_src.load(buf + K_TILE_BYTES, i, wave, lane);
    if (wave < 2)
      lds_dma4(buf + 2 * K_TILE_BYTES + wave * 256, lane * 4,
               dma_rsrc(rowvec + (int64_t)i * ICSA_BLOCK, min(ICSA_BLOCK, p.TQ - i * ICSA_BLOCK) * 4));
  };
  // Everything the prologue reads is requested before any of it is waited for: the first
  // tiles, the interval partials (exact part), K and V.
  int i = next();
  unsigned long long sel = cur;                        // interval: block i's word
  if (i >= 0) issue(0, i);
  float px[BWKV_SUM_AHEAD];
  const float* part = kInterval ? nullptr : (tid < ICSA_D ? p.dkc_part : p.dvc_part) +
                                                ((int64_t)bh * p.NKVp + blk) * ICSA_D + (tid & 127);
  const int64_t part_st = (int64_t)p.B * p.H * p.NKVp * ICSA_D;
  auto load_parts = [&](int sp0) {
#pragma unroll
    for (int u = 0; u < BWKV_SUM_AHEAD; ++u) px[u] = part[min(sp0 + u, p.nsplit - 1) * part_st];
  };
  if (!kInterval) load_parts(0);
  bf16x8 kf[8], vf[8];
  if (kInterval) {
    load_q_frags(kf, p.kcb + ((int64_t)bh * p.NKVp + key0) * ICSA_D, ICSA_D, 32);
    load_q_frags(vf, p.vcb + ((int64_t)bh * p.NKVp + key0) * ICSA_D, ICSA_D, 32);
  } else {                                             // keys past TKV read as zero
    const int kv = max(0, min(32, p.TKV - key0));
    load_q_frags(kf, p.k + (int64_t)b * p.k_sb + (int64_t)h * p.k_sh + (int64_t)key0 * p.k_st, p.k_st, kv);
    load_q_frags(vf, p.v + (int64_t)b * p.v_sb + (int64_t)h * p.v_sh + (int64_t)key0 * p.v_st, p.v_st, kv);
  }
  if (!kInterval) {                                    // interval sums of the block, in split order
    float sum = 0.f;
    for (int sp0 = 0;;) {
#pragma unroll
      for (int u = 0; u < BWKV_SUM_AHEAD; ++u)
        if (sp0 + u < p.nsplit) sum += px[u];
      sp0 += BWKV_SUM_AHEAD;
      if (sp0 >= p.nsplit) break;
      load_parts(sp0);
    }
    ivec[tid] = tid < ICSA_D ? sum * p.scale : sum;
  }
  settle_frags(kf);
  settle_frags(vf);

  floatx16 dk[4] = {}, dv[2] = {};
  floatx16 s, dp;
  bf16x8 pf[4], dsf[2];

  for (int n = 0; i >= 0; ++n) {
    // exact: a key past TKV (zero K and V rows) only reaches its own dk / dv row, not stored
    const bool on = !kInterval || (ckey < p.NKV && ((sel >> (32 * kh + li)) & 1ull) == 0ull);
    const int in = next();
    unsigned char* buf = smem_dyn + (n & 1) * BWKV_BUF_BYTES;
    BW_WAIT(0);                                      // block n's tiles, the only loads in flight
    const int qvalid = min(ICSA_BLOCK, p.TQ - i * ICSA_BLOCK);
    if (qvalid < ICSA_BLOCK) {                       // zero Q / dO rows and lse / D past TQ
      bw_fill_rows(buf, qvalid, wave, lane);
      bw_fill_rows(buf + K_TILE_BYTES, qvalid, wave, lane);
      if (wave < 2 && lane >= qvalid) reinterpret_cast<float*>(buf + 2 * K_TILE_BYTES + wave * 256)[lane] = 0.f;
    }
    ATT_BARRIER();                                   // block n complete; block n - 1's buffer and P read by all
    if (in >= 0) issue(n + 1, in);                   // into that buffer
    const unsigned char* dos = buf + K_TILE_BYTES;
    bw_scores(s, dp, buf, dos, ro, kf, vf);          // S[row][key], dP
    const float* lse_l = reinterpret_cast<const float*>(buf + 2 * K_TILE_BYTES) + 32 * rh + 4 * hl;
#pragma unroll
    for (int g = 0; g < 4; ++g) {                    // acc_row(4 g + x, lane) = 8 g + 4 hl + x
      const floatx4 l4 = *reinterpret_cast<const floatx4*>(lse_l + 8 * g);
      const floatx4 d4 = *reinterpret_cast<const floatx4*>(lse_l + 64 + 8 * g);
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int e = 4 * g + x;
        const float ex = __builtin_amdgcn_exp2f(fmaf(s[e], cexp, -l4[x]));
        const float pr = !kInterval || on ? ex : 0.f;
        pf[e >> 3][e & 7] = (bf16)pr;
        dsf[e >> 3][e & 7] = (bf16)(pr * (dp[e] - dmul * d4[x]));
      }
    }
#pragma unroll
    for (int m = 0; m < 2; ++m)
      *reinterpret_cast<bf16x8*>(pbuf + ((2 * wave + m) * 64 + lane) * 16) = pf[m];
    bw_accum<4, 2>(dk, buf, tro[0], 2 * rh, dsf);       // dK^T += Q^T dS, own rows
    ATT_BARRIER();                                   // P of both row halves in LDS
    // P operands by 16-row step: own rows from registers, the other half's from LDS
#pragma unroll
    for (int m = 0; m < 2; ++m)
      pf[2 + m] = *reinterpret_cast<const bf16x8*>(pbuf + ((2 * (wave ^ 2) + m) * 64 + lane) * 16);
    bw_accum<2, 2>(dv, dos, tro[0] ^ (rh << 7), 2 * rh, pf);     // dV^T += dO^T P, dims 64 rh ..
    bw_accum<2, 2>(dv, dos, tro[0] ^ (rh << 7), 2 * (rh ^ 1), pf + 2);
    i = in;
    sel = cur;
  }

  __syncthreads();
  float* o_lds = reinterpret_cast<float*>(smem_dyn + kh * BW_STAGE_BYTES);
  float* v_lds = reinterpret_cast<float*>(smem_dyn + (2 + kh) * BW_STAGE_BYTES);
  AlphaView one;
  one.p = nullptr; one.scalar = 1.f; one.sb = one.ss = one.sh = one.sd = 0; one.dtype = ICSA_DT_F32;
  {
    const int lr = lane & 31;
#pragma unroll
    for (int ds = 0; ds < 2; ++ds)
#pragma unroll
      for (int e = 0; e < 16; ++e) v_lds[lr * O_LDS_STRIDE + 64 * rh + 32 * ds + acc_row(e, lane)] = dv[ds][e];
  }
  // dK: both row halves; the interval's dS lacked its 1 / 64 (partials: dk without the scale)
  bw_reduce_stage(o_lds, dk, rh, kInterval ? 1.0f / 64.0f : p.scale);
  const float* src = rh == 0 ? o_lds : v_lds;          // waves 0, 1 store dk, waves 2, 3 dv
  if (kInterval) {
    const int64_t base = (((int64_t)split * p.B * p.H + bh) * p.NKVp) * ICSA_D;
    store_rows(src, OutView{(rh == 0 ? p.dkc_part : p.dvc_part) + base, 0, ICSA_D, 0, ICSA_DT_F32}, 0, 0, key0, 32,
               nullptr, one);
  } else {
    const int kv = max(0, min(32, p.TKV - key0));     // rows past TKV are not stored
    store_rows(src, rh == 0 ? p.dk : p.dv, b, h, key0, kv, ivec + rh * ICSA_D, one);
  }
}

// Two launches: the query-major part with the interval part and the transposed bitmap (which
// do not depend on each other: their last rounds overlap; 345 us against 295 + 61 + 8 us one
// after another at 40 heads, 7,800 tokens), then the exact key-major part, which needs the
// other two.
__global__ void __launch_bounds__(BW_THREADS) __attribute__((amdgpu_waves_per_eu(2)))
icsa_sparse_bwd_query_kernel(SparseBwdParams p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_bw[];
  const int BH = p.B * p.H, n_iv = BH * p.nc * p.nsplit, n_tr = BH * p.nc;
  int blk = blockIdx.x;
  if (blk < xcd_grid(n_iv)) {                          // the longest workgroups first
    const int work = xcd_remap(blk, n_iv);
    if (work >= 0) bw_dkv<true>(p, smem_bw, work);
    return;
  }
  blk -= xcd_grid(n_iv);
  if (blk < xcd_grid(n_tr)) {
    if (blk < n_tr) bw_transpose_bits(p, blk / p.nc, blk % p.nc);
    return;
  }
  const int work = xcd_remap(blk - xcd_grid(n_tr), BH * p.NQ);
  if (work >= 0) bw_dq(p, smem_bw, work);
}

__global__ void __launch_bounds__(BW_THREADS) __attribute__((amdgpu_waves_per_eu(2)))
icsa_sparse_bwd_key_kernel(SparseBwdParams p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_bw[];
  const int work = xcd_remap(blockIdx.x, p.B * p.H * p.NKV);
  if (work >= 0) bw_dkv<false>(p, smem_bw, work);
}

hipError_t launch_sparse_bwd(const SparseBwdParams& p, hipStream_t stream) {
  const int BH = p.B * p.H;
  if (BH == 0 || p.NQ == 0) return hipSuccess;
  if (p.top_k < 1 || p.top_k > BW_MAX_TOPK || p.NKV < 1 || p.nc > BW_MAX_CHUNKS ||
      p.NKVp != p.nc * ICSA_BLOCK || p.NQ > BW_MAX_NQ || p.nsplit < 1 ||
      (int64_t)p.nsplit * p.qb_per_split < p.NQ)
    return hipErrorInvalidValue;
  static std::atomic<unsigned> set_q{0u}, set_k{0u};
  hipError_t attr = ensure_lds_limit(reinterpret_cast<const void*>(icsa_sparse_bwd_query_kernel), BW_LDS_BYTES, &set_q);
  if (attr != hipSuccess) return attr;
  attr = ensure_lds_limit(reinterpret_cast<const void*>(icsa_sparse_bwd_key_kernel), BW_LDS_BYTES, &set_k);
  if (attr != hipSuccess) return attr;
  hipLaunchKernelGGL(icsa_sparse_bwd_rows_kernel, dim3(p.NQ, BH), dim3(256), 0, stream, p);
  const int grid = xcd_grid(BH * p.nc * p.nsplit) + xcd_grid(BH * p.nc) + xcd_grid(BH * p.NQ);
  hipLaunchKernelGGL(icsa_sparse_bwd_query_kernel, dim3(grid), dim3(BW_THREADS), BW_LDS_BYTES, stream, p);
  hipLaunchKernelGGL(icsa_sparse_bwd_key_kernel, dim3(xcd_grid(BH * p.NKV)), dim3(BW_THREADS), BW_LDS_BYTES, stream, p);
  return hipGetLastError();
}
