// Stage 3: bf16 MFMA flash attention for the peaked query blocks (and the dense baseline).
//
// Reference: flash_attn_func(q_flat, new_k, new_v) at editing_sparse_attention.py:209-215 --
// dense non-causal softmax(q k^T / sqrt(D)) v of every peaked 64-row query block over the
// whole new KV, followed by the scatter and residual of :217-232.
//
// The new KV is never materialised: key tile j < n_tgt_tiles is target tile j of the
// original sequence (keys >= t_limit masked: the partial last target tile), tile
// n_tgt_tiles + r is source block sel_base + sel[r] (tokens >= Sk are zero keys with
// logit 0, exactly like the reference's zero padding of k_padded).  K is read in place;
// V^T holds tile j at columns 64 j .. 64 j + 63 (the pipeline writes it in that order).
//
// Work is dealt in items: four 64-row query blocks of one head against all key tiles.  A
// workgroup runs a sequence of segments (runs of tiles of one item): several whole items, or
// one of the equal ranges ("chunks") that the tiles of the last, incomplete round's items
// are cut into, whose partial O, max and sum icsa_flash_combine_kernel adds up.  The tile
// stream runs across segment boundaries, so the next item's tiles arrive while an item
// ends.  Measured against one workgroup per item, with an epilogue of its own: 32 items of
// 72 tiles (2 heads, 8,192 tokens) 101 -> 30 us plus 9 us for the sums; 640 items of 576
// tiles (5 heads, 65,536 tokens; 2.5 rounds) 2,825 -> 2,536 + 11 us; 10,240 items of 8
// tiles (512 keys, 40 heads, 65,520 queries) 853 -> 768-790 us; 5,120 items of 576 tiles (40
// heads) unchanged at 19.9 ms.  The rate is then about 1.2 PFLOP/s at every size that
// fills the chip, the engine clock under this load being 1.7-1.9 GHz; with 8 tiles an item,
// timing copies without the output stores and without the Q loads took 693 and 755 us (both:
// 641 us) when the kernel took 775.
//
// Workgroup = 8 waves = an item's query blocks (wave w: block w/2, rows 32*(w%2)..+31),
// all sharing each K / V^T tile.  The waves form two groups, G0 = waves 0-3 and G1 = waves
// 4-7, so every SIMD holds one wave of each.  The groups run the same sequence of phases
//     GEMM(k) = { S(k) = K(k) Q^T ;  O += V(k-1)^T P(k-1) }      (32 MFMAs)
//     SOFT(k) = { row max, lazy rescale, P(k) = exp2(S(k) c - m) } (~1000 VALU cycles)
// G1 one slot behind G0, with a workgroup barrier between slots: in every slot one wave per
// SIMD feeds the matrix pipe while the other keeps the vector ALU busy ("ping-pong").
//
// Tiles arrive by direct global->LDS buffer loads (LDS DMA: lane l of a load lands at
// M0 + 16 l), four buffers deep.  Issuing LDS DMA blocks the issuing wave while the CU's
// vector-memory path takes earlier requests, so only waves in their SOFT phase issue it,
// one 1-KB segment between every 8 exponentials (group 1: K tiles, group 0: V^T tiles; the
// slot schedule below).  The LDS XOR swizzle is applied on the global side: each lane
// fetches the chunk that belongs in its LDS slot.  Per-lane global offsets are computed
// once, the tile start is the scalar base of a buffer resource whose range covers only key
// rows below Sk, and every LDS offset is hoisted out of the loop.
//
// Softmax state: probabilities are taken relative to a reference max m_ref.  A segment starts
// without one (its rows are other queries, maybe another head's) and takes its first tile's
// row max, before any exponential.  From then on the probabilities come first and are checked
// afterwards: only when a lane's partial sum of the tile exceeds 2^64 (or is NaN) is the row max
// of the tile taken, the reference raised, O / l rescaled and the tile recomputed.  In the
// common case no per-tile max reduction precedes the exponentials.  Exact in real arithmetic.
// (The first tile by that check as well, two passes of exponentials: 8 tiles an item, forward
// 811-823 us a call against 789-806.)
#include "attn_tile.h"
#include "flash_plan.h"
#include "icsa_kernels.h"

#define FA_THREADS (FA_WAVES * 64)
#define FA_NBUF 4                                            // K and V^T tile buffers
#define FA_TILE_BYTES (FA_NBUF * (K_TILE_BYTES + V_TILE_BYTES))
#define FA_JUNK_OFF FA_TILE_BYTES                            // landing area of disabled DMA
#define FA_STAGE_OFF (FA_JUNK_OFF + 4096)                    // 2 KB of output staging per wave
#define FA_STAGE_WAVE 2048
#define FA_LDS_BYTES (FA_STAGE_OFF + FA_WAVES * FA_STAGE_WAVE)
// A lane's 32 probabilities of a tile sum to at most 2^64 relative to the row's reference
// max before the reference is raised: O and l then stay below 2^64 * keys * |v|, far inside
// the fp32 range, and bf16(p) keeps its relative precision at any magnitude.
#define FA_PSUM_MAX 18446744073709551616.0f
// The reference max before the first tile: finite, so that a tile whose scores are all -inf
// leaves O = l = 0 instead of inf - inf.
#define FA_M_NONE (-3.4028234663852886e38f)
#ifndef FA_PF
#define FA_PF 5             // operand prefetch depth (MFMA steps); 3, 4, 6 and 8 measured slower
#endif

namespace {

typedef const __attribute__((address_space(4))) int* const_int_ptr;
// A wave-uniform int of global memory through the scalar cache: a vector load would have to
// be waited for behind the tile DMA in flight.  Only for data written by earlier kernels.
__device__ __forceinline__ int uniform_load(const int* p) {
  return *(const_int_ptr)(unsigned long long)p;
}

// The parameter block re-read from the kernel-argument segment: what only a segment boundary
// needs does not stay in scalar registers (which spill into vector lanes) through the tiles.
__device__ __forceinline__ const FlashParams& cold_params() {
  auto kp = (const __attribute__((address_space(4))) FlashParams*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(kp));
  return *(const FlashParams*)kp;
}

// Iterations [lo, hi) of chunk c: the split items' tiles as one sequence, cut in n_chunk ranges
__host__ __device__ __forceinline__ int64_t chunk_start(int c, int n_split, int n_tiles, int n_chunk) {
  return (int64_t)c * ((int64_t)n_split * n_tiles) / n_chunk;
}

// d-subtile ds of one wave's 32 output rows straight from the accumulators (lane (li, hl)
// holds dims 32 ds + 8 g + 4 hl + x of query li; g, x = 0..3): 1 / l, residual, output type.
// The rows pass through 2 KB of the wave's own LDS, 64 bytes of each at a time, so that a
// store instruction writes 16 segments of 64 bytes; stores straight from the accumulators
// are 64 segments of 16 bytes, four times the requests.  16-byte chunk c of row r sits at
// chunk c ^ (r / 4 % 4): writes (one chunk of 16 rows) and reads (4 chunks of 4 rows) both
// touch every bank once.
template <bool kBf16, bool kAlphaD>
__device__ __forceinline__ void store_subtile(unsigned char* stage, const floatx16& o, int ds, float inv_l,
                                              const OutView& out, int b, int h, int tok0, int n_rows,
                                              const float* oc_row, const AlphaView& alpha) {
  const int lane = threadIdx.x & 63, li = lane & 31, hl = lane >> 5;
  float v[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = o[i] * inv_l;
  if (oc_row != nullptr && li < n_rows) {
    const float a0 = kAlphaD ? 0.f : alpha_at(alpha, b, tok0 + li, h, 0);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d = 32 * ds + 8 * g + 4 * hl;
      const floatx4 c = *reinterpret_cast<const floatx4*>(oc_row + d);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[4 * g + e] = fmaf(kAlphaD ? alpha_at(alpha, b, tok0 + li, h, d + e) : a0, c[e], v[4 * g + e]);
    }
  }
  unsigned char* wr = stage + li * 64;
  const int wx = (li >> 2) & 3;
  const int64_t off = (int64_t)b * out.sb + (int64_t)tok0 * out.ss + (int64_t)h * out.sh + 32 * ds;
  auto store_rows64 = [&](unsigned char* dst, int64_t row_bytes) {    // 32 staged rows of 64 bytes
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = 16 * i + (lane >> 2);
      const u32x4 x = *reinterpret_cast<const u32x4*>(stage + r * 64 + (((lane & 3) ^ ((r >> 2) & 3)) << 4));
      if (r < n_rows) *reinterpret_cast<u32x4*>(dst + r * row_bytes + 16 * (lane & 3)) = x;
    }
  };
  if constexpr (kBf16) {
#pragma unroll
    for (int pr = 0; pr < 2; ++pr) {               // lane halves swap: dims 8 (2 pr + hl) .. + 7
      bf16x4 lo, hi;
#pragma unroll
      for (int e = 0; e < 4; ++e) { lo[e] = (bf16)v[8 * pr + e]; hi[e] = (bf16)v[8 * pr + 4 + e]; }
      const u32x2 x = __builtin_bit_cast(u32x2, lo), y = __builtin_bit_cast(u32x2, hi);
      const auto w0 = __builtin_amdgcn_permlane32_swap(x[0], y[0], false, false);
      const auto w1 = __builtin_amdgcn_permlane32_swap(x[1], y[1], false, false);
      *reinterpret_cast<u32x4*>(wr + (((2 * pr + hl) ^ wx) << 4)) = u32x4{w0[0], w1[0], w0[1], w1[1]};
    }
    store_rows64(reinterpret_cast<unsigned char*>(reinterpret_cast<bf16*>(out.p) + off), out.ss * 2);
  } else {
#pragma unroll
    for (int pr = 0; pr < 2; ++pr) {               // dims 16 pr .. + 15
#pragma unroll
      for (int g = 0; g < 2; ++g)
        *reinterpret_cast<floatx4*>(wr + (((2 * g + hl) ^ wx) << 4)) =
            floatx4{v[8 * pr + 4 * g], v[8 * pr + 4 * g + 1], v[8 * pr + 4 * g + 2], v[8 * pr + 4 * g + 3]};
      store_rows64(reinterpret_cast<unsigned char*>(reinterpret_cast<float*>(out.p) + off + 16 * pr), out.ss * 4);
    }
  }
}

}  // namespace

template <bool kBf16, bool kAlphaD>
__global__ void __launch_bounds__(FA_THREADS) __attribute__((amdgpu_waves_per_eu(2)))
icsa_flash_kernel(FlashParams p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int ngrp = (p.n_qblk + FA_QBLK_PER_WG - 1) / FA_QBLK_PER_WG;
  const int n_tiles = p.n_tgt_tiles + p.n_sel;
  const int tid = threadIdx.x;
  // wave index made provably wave-uniform (a scalar), so per-group branches stay uniform
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int li = lane & 31, hl = lane >> 5;
  const int group = wave >> 2;                        // 0: leads, 1: one slot behind
  const bool lag = group == 1;

  // ---- this workgroup's segments (runs of tiles of one item) ----
  // The first: len0 tiles from tile0 of item0; each further one: len1 tiles from tile1 of the
  // item `step` away; n_it tiles in all.  A chunk that ends one item and starts the next
  // takes the start first: all chunks then begin near tile 0 and walk the keys side by side
  // (a window of n_tiles - chunk length tiles that L2 holds) instead of being spread over
  // all of them.
  int item0, tile0 = 0, len0 = n_tiles, tile1 = 0, len1 = n_tiles, step = 1, n_it, chunk = -1;
  if ((int)blockIdx.x < FA_XCDS * p.n_bundle) {
    const FlashRun run = flash_whole_run(blockIdx.x, p.n_whole, p.n_bundle);
    if (run.count == 0) return;
    item0 = run.first;
    step = p.n_bundle;
    n_it = run.count * n_tiles;
  } else {
    chunk = xcd_remap(blockIdx.x - FA_XCDS * p.n_bundle, p.n_chunk);
    if (chunk < 0) return;
    const int n_split = p.B * p.H * ngrp - p.n_whole;
    const int64_t lo = chunk_start(chunk, n_split, n_tiles, p.n_chunk);
    n_it = (int)(chunk_start(chunk + 1, n_split, n_tiles, p.n_chunk) - lo);    // <= n_tiles
    if (n_it <= 0) return;
    item0 = p.n_whole + (int)(lo / n_tiles);
    tile0 = (int)(lo % n_tiles);
    len0 = min(n_it, n_tiles - tile0);
    if (len0 < n_it) {
      tile1 = tile0;
      len1 = len0;
      step = -1;
      ++item0;
      tile0 = 0;
      len0 = n_it - len1;
    }
  }

  // ---- per-lane offsets, hoisted out of the loop ----
  int kro[8], vro[4];                                 // MFMA operand read offsets (bytes)
#pragma unroll
  for (int kk = 0; kk < 8; ++kk) kro[kk] = k_lds_off(li, 2 * kk + hl) * 2;   // + 32 rows per sub-tile
#pragma unroll
  for (int m = 0; m < 4; ++m) vro[m] = v_lds_off(li, 2 * m + hl) * 2;        // + 32 d rows per sub-tile

  // buffer of iteration j's tile
  auto kbuf = [&](int j) -> unsigned char* { return smem + (j % FA_NBUF) * K_TILE_BYTES; };
  auto vbuf = [&](int j) -> unsigned char* {
    return smem + FA_NBUF * K_TILE_BYTES + (j % FA_NBUF) * V_TILE_BYTES;
  };

  // ---- DMA cursor: the next tile this wave's group fetches (K: group 1, V^T: group 0) ----
  // It runs 2 to 4 tiles ahead of the computation, across item boundaries.
  const int dw = wave & 3;
  int dofs[4];                            // segment offsets: K rows (group 1) / V^T rows (group 0)
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int sg = 4 * dw + i;
    if (lag) {
      const int kr = 4 * sg + (lane >> 4), kc = (lane & 15) ^ (kr & 15);
      dofs[i] = (int)(((int64_t)kr * p.k_ss + 8 * kc) * 2);
    } else {
      const int vd = 8 * sg + (lane >> 3), vc = (lane & 7) ^ ((vd >> 1) & 7);
      dofs[i] = (int)(((int64_t)vd * p.vt_sd + 8 * vc) * 2);
    }
  }
  int d_j = 0, d_tile = tile0, d_left = len0, d_item = item0, d_bh = 0;
  int d_tok = 0;                          // group 1: token start of the cursor's tile
  unsigned kv_ring = 0;                   // group 1: real key rows of the last four tiles, 8 bits each
  const bf16* d_base = nullptr;           // K / V^T of the cursor's head
  auto d_head = [&]() {
    d_bh = d_item / ngrp;
    const int b = d_bh / p.H, h = d_bh % p.H;
    d_base = lag ? p.k + (int64_t)b * p.k_sb + (int64_t)h * p.k_sh : p.vt + (int64_t)b * p.vt_sb + (int64_t)h * p.vt_sh;
  };
  auto d_token = [&]() {                  // fetched one call ahead: the scalar load's latency is hidden
    d_tok = d_tile * ATT_BN;
    if (d_tile >= p.n_tgt_tiles && d_j < n_it)
      d_tok = (p.sel_base + uniform_load(p.sel + (int64_t)d_bh * p.sel_stride + (d_tile - p.n_tgt_tiles))) * ATT_BN;
  };
  d_head();
  if (lag) d_token();
  __amdgpu_buffer_rsrc_t dma_rs = make_rsrc(d_base, 0);
  unsigned char* dma_dst = smem;
  // Sets up this wave's part of the next tile.  Byte ranges fit 32 bits (checked at launch),
  // so only the base addresses take 64-bit arithmetic: the setup runs in the SOFT phase,
  // where its scalar work competes with the exponentials.  Past the last tile the issue
  // stays branch-free: an empty range into a junk LDS area.
  const int k_row_bytes = (int)p.k_ss * 2;
  const int v_rec = (ICSA_D - 1) * (int)p.vt_sd * 2 + ATT_BN * 2;
  auto dma_setup = [&]() __attribute__((always_inline)) {
    const bool on = d_j < n_it;
    if (lag) {
      const int k_valid = on ? min(ATT_BN, p.Sk - d_tok) : 0;
      const int k_rec = k_valid > 0 ? (k_valid - 1) * k_row_bytes + ICSA_D * 2 : 0;
      dma_rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(d_base + (on ? (int64_t)d_tok * p.k_ss : 0)), (short)0,
                                                 k_rec, 0x00020000);
      kv_ring = (kv_ring << 8) | (unsigned)max(k_valid, 0);
    } else {
      dma_rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(d_base + (int64_t)(on ? d_tile : 0) * ATT_BN),
                                                 (short)0, on ? v_rec : 0, 0x00020000);
    }
    dma_dst = !on ? smem + FA_JUNK_OFF : (lag ? kbuf(d_j) : vbuf(d_j)) + dw * 4096;
    ++d_j;
    ++d_tile;
    if (--d_left == 0) {
      d_tile = tile1;
      d_left = len1;
      d_item += step;
      if (d_j < n_it) d_head();
    }
    if (lag) d_token();
  };
  auto dma_seg = [&](int i) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(dma_rs, (lds_ptr)(dma_dst + 1024 * i), 16, dofs[i], 0, 0, 0);
  };
  auto issue_all = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i) dma_seg(i);
  };

  struct Seg { int item, qblk, q_valid; };
  auto seg_of = [&](int item) -> Seg {
    const FlashParams& cp = cold_params();
    Seg s;
    s.item = item;
    const int bh = item / ngrp, slot = item % ngrp * FA_QBLK_PER_WG + (wave >> 1);
    const bool on = slot < cp.n_qblk;
    s.qblk = !on ? 0 : (cp.qblocks ? uniform_load(cp.qblocks + (int64_t)bh * cp.qb_stride + cp.qb_offset + slot) : slot);
    s.q_valid = on ? max(0, min(32, cp.Sq - s.qblk * ICSA_BLOCK - 32 * (wave & 1))) : 0;
    return s;
  };
  Seg sg = seg_of(item0);                             // the segment whose output is in O
  Seg nx = sg;                                        // the one after it, looked up a segment ahead
  if (n_it > len0) nx = seg_of(item0 + step);

  floatx16 o[4] = {};
  floatx16 s[2];
  bf16x8 qf[8];
  bf16x8 pf[4];
  float m_ref = FA_M_NONE, l_run = 0.f;
  const float c = p.scale_log2;

  auto load_q = [&](const Seg& g) __attribute__((always_inline)) {
    const FlashParams& cp = cold_params();
    const int bh = g.item / ngrp, b = bh / cp.H, h = bh % cp.H;
    load_q_frags(qf, cp.q + (int64_t)b * cp.q_sb + (int64_t)(g.qblk * ICSA_BLOCK + 32 * (wave & 1)) * cp.q_ss +
                         (int64_t)h * cp.q_sh, cp.q_ss, g.q_valid);
  };
  // The finished segment's O: to its output rows, or (a part of an item) to the partials.
  auto flush = [&](bool part) __attribute__((always_inline)) {
    const FlashParams& cp = cold_params();
    if (part) {
      const int u = chunk + (sg.item - cp.n_whole);
      float* dst = cp.part + (int64_t)u * FA_PART_FLOATS + wave * FA_PART_WAVE;
#pragma unroll
      for (int ds = 0; ds < 4; ++ds)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *reinterpret_cast<floatx4*>(dst + ((ds * 4 + g) * 64 + lane) * 4) =
              floatx4{o[ds][4 * g], o[ds][4 * g + 1], o[ds][4 * g + 2], o[ds][4 * g + 3]};
      dst[4096 + lane] = m_ref;
      dst[4096 + 64 + lane] = l_run;
      return;
    }
    const int bh = sg.item / ngrp, b = bh / cp.H, h = bh % cp.H;
    const float inv_l = 1.f / xhalf_sum(l_run);
    const float* oc = cp.out_c ? cp.out_c + ((int64_t)bh * cp.nb_q + sg.qblk) * ICSA_D : nullptr;
    const OutView ov = cp.out;
    const AlphaView av = cp.alpha;
#pragma unroll
    for (int ds = 0; ds < 4; ++ds) {
      store_subtile<kBf16, kAlphaD>(smem + FA_STAGE_OFF + wave * FA_STAGE_WAVE, o[ds], ds, inv_l, ov, b, h,
                    sg.qblk * ICSA_BLOCK + 32 * (wave & 1), sg.q_valid, oc, av);
      __builtin_amdgcn_sched_barrier(0);              // one sub-tile's temporaries at a time
    }
  };

  // GEMM(k): O += V(k-1)^T P(k-1) and S(k) = K(k) Q^T.  Operands are read from LDS into
  // registers FA_PF MFMA steps ahead of their use (explicit software pipeline), so the
  // matrix pipe does not wait on LDS latency.
  auto gemm_pv = [&](int k) __attribute__((always_inline)) {
    const unsigned char* vs = vbuf(k - 1);
    bf16x8 va[16];
#pragma unroll
    for (int t = 0; t < FA_PF; ++t)
      va[t] = *reinterpret_cast<const bf16x8*>(vs + vro[t >> 2] + (t & 3) * 32 * ATT_BN * 2);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      if (t + FA_PF < 16) {
        const int u = t + FA_PF;
        va[u] = *reinterpret_cast<const bf16x8*>(vs + vro[u >> 2] + (u & 3) * 32 * ATT_BN * 2);
      }
      o[t & 3] = mfma32x32x16(va[t], pf[t >> 2], o[t & 3]);
      __builtin_amdgcn_sched_barrier(0);    // keep the read-ahead order
    }
  };
  auto gemm_qk = [&](int k) __attribute__((always_inline)) {
    const unsigned char* ks = kbuf(k);
    bf16x8 ka[16];
    floatx16 acc0 = {}, acc1 = {};
#pragma unroll
    for (int t = 0; t < FA_PF; ++t)
      ka[t] = *reinterpret_cast<const bf16x8*>(ks + kro[t >> 1] + (t & 1) * 32 * ICSA_D * 2);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      if (t + FA_PF < 16) {
        const int u = t + FA_PF;
        ka[u] = *reinterpret_cast<const bf16x8*>(ks + kro[u >> 1] + (u & 1) * 32 * ICSA_D * 2);
      }
      if (t & 1) acc1 = mfma32x32x16(ka[t], qf[t >> 1], acc1);
      else acc0 = mfma32x32x16(ka[t], qf[t >> 1], acc0);
      __builtin_amdgcn_sched_barrier(0);
    }
    s[0] = acc0;
    s[1] = acc1;
  };
  // SOFT(k): mask, P(k) against the reference max, and -- only when some probability of the
  // tile left the allowed range -- a rescale to the tile's row max and a second pass.  The
  // wave's DMA segments go out one at a time between the exponentials of the first pass.
  auto soft = [&](int tile, bool first) __attribute__((always_inline)) {
    const int mask_from = tile < p.n_tgt_tiles ? p.t_limit - tile * ATT_BN : ATT_BN;
    if (mask_from < ATT_BN) {
      // keys >= mask_from as one 64-bit word; element i of sub-tile sub is key
      // 32 sub + 8 (i / 4) + 4 hl + i % 4, bit 8 (i / 4) + i % 4 of word sub of the word
      // shifted by 4 hl.  Integer selects: per-element compares would hold 32 lane masks in
      // scalar registers, which spill into vector lanes and slow every SOFT phase.
      const unsigned long long mw = (~0ull << max(mask_from, 0)) >> (4 * hl);
#pragma unroll
      for (int sub = 0; sub < 2; ++sub) {
        const unsigned wd = (unsigned)(mw >> (32 * sub));
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int kb = 8 * (i >> 2) + (i & 3);
          const unsigned all = (unsigned)((int)(wd << (31 - kb)) >> 31);
          s[sub][i] = __uint_as_float((all & 0xff800000u) | (__float_as_uint(s[sub][i]) & ~all));
        }
      }
    }
    float rs = 0.f;
    if (!first) {
      // four partial sums: a single chain of 32 dependent adds measured 0.4 % slower
      float rsv[4];
#pragma unroll
      for (int sb = 0; sb < 2; ++sb)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          if ((i & 7) == 0) {                // DMA segment 2 sb + i / 8 before every 8th exponential
            __builtin_amdgcn_sched_barrier(0);
            dma_seg(2 * sb + (i >> 3));
            __builtin_amdgcn_sched_barrier(0);
          }
          const float e = __builtin_amdgcn_exp2f(fmaf(s[sb][i], c, -m_ref));
          if (sb == 0 && i < 4) rsv[i] = e;      // no adds of 0.f (not foldable: signed zeros)
          else rsv[i & 3] += e;
          pf[2 * sb + (i >> 3)][i & 7] = (bf16)e;
        }
      rs = (rsv[0] + rsv[1]) + (rsv[2] + rsv[3]);
    } else {
      issue_all();
    }
    // The partial sum exceeds FA_PSUM_MAX (or is NaN) only when a score rose far above the
    // reference: then, and in a segment's first tile, raise the reference of every row whose
    // tile max exceeds it, rescale O and l, and (re)compute the tile's probabilities.
    if (first || __ballot(!(rs <= FA_PSUM_MAX)) != 0ull) {
      float mx = -INFINITY;
#pragma unroll
      for (int sub = 0; sub < 2; ++sub)
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[sub][i]);
      mx = xhalf_max(mx) * c;
      const float mn = mx > m_ref ? mx : m_ref;
      const float a = __builtin_amdgcn_exp2f(m_ref - mn);
#pragma unroll
      for (int ds = 0; ds < 4; ++ds)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[ds][i] *= a;
      l_run *= a;
      m_ref = mn;
      rs = 0.f;
#pragma unroll
      for (int sb = 0; sb < 2; ++sb)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float e = __builtin_amdgcn_exp2f(fmaf(s[sb][i], c, -m_ref));
          rs += e;
          pf[2 * sb + (i >> 3)][i & 7] = (bf16)e;
        }
    }
    l_run += rs;
  };

  // Slot schedule.  Every slot ends with a workgroup barrier; group 0 runs GEMM(k) in slot
  // 2k and SOFT(k) in slot 2k + 1, group 1 one slot later.  Issuing LDS-DMA blocks the
  // issuing wave while the CU's vector-memory path drains earlier requests (about 22
  // s_memtime ticks per 1-KB instruction), so the tile DMA is issued only by waves in their
  // SOFT phase, one segment between every 8 exponentials, never by a GEMM wave:
  //   K(j): group 1 during SOFT(j - 4), slot 2j - 6; waited for by group 1 at the end of its
  //         GEMM(j - 1), slot 2j - 1; read in slots 2j (group 0) and 2j + 1 (group 1);
  //   V(j): group 0 during SOFT(j - 2), slot 2j - 3; waited for by group 0 at the end of its
  //         SOFT(j), slot 2j + 1; read (as PV(j)) in slots 2j + 2 and 2j + 3.
  // Four buffers per kind: K(j) overwrites K(j - 4), last read in slot 2j - 7; V(j)
  // overwrites V(j - 4), last read (PV(j - 4)) in slot 2j - 5.  Loads complete in issue
  // order, so vmcnt(8) waits for all but this wave's two newest tiles.  Slots past the last
  // tile issue empty-range loads into a junk LDS area (the issue stays branch-free).
  // A segment boundary costs no slot: Q of the next segment is requested in the SOFT phase
  // of the last tile (its registers are free since that tile's QK) and first used after the
  // next GEMM's PV and the output, which are written from the accumulators between that
  // GEMM's PV and QK (the scores and probabilities are not live there).  These loads and
  // stores are newer than the tiles waited for next (group 0's in the same SOFT phase for Q and
  // in the following one for the output, group 1's in the writing GEMM phase and in the
  // following one), so the wait allows 8 more in flight where at least 8 are sure: Q is 8 loads
  // of a wave with any row; the output at least 8 stores of a wave with more than 16 rows (of
  // fewer, the bf16 form issues 4: its second store of a sub-tile, rows 16 .. 31, is skipped).
  // zero key rows >= k_valid of a group-1 wave's K segments (rows 16 dw .. 16 dw + 15)
  auto fill_tail4 = [&](int j, int k_valid) {
    if (k_valid >= ATT_BN) return;
    const int row = 16 * dw + (lane >> 2);
    if (row >= k_valid) {
      unsigned char* dst = kbuf(j) + row * ICSA_D * 2 + (lane & 3) * 64;
#pragma unroll
      for (int e = 0; e < 4; ++e) *reinterpret_cast<u32x4*>(dst + 16 * e) = u32x4{0u, 0u, 0u, 0u};
    }
  };
  // wait for a tile, leaving the two tiles issued after it (past the last tile: the empty
  // loads) in flight, and with `extra` the 8 loads or stores of a segment boundary
  auto wait_tile = [&](bool extra) {
    if (extra) asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
  };
  // group 1, at the end of GEMM(j - 1): K(j) complete, rows past Sk zero
  auto wait_k = [&](int j, bool extra) {
    if (!lag || j >= n_it) return;
    wait_tile(extra);
    fill_tail4(j, (int)((kv_ring >> 16) & 0xff));
  };
  if (lag) {
    for (int j = 0; j < 3; ++j) { dma_setup(); issue_all(); }
  } else {
    dma_setup(); issue_all();
    dma_setup(); issue_all();
  }
  load_q(sg);
  if (lag) {                               // K(0); its two newer tiles and Q as well
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    fill_tail4(0, (int)((kv_ring >> 16) & 0xff));
  }
  ATT_BARRIER();
  if (lag) {                               // slot 0 for group 1: K(3)
    dma_setup();
    issue_all();
    ATT_BARRIER();
  }
  __builtin_amdgcn_s_setprio(1);           // the matrix-feeding wave wins issue ties
  gemm_qk(0);
  __builtin_amdgcn_s_setprio(0);
  wait_k(1, false);
  ATT_BARRIER();
  int tile = tile0;                        // tile of iteration k
  int seg_len = len0;
  int k = 0;
  // A wave without rows in any of the workgroup's items only moves tiles: its products and
  // exponentials would take issue slots from the others (calls of one head, 64 queries, 1,000
  // keys 29.9 -> 25.6 us; 320 heads, 1 query, 512 keys 50.6 -> 45.2; 640 heads, 64 queries, 2,048
  // keys 366 -> 359).  Decided once: the same test around every product and exponential
  // costs 168 spilled vector registers and 2 to 3 times the time.
  if (sg.q_valid == 0 && (n_it <= len0 || (ngrp == 1 && p.qblocks == nullptr))) {
    for (;;) {
      dma_setup();
      issue_all();
      if (!lag) wait_tile(false);
      ATT_BARRIER();
      if (k + 1 == n_it) break;
      wait_k(k + 2, false);
      ATT_BARRIER();
      ++k;
    }
    if (!lag) ATT_BARRIER();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    return;
  }
  // Every segment goes through the general iteration below for its first and its last tile
  // and through the plain loop for those between.
  bool wrote = false;                      // the GEMM phase before this SOFT phase issued 8 stores or more
  bool first = true;                       // the segment's first iteration
  int last = len0 - 1;                     // and its last
  for (;;) {
    const bool ends = k == last, more = k + 1 < n_it;
    bool q_ahead = false, writes = false;
    if (ends && more) {
      load_q(nx);
      q_ahead = nx.q_valid > 0;
      __builtin_amdgcn_sched_barrier(0);
    }
    dma_setup();
    soft(tile, first);
    if (!lag) wait_tile(wrote || q_ahead);            // V(k)
    ATT_BARRIER();
    __builtin_amdgcn_s_setprio(1);
    gemm_pv(k + 1);
    if (!more) break;
    if (ends) {
      __builtin_amdgcn_s_setprio(0);
      writes = sg.q_valid > 16;
      if (sg.q_valid > 0) flush(seg_len != n_tiles);
#pragma unroll
      for (int ds = 0; ds < 4; ++ds) o[ds] = floatx16{};
      l_run = 0.f;
      m_ref = FA_M_NONE;             // other rows: nothing of this segment's scores carries over
      tile = tile1 - 1;
      seg_len = len1;
      last = k + len1;
      sg = nx;
      if (n_it - (k + 1) > len1) nx = seg_of(sg.item + step);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_setprio(1);
    }
    gemm_qk(k + 1);
    __builtin_amdgcn_s_setprio(0);
    wait_k(k + 2, wrote || writes);
    ATT_BARRIER();
    ++k;
    ++tile;
    if (!ends) {
      for (; k < last; ++k, ++tile) {
        dma_setup();
        soft(tile, false);
        if (!lag) wait_tile(false);
        ATT_BARRIER();
        __builtin_amdgcn_s_setprio(1);
        gemm_pv(k + 1);
        gemm_qk(k + 1);
        __builtin_amdgcn_s_setprio(0);
        wait_k(k + 2, false);
        ATT_BARRIER();
      }
    }
    wrote = writes;
    first = ends;
  }
  __builtin_amdgcn_s_setprio(0);
  if (!lag) ATT_BARRIER();       // group 1's last SOFT phase ends here
  // empty-range DMA of the last slots may still be in flight towards the junk area
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (sg.q_valid > 0) flush(seg_len != n_tiles);
}

// ------------------------------------------------------------------------------------------
// Sums the partials of every split item and writes its rows: workgroup (item, wave of the
// flash workgroup), wave ds: d-subtile ds of its 32 queries.  Segments in tile order, the
// running reference max as in the flash loop: a fixed order, bitwise reproducible.
// ------------------------------------------------------------------------------------------
#define FC_AHEAD 4                                   // partials requested together

template <bool kBf16, bool kAlphaD>
__global__ void __launch_bounds__(256) icsa_flash_combine_kernel(FlashParams p) {
  __shared__ __attribute__((aligned(16))) unsigned char stage[4][FA_STAGE_WAVE];
  const int ngrp = (p.n_qblk + FA_QBLK_PER_WG - 1) / FA_QBLK_PER_WG;
  const int n_tiles = p.n_tgt_tiles + p.n_sel, n_split = p.B * p.H * ngrp - p.n_whole;
  const int r = blockIdx.x / FA_WAVES, w = blockIdx.x % FA_WAVES;
  const int ds = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int bh = (p.n_whole + r) / ngrp, grp = (p.n_whole + r) % ngrp;
  const int slot = grp * FA_QBLK_PER_WG + (w >> 1);
  if (slot >= p.n_qblk) return;                      // uniform for the workgroup
  const int qblk = p.qblocks ? p.qblocks[(int64_t)bh * p.qb_stride + p.qb_offset + slot] : slot;
  const int q_valid = min(32, p.Sq - qblk * ICSA_BLOCK - 32 * (w & 1));
  if (q_valid <= 0) return;
  // chunks c0 .. c1 - 1 hold tiles of the item: the last one that starts at or before its
  // first tile, up to the last that starts before its end
  auto start = [&](int c) -> int64_t { return chunk_start(c, n_split, n_tiles, p.n_chunk); };
  const int64_t t0 = (int64_t)r * n_tiles, t1 = t0 + n_tiles;
  int c0 = (int)((int64_t)r * p.n_chunk / n_split);
  while (c0 + 1 < p.n_chunk && start(c0 + 1) <= t0) ++c0;
  while (c0 > 0 && start(c0) > t0) --c0;
  int c1 = c0 + 1;
  while (c1 < p.n_chunk && start(c1) < t1) ++c1;
  if (c1 - c0 == 1) return;                          // one workgroup had the whole item
  const float* base = p.part + ((int64_t)(c0 + r) * FA_WAVES + w) * FA_PART_WAVE;
  floatx16 acc = {};
  float m = FA_M_NONE, l = 0.f;
  for (int i = 0; i < c1 - c0; i += FC_AHEAD) {
    floatx4 v[FC_AHEAD][4];
    float ms[FC_AHEAD], ls[FC_AHEAD];
#pragma unroll
    for (int a = 0; a < FC_AHEAD; ++a) {
      const float* src = base + (int64_t)min(i + a, c1 - c0 - 1) * FA_PART_FLOATS;
#pragma unroll
      for (int g = 0; g < 4; ++g) v[a][g] = *reinterpret_cast<const floatx4*>(src + ((ds * 4 + g) * 64 + lane) * 4);
      ms[a] = src[4096 + lane];
      ls[a] = src[4096 + 64 + lane];
    }
#pragma unroll
    for (int a = 0; a < FC_AHEAD; ++a) {
      if (i + a >= c1 - c0) break;
      const float mn = ms[a] > m ? ms[a] : m;
      const float fo = __builtin_amdgcn_exp2f(m - mn), fn = __builtin_amdgcn_exp2f(ms[a] - mn);
#pragma unroll
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[4 * g + e] = fmaf(v[a][g][e], fn, acc[4 * g + e] * fo);
      l = fmaf(ls[a], fn, l * fo);
      m = mn;
    }
  }
  const float* oc = p.out_c ? p.out_c + ((int64_t)bh * p.nb_q + qblk) * ICSA_D : nullptr;
  store_subtile<kBf16, kAlphaD>(stage[ds], acc, ds, 1.f / xhalf_sum(l), p.out, bh / p.H, bh % p.H,
                qblk * ICSA_BLOCK + 32 * (w & 1), q_valid, oc, p.alpha);
}

// kAlphaD: the residual weight varies along the head dim (its own instantiation: its gathers
// would cost the usual one registers)
template <bool kBf16, bool kAlphaD>
static hipError_t run_flash(const FlashParams& p, int64_t n_work, hipStream_t stream) {
  static std::atomic<unsigned> lds_set{0u};
  const hipError_t attr = ensure_lds_limit(reinterpret_cast<const void*>(icsa_flash_kernel<kBf16, kAlphaD>),
                                           FA_LDS_BYTES, &lds_set);
  if (attr != hipSuccess) return attr;
  hipLaunchKernelGGL((icsa_flash_kernel<kBf16, kAlphaD>), dim3(FA_XCDS * p.n_bundle + xcd_grid(p.n_chunk)),
                     dim3(FA_THREADS), FA_LDS_BYTES, stream, p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || p.n_chunk == 0) return e;
  hipLaunchKernelGGL((icsa_flash_combine_kernel<kBf16, kAlphaD>), dim3((unsigned)(n_work - p.n_whole) * FA_WAVES),
                     dim3(256), 0, stream, p);
  return hipGetLastError();
}

hipError_t launch_flash(FlashParams p, hipStream_t stream) {
  const int64_t n_work = flash_items(p.B * p.H, p.n_qblk);
  const int n_tiles = p.n_tgt_tiles + p.n_sel;
  if (n_work == 0) return hipSuccess;
  if (n_tiles <= 0 || n_work > 0x7fffffffLL / 2) return hipErrorInvalidValue;
  // per-(b, h) slices must be addressable with 32-bit buffer offsets
  if ((int64_t)p.Sk * p.k_ss * 2 > 0x7fffffffLL || (int64_t)ICSA_D * p.vt_sd * 2 > 0x7fffffffLL)
    return hipErrorInvalidValue;
  FlashPlan f = flash_plan(n_work, n_tiles, true);
  if (f.part_bytes > p.part_bytes) f = flash_plan(n_work, n_tiles, false);
  p.n_whole = f.n_whole; p.n_chunk = f.n_chunk; p.n_bundle = f.n_bundle;
  const bool alpha_d = p.out_c != nullptr && p.alpha.p != nullptr && p.alpha.sd != 0;
  if (p.out.dtype == ICSA_DT_BF16)
    return alpha_d ? run_flash<true, true>(p, n_work, stream) : run_flash<true, false>(p, n_work, stream);
  return alpha_d ? run_flash<false, true>(p, n_work, stream) : run_flash<false, false>(p, n_work, stream);
}
