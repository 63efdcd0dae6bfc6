// Paged decode attention (one query token per sequence, GQA) on MFMA.
//
// A wave walks the 32-token tiles of a (sequence, kv head) item or of a part of it. Per tile, with the GQA
// group of G <= 16 query heads padded to 16 MFMA columns:
//   S^T[tok, head] = K[tok, :] . Q[head, :]^T   (mfma_f32_16x16x32_bf16, K rows as the A
//                                                operand straight from the cache: 16-B loads)
//   online softmax along tokens (exp2 domain; max across the 4 lane groups = 2 shuffles)
//   O[head, d] += P[head, tok] . V[tok, d]       (the S^T accumulator IS the A operand with a
//                                                permuted token order, so P never leaves
//                                                registers; the V tile is staged row-major in
//                                                a per-wave LDS tile and read as the B operand
//                                                with the transposing ds_read_b64_tr_b16, as
//                                                in the prefill kernel)
// Who takes what:
//   unsplit items, many of them     a wave each, 4 independent ones a workgroup (decode_attn_kernel)
//   unsplit items, up to 256        a workgroup each, its waves' partial results merged in LDS
//                                   (decode_attn_wg_kernel)
//   KV splits, head dim 128         a workgroup each, likewise (decode_attn_split_kernel)
//   KV splits, head dim 64          a wave each (decode_attn_kernel)
// With splits their (m, l, O) go to a workspace merged by decode_reduce_kernel. The decode graph's default
// are the fused forms of the first three (decode_attn_fused_kernel, decode_attn_split_kernel): the same tile
// loop after a prologue that replaces dli_splitk_rope_cache, in which the QKV GEMM's split-K slabs are
// reduced, q/k rotated and k/v written to the paged cache inside the attention wave.
//
// Layouts: q rows of stride q_stride (the fused QKV buffer), k_cache and v_cache
// [nblk,Hkv,bs,hd] (token-major: the per-step cache write is a contiguous row),
// block_tables [B, max_blocks], out [B, Hq, hd].
#include "common.h"
#include <limits.h>
#include <stdlib.h>
#include <type_traits>

#define DEC_WAVES 4
#define DEC_TILE 32
#define DEC_TARGET 3072
#define DEC_MIN_TILES 2

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));

// The tile loop shared by the plain and the fused kernel: one wave = one (sequence, kv head,
// split) item with its Q^T fragments already in registers.
// The tile loop over tokens [s_begin, s_end): leaves the unnormalised O rows in o_acc, the
// running max of head `col` in m_run and this lane's partial denominator in l_part.
// The first 64-block window of the block-table row of tokens [s_begin, s_end), one block id
// per lane (decode_attn_loop's bt_lane0): loaded by the caller so that the load can be
// issued ahead of the prologue's cache write and its fence.
__device__ __forceinline__ int decode_bt_window(const int* __restrict__ block_tables,
                                                int max_blocks, int b, int s_begin, int s_end,
                                                int block_size, int lane) {
  const int last_blk = max(s_end - 1, 0) / block_size;
  return block_tables[(long)b * max_blocks + min(s_begin / block_size + lane, last_blk)];
}

// [s_begin, s_end) of wave wv when WPI waves split the tokens [from, to) by whole tiles
template <int WPI>
__device__ __forceinline__ void decode_wg_range(int from, int to, int wv, int& s_begin, int& s_end) {
  const int tiles = (max(to - from, 0) + DEC_TILE - 1) / DEC_TILE;
  const int per = (tiles + WPI - 1) / WPI;
  s_begin = min(to, from + wv * per * DEC_TILE);
  s_end = min(to, s_begin + per * DEC_TILE);
}

// KV splits of a step, from its contexts, for units of W waves (head dim 128: a workgroup of 4; 64: a wave).
// Ragged contexts: split_tokens (whole tiles) deals the step's tiles to about decode_ragged_units units, so
// that one long context among short ones is cut as finely as the step can use; near-equal ones (the mean at
// least 3/4 of the longest) are cut in the power of two that gives 2048 waves or more, which leaves no
// short last split and CUs with equal shares (by waves, 64 x 1000 tokens: 59 us, dealt to DEC_TARGET 62; 24 of
// 500 - 8000: 62 us, cut like equal ones 101). At least DEC_MIN_TILES tiles a split, and no sequence takes
// more than num_splits. Sequence b has max(1, ceil(context / split_tokens)) equal ones, listed sequence
// by sequence: `pair` of that list is (b, split); b = -1 past its end. Every wave works this out for
// itself: a few loads and scans.
// A workgroup's split keeps 3 of a CU's 4 slots: about 768 run at once, half of one more a sequence and
// head is rounding (24 of 500 - 8000: 57.9 us dealt to 768 and the rounding up, 960 at most; 52.6 so).
template <int W> __host__ __device__ static inline int decode_ragged_units(int items) {
  return W == 1 ? DEC_TARGET : items < 768 ? 768 - items / 2 : 384;
}
template <int W> __host__ __device__ static inline int decode_even_splits(int items) {
  int n = 1;
  while ((long)items * n < 2048 / W) n *= 2;
  return n;
}
struct DecSplit { int b, split, split_tokens, last; };
// inclusive scan over the wave's lanes (values >= 0) by lane shifts in the registers
template <bool MAX>
__device__ __forceinline__ int wave_scan(int v) {
  const auto step = [&](int t) { v = MAX ? max(v, t) : v + t; };
  step(__builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false));   // row_shr 1, 2, 4, 8
  step(__builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false));
  step(__builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false));
  step(__builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false));
  step(__builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));   // row_bcast 15, 31
  step(__builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));
  return v;
}
template <int W>
__device__ __forceinline__ DecSplit decode_split(const int* __restrict__ context_lens, int B, int hkv,
                                                 int num_splits, int pair, int lane) {
  // the first 256 contexts stay in registers
  int ctx[4], sum = 0, longest = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) ctx[k] = 64 * k + lane < B ? context_lens[64 * k + lane] : 0;
  const auto count = [&](int c) {
    const int tiles = (c + DEC_TILE - 1) / DEC_TILE;
    sum += tiles;
    longest = max(longest, tiles);
  };
#pragma unroll
  for (int k = 0; k < 4; ++k) count(ctx[k]);
  for (int i = 256 + lane; i < B; i += 64) count(context_lens[i]);
  sum = __builtin_amdgcn_readlane(wave_scan<false>(sum), 63);
  longest = __builtin_amdgcn_readlane(wave_scan<true>(longest), 63);
  const int even = decode_even_splits<W>(B * hkv);
  const int share = 4l * sum >= 3l * longest * B ? (longest + even - 1) / even
                                                 : (sum * hkv + decode_ragged_units<W>(B * hkv) - 1) / decode_ragged_units<W>(B * hkv);
  const int per = max(max(share, (longest + num_splits - 1) / num_splits), max(W, DEC_MIN_TILES));
  DecSplit r{-1, 0, per * DEC_TILE, 0};
  const auto find = [&](int i0, int c) {
    const int n = i0 + lane < B ? max(1, (c + r.split_tokens - 1) / r.split_tokens) : 0;
    const int upto = wave_scan<false>(n);
    const unsigned long long past = __ballot(upto > pair);
    if (past) {
      const int l = __ffsll(past) - 1;
      r.b = i0 + l;
      r.last = __builtin_amdgcn_readlane(n, l) - 1;
      r.split = pair - (__builtin_amdgcn_readlane(upto, l) - 1 - r.last);
      // equal splits: a short last one, at the same place of every sequence's list, would fall to the
      // same XCDs (200 contexts of 700 - 1000, two splits each: 169 -> 164 us)
      const int tiles = (__builtin_amdgcn_readlane(c, l) + DEC_TILE - 1) / DEC_TILE;
      r.split_tokens = DEC_TILE * max(1, (tiles + r.last) / (r.last + 1));
    }
    pair -= __builtin_amdgcn_readlane(upto, 63);
    return past != 0;
  };
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (64 * k >= B || find(64 * k, ctx[k])) return r;
  for (int i0 = 256; i0 < B; i0 += 64)
    if (find(i0, i0 + lane < B ? context_lens[i0 + lane] : 0)) return r;
  return r;
}
// units a split launch needs at most: the even splits, or decode_ragged_units and the rounding up of every
// sequence
template <int W> static inline long decode_split_items(int items, int num_splits) {
  const long even = (long)items * decode_even_splits<W>(items), ragged = decode_ragged_units<W>(items) + items;
  const long all = (long)items * num_splits, most = even > ragged ? even : ragged;
  return all < most ? all : most;
}

template <int HD, bool PIPE>
__device__ __forceinline__ void decode_attn_loop(
    const bf16x8 (&qf)[HD / 32], u16* vt, int lane, int b, int kvh, int s_begin, int s_end,
    const u16* __restrict__ k_cache, const u16* __restrict__ v_cache,
    const int* __restrict__ block_tables, int max_blocks, int hkv, int block_size,
    float scale_log2, int bt_lane0, f32x4 (&o_acc)[HD / 16], float& m_run, float& l_part) {
  constexpr int DB = HD / 16;     // 16-wide output column blocks (= V pieces per lane)
  constexpr int KK = HD / 32;
  constexpr int VROW = HD + 16;   // padded LDS row of the V tile, in u16
  constexpr int VCH = HD / 8;     // 16-B chunks per V row
  const int col = lane & 15, grp = lane >> 4;
  const int* bt = block_tables + (long)b * max_blocks;
  // the split's block ids, one per lane, read once per 64-block window (token -> block by a
  // lane shuffle): the per-tile K/V loads no longer wait on a dependent block-table load
  const int last_blk = max(s_end - 1, 0) / block_size;
  int win = s_begin / block_size;
  int bt_lane = bt_lane0;
  const long kv_head_stride = (long)block_size * HD;           // elements per (blk, head)
  m_run = -INFINITY;                // running max for head `col` (replicated over groups)
  l_part = 0.f;                     // this lane's partial denominator for head `col`
#pragma unroll
  for (int i = 0; i < DB; ++i) o_acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};

  // PIPE: a tile's registers are refilled as soon as they are consumed, the keys behind the scores and
  // the values behind their LDS copy, so that the next tile's requests fly during this one's
  // arithmetic. It takes 150 registers, 3 waves a SIMD; unsplit items of short contexts do better
  // with 4 waves that load and compute in turn. 24 contexts of 500 to 8000 (266 MB) 54.1 -> 52.1 us, 64 of
  // 200 to 1900 48.9 -> 45.6.
  uint4 kreg[2][KK], vreg[DB];
  const auto load_k = [&](int t0) __attribute__((always_inline)) {
    if ((min(t0 + DEC_TILE, s_end) - 1) / block_size - win >= 64) {   // wave-uniform
      win = t0 / block_size;
      bt_lane = bt[min(win + lane, last_blk)];
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      int tok = t0 + 16 * s + col;
      tok = tok < s_end ? tok : s_end - 1;                     // clamp: always-written rows
      const int blk = __shfl(bt_lane, tok / block_size - win, 64), off = tok % block_size;
      const u16* kp = k_cache + ((long)blk * hkv + kvh) * kv_head_stride + (long)off * HD;
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) kreg[s][kk] = load16_once(kp + kk * 32 + grp * 8);
    }
  };
  // V rows t0 .. t0+31 (row-major, 16-B chunks; piece lane + 64m = row r, chunk c); behind load_k(t0)
  const auto load_v = [&](int t0) __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < DB; ++m) {
      const int piece = lane + 64 * m, r = piece / VCH, c = piece % VCH;
      const int tok = min(t0 + r, s_end - 1);                  // clamp: always-written rows
      const int blk = __shfl(bt_lane, tok / block_size - win, 64), off = tok % block_size;
      vreg[m] = load16_once(v_cache + ((long)blk * hkv + kvh) * kv_head_stride + (long)off * HD +
                            c * 8);
    }
  };
  if (PIPE && s_begin < s_end) {
    load_k(s_begin);
    load_v(s_begin);
  }
  for (int t0 = s_begin; t0 < s_end; t0 += DEC_TILE) {
    const bool more = PIPE && t0 + DEC_TILE < s_end;
    if (!PIPE) {
      load_k(t0);
      load_v(t0);
    }
    // ---- S^T = K . Q^T for the two 16-token subtiles
    f32x4 s_acc[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      s_acc[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < KK; ++kk)
        s_acc[s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            *reinterpret_cast<bf16x8*>(&kreg[s][kk]), qf[kk], s_acc[s], 0, 0, 0);
    }
    if (more) load_k(t0 + DEC_TILE);
    // lane holds S^T[tok = t0 + 16s + 4grp + r][head = col]
    float p[8];
    float tmax = -INFINITY;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int tok = t0 + 16 * s + 4 * grp + r;
        const float v = tok < s_end ? s_acc[s][r] * scale_log2 : -INFINITY;
        p[s * 4 + r] = v;
        tmax = fmaxf(tmax, v);
      }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
    const float m_new = fmaxf(m_run, tmax);
    const float alpha = exp2f(m_run - m_new);                  // m_run=-inf -> 0
    m_run = m_new;
    float psum = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) { p[j] = exp2f(p[j] - m_new); psum += p[j]; }
    l_part = l_part * alpha + psum;
    // rescale O rows (heads 4grp + r) by their head's alpha (held by lane 4grp + r)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float a = __shfl(alpha, 4 * grp + r, 64);
#pragma unroll
      for (int i = 0; i < DB; ++i) o_acc[i][r] *= a;
    }
    // stage the V tile in this wave's LDS rows (previous tile's reads retired below)
#pragma unroll
    for (int m = 0; m < DB; ++m) {
      const int piece = lane + 64 * m, r = piece / VCH, c = piece % VCH;
      *reinterpret_cast<uint4*>(vt + r * VROW + c * 8) = vreg[m];
    }
    if (more) load_v(t0 + DEC_TILE);
    // A operand: P[head=col][k = 8grp + j] in the permuted token order
    // pi(grp, j) = 16(j>>2) + 4grp + (j&3)
    bf16x8 pa;
#pragma unroll
    for (int j = 0; j < 8; ++j) pa[j] = (__bf16)p[j];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // V tile writes landed (same wave)
    // B operand: rows (tokens) 4grp+q and 16+4grp+q, columns 16i + 4p, transposed by
    // ds_read_b64_tr_b16 (lane 4q+p of each 16-lane group names row q, columns 4p..4p+3)
    const int qrow = (lane >> 2) & 3, pcol = lane & 3;
#pragma unroll
    for (int i = 0; i < DB; ++i) {
      const u16* a0 = vt + (4 * grp + qrow) * VROW + 16 * i + 4 * pcol;
      const u16* a1 = vt + (16 + 4 * grp + qrow) * VROW + 16 * i + 4 * pcol;
      s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) s16x4*)(a0));
      s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) s16x4*)(a1));
      s16x8 w = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      o_acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa, *reinterpret_cast<bf16x8*>(&w),
                                                        o_acc[i], 0, 0, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // reads done before next overwrite
  }
}

template <int HD, bool PIPE>
__device__ __forceinline__ void decode_attn_core(
    const bf16x8 (&qf)[HD / 32], u16* vt, int lane, int b, int kvh, int split, int G, int ctx,
    int s_begin, int s_end, u16* __restrict__ out, const u16* __restrict__ k_cache,
    const u16* __restrict__ v_cache, const int* __restrict__ block_tables, int max_blocks,
    int hq, int hkv, int block_size, float scale_log2, int num_splits,
    float* __restrict__ ws_o, float* __restrict__ ws_ml, int bt_lane0 = INT_MIN) {
  constexpr int DB = HD / 16;
  const int col = lane & 15, grp = lane >> 4;
  f32x4 o_acc[DB];
  float m_run, l_part;
  if (bt_lane0 == INT_MIN)
    bt_lane0 = decode_bt_window(block_tables, max_blocks, b, s_begin, s_end, block_size, lane);
  decode_attn_loop<HD, PIPE>(qf, vt, lane, b, kvh, s_begin, s_end, k_cache, v_cache, block_tables,
                       max_blocks, hkv, block_size, scale_log2, bt_lane0, o_acc, m_run, l_part);
  // ---- finalize: denominator of head `col`, then rows 4grp + r of O
  float l_tot = l_part + __shfl_xor(l_part, 16, 64);
  l_tot += __shfl_xor(l_tot, 32, 64);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int h = 4 * grp + r;
    const float lr = __shfl(l_tot, h, 64);
    const float mr = __shfl(m_run, h, 64);
    if (h >= G) continue;
    const int qh = kvh * G + h;
    const float inv = lr > 0.f ? 1.f / lr : 0.f;
    if (num_splits == 1) {
      u16* op = out + ((long)b * hq + qh) * HD;
#pragma unroll
      for (int i = 0; i < DB; ++i) op[16 * i + col] = f2bf(o_acc[i][r] * inv);
    } else {
      const long base = ((long)b * hq + qh) * num_splits + split;
      float* wo = ws_o + base * HD;
#pragma unroll
      for (int i = 0; i < DB; ++i) wo[16 * i + col] = o_acc[i][r] * inv;
      if (col == 0) {
        ws_ml[base * 2] = lr > 0.f ? mr : -INFINITY;
        ws_ml[base * 2 + 1] = lr;
      }
    }
  }}

// l = -1 ends the list for the reduce; a single split is the output itself and its list empty
__device__ __forceinline__ void decode_end_list(float* __restrict__ ws_ml, int b, int hq, int kvh,
                                                int G, int num_splits, int split, int last, int lane) {
  const int end = last == 0 ? 0 : split + 1;
  if (split == last && end < num_splits && lane < G)
    ws_ml[(((long)b * hq + kvh * G + lane) * num_splits + end) * 2 + 1] = -1.f;
}

// MINW = 4 waves per SIMD: <= 128 VGPRs, so every item of a 512-sequence batch (4096 waves)
// is resident at once (measured 7 % faster than the 166-VGPR / 2-waves build at ctx 66). A kernel of 2
// waves a SIMD that walked items and requested the next tile, across them too, served contexts of 768 and
// more until the loads here went past the caches: 256 of 984 195 us, this 168; 512 of 33 to 99 36, 33.
// Head dim 64, whose splits come here too: pipelined and past the caches; before, 24 contexts of 1000 and 12
// heads 27.6 us, so 23.4; 64 of 500 27.8, 24.3; 512 of 33 20.9, 17.7; one of 33 8.5, 7.3
template <int HD, int MINW, bool PIPE>
__global__ void __launch_bounds__(256, MINW) decode_attn_kernel(
    u16* __restrict__ out, const u16* __restrict__ q, int q_stride,
    const u16* __restrict__ k_cache, const u16* __restrict__ v_cache,
    const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ context_lens,
    int B, int hq, int hkv, int block_size, float scale_log2, int num_splits, int split_tokens,
    float* __restrict__ ws_o, float* __restrict__ ws_ml) {
  constexpr int KK = HD / 32;     // MFMA k-steps over head_dim
  constexpr int VROW = HD + 16;   // padded LDS row of the V tile, in u16
  __shared__ __attribute__((aligned(16))) u16 vtile_all[DEC_WAVES][DEC_TILE * VROW];
  u16* vt = vtile_all[threadIdx.x >> 6];
  const int lane = threadIdx.x & 63;
  // one WAVE per work item (sequence, kv head, at head dim 64 also KV split): no barriers, so every
  // resident wave of the chip streams a different (seq, head) pair concurrently
  const int item = blockIdx.x * DEC_WAVES + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kvh = item % hkv;
  DecSplit sp{item / hkv, 0, split_tokens, 0};
  // (head dim 128 with splits: decode_attn_split_kernel)
  const bool listed = HD == 64 && num_splits > 1;
  if (listed) sp = decode_split<1>(context_lens, B, hkv, num_splits, item / hkv, lane);
  if (sp.b < 0 || sp.b >= B) return;                           // wave-uniform exit
  const int b = sp.b, split = sp.split;
  split_tokens = sp.split_tokens;
  const int col = lane & 15, grp = lane >> 4;
  const int G = hq / hkv;
  const int ctx = context_lens[b];
  const int s_begin = split * split_tokens;
  const int s_end = min(ctx, s_begin + split_tokens);

  // Q^T fragments (B operand): head = col, dims 32kk + 8grp .. +7
  bf16x8 qf[KK];
  {
    const bool valid = col < G;
    const u16* qp = q + (long)b * q_stride + (long)(kvh * G + (valid ? col : 0)) * HD;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      uint4 v = valid ? *reinterpret_cast<const uint4*>(qp + kk * 32 + grp * 8)
                      : make_uint4(0, 0, 0, 0);
      qf[kk] = *reinterpret_cast<bf16x8*>(&v);
    }
  }
  decode_attn_core<HD, PIPE>(qf, vt, lane, b, kvh, split, G, ctx, s_begin, s_end, out, k_cache,
                       v_cache, block_tables, max_blocks, hq, hkv, block_size, scale_log2,
                       listed && sp.last > 0 ? num_splits : 1, ws_o, ws_ml);
  if (listed) decode_end_list(ws_ml, b, hq, kvh, G, num_splits, split, sp.last, lane);
}

// One (sequence, kv head) item, or one KV split of it, per workgroup of WPI waves: wave wv walks the
// wv-th of WPI equal slices of its 32-token tiles, then the partial (m, l, O) merge through
// LDS (each wave's V-tile rows are reused for its O partial) and the workgroup writes the
// GQA group's output rows. Small batches: with one item per wave most of the chip idles and
// each wave pays one HBM round trip per tile of the whole context.
template <int WPI>
__device__ __forceinline__ void decode_attn_wg(
    const bf16x8 (&qf)[4], u16 (*vtile_all)[DEC_TILE * 144], float (*ml_all)[16][2], int wv,
    int lane, int b, int kvh, int G, int s_begin, int s_end, int bt_lane0,
    u16* __restrict__ out, const u16* __restrict__ k_cache, const u16* __restrict__ v_cache,
    const int* __restrict__ block_tables, int max_blocks, int hq, int hkv, int block_size,
    float scale_log2, int num_splits = 1, int split = 0, float* __restrict__ ws_o = nullptr,
    float* __restrict__ ws_ml = nullptr) {
  constexpr int HD = 128, DB = HD / 16;
  static_assert(16 * HD * 4 <= DEC_TILE * 144 * 2, "O partials fit a wave's V tile");
  const int col = lane & 15, grp = lane >> 4;
  f32x4 o_acc[DB];
  float m_run, l_part;
  decode_attn_loop<HD, true>(qf, vtile_all[wv], lane, b, kvh, s_begin, s_end, k_cache, v_cache,
                       block_tables, max_blocks, hkv, block_size, scale_log2, bt_lane0, o_acc,
                       m_run, l_part);
  float l_tot = l_part + __shfl_xor(l_part, 16, 64);
  l_tot += __shfl_xor(l_tot, 32, 64);
  float* po = reinterpret_cast<float*>(vtile_all[wv]);
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int i = 0; i < DB; ++i) po[(4 * grp + r) * HD + 16 * i + col] = o_acc[i][r];
  if (grp == 0) {
    ml_all[wv][col][0] = m_run;
    ml_all[wv][col][1] = l_tot;
  }
  __syncthreads();
  // merge: thread t -> head t / 16, dims 8 (t % 16) .. +7
  const int h = threadIdx.x >> 4, d0 = (threadIdx.x & 15) * 8;
  if (h >= G) return;
  float M = -INFINITY;
#pragma unroll
  for (int w = 0; w < WPI; ++w) M = fmaxf(M, ml_all[w][h][0]);
  float den = 0.f, acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int w = 0; w < WPI; ++w) {
    const float mw = ml_all[w][h][0];
    const float e = mw == -INFINITY ? 0.f : exp2f(mw - M);
    den += e * ml_all[w][h][1];
    const float4* o4 = reinterpret_cast<const float4*>(
        reinterpret_cast<const float*>(vtile_all[w]) + h * HD + d0);
    const float4 a = o4[0], c = o4[1];
    acc[0] += e * a.x; acc[1] += e * a.y; acc[2] += e * a.z; acc[3] += e * a.w;
    acc[4] += e * c.x; acc[5] += e * c.y; acc[6] += e * c.z; acc[7] += e * c.w;
  }
  const float inv = den > 0.f ? 1.f / den : 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] *= inv;
  if (num_splits == 1) {
    store8(out + ((long)b * hq + kvh * G + h) * HD + d0, acc);
    return;
  }
  const long base = ((long)b * hq + kvh * G + h) * num_splits + split;
  float4* wo = reinterpret_cast<float4*>(ws_o + base * HD + d0);
  wo[0] = make_float4(acc[0], acc[1], acc[2], acc[3]);
  wo[1] = make_float4(acc[4], acc[5], acc[6], acc[7]);
  if (d0 == 0) {
    ws_ml[base * 2] = den > 0.f ? M : -INFINITY;
    ws_ml[base * 2 + 1] = den;
  }
}

// Small-batch form of decode_attn_kernel (head dim 128, one KV split): a workgroup per item.
__global__ void __launch_bounds__(256, 2) decode_attn_wg_kernel(
    u16* __restrict__ out, const u16* __restrict__ q, int q_stride,
    const u16* __restrict__ k_cache, const u16* __restrict__ v_cache,
    const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ context_lens,
    int B, int hq, int hkv, int block_size, float scale_log2) {
  constexpr int HD = 128, KK = HD / 32, VROW = HD + 16;
  __shared__ __attribute__((aligned(16))) u16 vtile_all[DEC_WAVES][DEC_TILE * VROW];
  __shared__ float ml_all[DEC_WAVES][16][2];
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int item = blockIdx.x;
  const int kvh = item % hkv, b = item / hkv;
  const int col = lane & 15, grp = lane >> 4;
  const int G = hq / hkv;
  bf16x8 qf[KK];
  {
    const bool valid = col < G;
    const u16* qp = q + (long)b * q_stride + (long)(kvh * G + (valid ? col : 0)) * HD;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      uint4 v = valid ? *reinterpret_cast<const uint4*>(qp + kk * 32 + grp * 8)
                      : make_uint4(0, 0, 0, 0);
      qf[kk] = *reinterpret_cast<bf16x8*>(&v);
    }
  }
  int s_begin, s_end;
  decode_wg_range<DEC_WAVES>(0, context_lens[b], wv, s_begin, s_end);
  const int bt0 = decode_bt_window(block_tables, max_blocks, b, s_begin, s_end, block_size, lane);
  decode_attn_wg<DEC_WAVES>(qf, vtile_all, ml_all, wv, lane, b, kvh, G, s_begin, s_end, bt0,
                            out, k_cache, v_cache, block_tables, max_blocks, hq, hkv,
                            block_size, scale_log2);
}

// Fused variants for the decode graph: the QKV GEMM's split-K slabs go straight into the attention
// wave instead of through dli_splitk_rope_cache. The item that holds the new token (sequence b, kv
// head h): lane l sums the slabs of this token's k and v for dims l and l + 64 of head h, rounds to
// bf16, rotates k (RoPE) and writes both into the paged cache at slot_mapping[b]. Every item builds
// its Q^T fragments (head col of the GQA group, dims 32kk + 8grp .. +7 and their RoPE partners 64
// apart, which the same lane holds) from the slabs. Numerics equal the unfused kernels: sum -> bf16
// -> rotate -> bf16. The q rows never go to memory, and one kernel per layer and its slab pass are
// gone.
// SPL > 0: src = the QKV GEMM's fp32 split-K slabs [SPL, B, N]; SPL == 0: the bf16 QKV rows [B, N] of
// an unsplit GEMM (the same prologue minus the slab sum). S16: the slabs are fp16 x 1/16 (EPI_SLAB16),
// read as 16-bit words.
template <int SPL, bool S16>
__device__ __forceinline__ void fused_query(bf16x8 (&qf)[4], const void* __restrict__ src,
                                            long rowoff, long splitstride,
                                            const float* __restrict__ cs, int kvh, int G, int lane) {
  constexpr int HD = 128, HALF = 64, KK = HD / 32;
  const float* ws = static_cast<const float*>(src);
  const u16* qkv = static_cast<const u16*>(src);
  const u16* ws16 = static_cast<const u16*>(src);
  const int col = lane & 15, grp = lane >> 4;
  // head col of the group, dims 32kk + 8grp .. +7 (kk < 2: first half, its RoPE partner is
  // fragment kk + 2 of the same lane)
  if (col < G) {
    const float* qp = ws + rowoff + (long)(kvh * G + col) * HD;
#pragma unroll
    for (int kp2 = 0; kp2 < KK / 2; ++kp2) {
      const int d1 = 32 * kp2 + 8 * grp;
      float x1[8] = {0, 0, 0, 0, 0, 0, 0, 0}, x2[8] = {0, 0, 0, 0, 0, 0, 0, 0};
      if constexpr (SPL == 0) {
        const u16* qr = qkv + rowoff + (long)(kvh * G + col) * HD;
        load8(qr + d1, x1);
        load8(qr + HALF + d1, x2);
      }
      if constexpr (S16) {
        const u16* qh = ws16 + rowoff + (long)(kvh * G + col) * HD;
        uint4 ua[SPL], uc[SPL];
#pragma unroll
        for (int s = 0; s < SPL; ++s) {
          ua[s] = *reinterpret_cast<const uint4*>(qh + s * splitstride + d1);
          uc[s] = *reinterpret_cast<const uint4*>(qh + s * splitstride + HALF + d1);
        }
#pragma unroll
        for (int s = 0; s < SPL; ++s) {
          float fa[8], fc[8];
          unpack8h(ua[s], fa);
          unpack8h(uc[s], fc);
#pragma unroll
          for (int j = 0; j < 8; ++j) { x1[j] += fa[j]; x2[j] += fc[j]; }
        }
      }
#pragma unroll
      for (int s = 0; s < (S16 ? 0 : SPL); ++s) {
        const float4* a = reinterpret_cast<const float4*>(qp + s * splitstride + d1);
        const float4* c = reinterpret_cast<const float4*>(qp + s * splitstride + HALF + d1);
        const float4 a0 = a[0], a1 = a[1], c0 = c[0], c1 = c[1];
        x1[0] += a0.x; x1[1] += a0.y; x1[2] += a0.z; x1[3] += a0.w;
        x1[4] += a1.x; x1[5] += a1.y; x1[6] += a1.z; x1[7] += a1.w;
        x2[0] += c0.x; x2[1] += c0.y; x2[2] += c0.z; x2[3] += c0.w;
        x2[4] += c1.x; x2[5] += c1.y; x2[6] += c1.z; x2[7] += c1.w;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float q1 = bf2f(f2bf(x1[j])), q2 = bf2f(f2bf(x2[j]));
        const float co = cs[d1 + j], si = cs[HALF + d1 + j];
        qf[kp2][j] = (__bf16)(q1 * co - q2 * si);
        qf[kp2 + 2][j] = (__bf16)(q2 * co + q1 * si);
      }
    }
  } else {
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      uint4 z = make_uint4(0, 0, 0, 0);
      qf[kk] = *reinterpret_cast<bf16x8*>(&z);
    }
  }
}

// this token's k (rotated) and v -> paged cache (lane: dims lane, lane + 64)
template <int SPL, bool S16>
__device__ __forceinline__ void fused_cache_row(const void* __restrict__ src, long rowoff,
                                                long splitstride, const float* __restrict__ cs,
                                                int slot, int kvh, int hq, int hkv, int block_size,
                                                u16* __restrict__ k_cache, u16* __restrict__ v_cache,
                                                int lane) {
  constexpr int HD = 128, HALF = 64;
  const float* ws = static_cast<const float*>(src);
  const u16* qkv = static_cast<const u16*>(src);
  const u16* ws16 = static_cast<const u16*>(src);
  const float* kp = ws + rowoff + (long)(hq + kvh) * HD;
  const float* vp = ws + rowoff + (long)(hq + hkv + kvh) * HD;
  float k1 = 0.f, k2 = 0.f, v1 = 0.f, v2 = 0.f;
  if constexpr (S16) {
    const u16* kh = ws16 + rowoff + (long)(hq + kvh) * HD;
    const u16* vh = ws16 + rowoff + (long)(hq + hkv + kvh) * HD;
#pragma unroll
    for (int s = 0; s < SPL; ++s) {
      k1 += h2f(kh[s * splitstride + lane]) * SLAB16_UNSCALE;
      k2 += h2f(kh[s * splitstride + HALF + lane]) * SLAB16_UNSCALE;
      v1 += h2f(vh[s * splitstride + lane]) * SLAB16_UNSCALE;
      v2 += h2f(vh[s * splitstride + HALF + lane]) * SLAB16_UNSCALE;
    }
  } else if constexpr (SPL > 0) {
#pragma unroll
    for (int s = 0; s < SPL; ++s) {
      k1 += kp[s * splitstride + lane];
      k2 += kp[s * splitstride + HALF + lane];
      v1 += vp[s * splitstride + lane];
      v2 += vp[s * splitstride + HALF + lane];
    }
  } else {
    const u16* kr = qkv + rowoff + (long)(hq + kvh) * HD;
    const u16* vr = qkv + rowoff + (long)(hq + hkv + kvh) * HD;
    k1 = bf2f(kr[lane]); k2 = bf2f(kr[HALF + lane]);
    v1 = bf2f(vr[lane]); v2 = bf2f(vr[HALF + lane]);
  }
  k1 = bf2f(f2bf(k1)); k2 = bf2f(f2bf(k2));
  const float co = cs[lane], si = cs[HALF + lane];
  const int blk = slot / block_size, off = slot - blk * block_size;
  const long dst = (((long)blk * hkv + kvh) * block_size + off) * HD;
  k_cache[dst + lane] = f2bf(k1 * co - k2 * si);
  k_cache[dst + HALF + lane] = f2bf(k2 * co + k1 * si);
  v_cache[dst + lane] = f2bf(v1);
  v_cache[dst + HALF + lane] = f2bf(v2);
}

// One KV split per item. WPI = 1: one wave per (sequence, kv head) item, 4 items per workgroup
// (large batches). WPI = DEC_WAVES: one workgroup per item for small batches, where 4 items per
// workgroup leave most of the chip idle and each wave walks the whole context serially (one HBM
// round trip per 32-token tile): wave 0 writes the new k/v row, every wave builds the Q fragments,
// wave w takes the w-th quarter of the context's tiles, and the partial (m, l, O) merge
// through LDS (the V-tile rows are reused for the O partials).
template <int SPL, int WPI, bool S16 = false>
__global__ void __launch_bounds__(256, WPI > 1 ? 2 : 4) decode_attn_fused_kernel(
    u16* __restrict__ out, const void* __restrict__ src, int N,
    const int* __restrict__ positions, const int* __restrict__ slot_mapping,
    const float* __restrict__ cos_sin, u16* __restrict__ k_cache, u16* __restrict__ v_cache,
    const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ context_lens,
    int B, int hq, int hkv, int block_size, float scale_log2) {
  constexpr int HD = 128, KK = HD / 32, VROW = HD + 16;
  static_assert(WPI == 1 || WPI == DEC_WAVES, "one item per wave or per workgroup");
  __shared__ __attribute__((aligned(16))) u16 vtile_all[DEC_WAVES][DEC_TILE * VROW];
  __shared__ float ml_all[WPI > 1 ? WPI : 1][16][2];
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  u16* vt = vtile_all[wv];
  const int lane = threadIdx.x & 63;
  const int item = WPI > 1 ? (int)blockIdx.x : (int)blockIdx.x * DEC_WAVES + wv;
  if (item >= B * hkv) return;                                 // wave-uniform exit (WPI 1)
  const int kvh = item % hkv, b = item / hkv;
  const int G = hq / hkv;
  const int ctx = context_lens[b];
  const float* cs = cos_sin + (long)positions[b] * HD;
  const long rowoff = (long)b * N;
  const long splitstride = (long)B * N;
  // first the query: its slab loads do not wait on the cache write below
  bf16x8 qf[KK];
  fused_query<SPL, S16>(qf, src, rowoff, splitstride, cs, kvh, G, lane);
  // the block-table window too: every load the tile loop's first tile waits on except the
  // new cache row is issued before the fence below
  int s_begin = 0, s_end = ctx;
  if constexpr (WPI > 1) decode_wg_range<WPI>(0, ctx, wv, s_begin, s_end);
  const int bt0 = decode_bt_window(block_tables, max_blocks, b, s_begin, s_end, block_size, lane);
  const int slot = slot_mapping[b];
  if (slot >= 0 && (WPI == 1 || wv == 0))
    fused_cache_row<SPL, S16>(src, rowoff, splitstride, cs, slot, kvh, hq, hkv, block_size, k_cache,
                              v_cache, lane);
  // the tile loop below reads this row back (other lanes of this wave): order the stores
  // before those loads
  __threadfence_block();
  if constexpr (WPI == 1) {
    decode_attn_core<HD, false>(qf, vt, lane, b, kvh, 0, G, ctx, 0, ctx, out, k_cache, v_cache,
                         block_tables, max_blocks, hq, hkv, block_size, scale_log2, 1, nullptr,
                         nullptr, bt0);
  } else {
    __syncthreads();                       // wave 0's cache row visible to the other waves
    decode_attn_wg<WPI>(qf, vtile_all, ml_all, wv, lane, b, kvh, G, s_begin, s_end, bt0, out,
                        k_cache, v_cache, block_tables, max_blocks, hq, hkv, block_size,
                        scale_log2);
  }
}

// Several KV splits per sequence, dealt to workgroups from the step's contexts: a split's 4 waves merge
// through LDS, so a context of up to 4 tiles is one split and its output, and a longer one leaves a
// quarter of the partial results. SPL >= 0, fused: the wave with the new token writes its cache row, the
// others do not read it; SPL < 0: src = the q rows (stride N), already rotated, the cache written.
// With its reduce, from a wave a split: 1 context of 75 tokens 12.0 -> 8.1 us, 1 of 2000 14.2 -> 10.9, 16 of
// 1000 22.6 -> 20.1, 32 of 2000 54.2 -> 52.5.
template <int SPL, bool S16>
__global__ void __launch_bounds__(256, 2) decode_attn_split_kernel(
    u16* __restrict__ out, const void* __restrict__ src, int N,
    const int* __restrict__ positions, const int* __restrict__ slot_mapping,
    const float* __restrict__ cos_sin, u16* __restrict__ k_cache, u16* __restrict__ v_cache,
    const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ context_lens,
    int B, int hq, int hkv, int block_size, float scale_log2, int num_splits,
    float* __restrict__ ws_o, float* __restrict__ ws_ml) {
  constexpr int HD = 128, KK = HD / 32, VROW = HD + 16;
  __shared__ __attribute__((aligned(16))) u16 vtile_all[DEC_WAVES][DEC_TILE * VROW];
  __shared__ float ml_all[DEC_WAVES][16][2];
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int kvh = blockIdx.x % hkv;
  const DecSplit sp = decode_split<DEC_WAVES>(context_lens, B, hkv, num_splits, blockIdx.x / hkv, lane);
  if (sp.b < 0) return;                                        // workgroup-uniform exit
  const int b = sp.b, split = sp.split, G = hq / hkv;
  const int ctx = context_lens[b];
  const int from = split * sp.split_tokens;
  int s_begin, s_end;
  decode_wg_range<DEC_WAVES>(from, min(ctx, from + sp.split_tokens), wv, s_begin, s_end);
  const int bt0 = decode_bt_window(block_tables, max_blocks, b, s_begin, s_end, block_size, lane);
  bf16x8 qf[KK];
  if constexpr (SPL < 0) {
    const int col = lane & 15, grp = lane >> 4;
    const u16* qp = static_cast<const u16*>(src) + (long)b * N + (long)(kvh * G + (col < G ? col : 0)) * HD;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      uint4 v = col < G ? *reinterpret_cast<const uint4*>(qp + kk * 32 + grp * 8) : make_uint4(0, 0, 0, 0);
      qf[kk] = *reinterpret_cast<bf16x8*>(&v);
    }
  } else {
    const float* cs = cos_sin + (long)positions[b] * HD;
    const long rowoff = (long)b * N;
    const long splitstride = (long)B * N;
    fused_query<SPL, S16>(qf, src, rowoff, splitstride, cs, kvh, G, lane);
    const int slot = slot_mapping[b];
    if (slot >= 0 && (ctx > 0 ? s_begin < ctx && s_end == ctx : wv == 0)) {
      fused_cache_row<SPL, S16>(src, rowoff, splitstride, cs, slot, kvh, hq, hkv, block_size, k_cache,
                                v_cache, lane);
      __threadfence_block();               // read back by other lanes of this wave
    }
  }
  decode_attn_wg<DEC_WAVES>(qf, vtile_all, ml_all, wv, lane, b, kvh, G, s_begin, s_end, bt0, out,
                            k_cache, v_cache, block_tables, max_blocks, hq, hkv, block_size, scale_log2,
                            sp.last == 0 ? 1 : num_splits, split, ws_o, ws_ml);
  if (wv == 0) decode_end_list(ws_ml, b, hq, kvh, G, num_splits, split, sp.last, lane);
}

// out[b, h, :] = sum_s w_s o_s / sum_s w_s,  w_s = exp2(m_s - M) * l_s, over the splits before the
// first one with l = -1; none: the row is there already. A wave per row, the splits' (m, l) one per
// lane, up to 16 splits' outputs in flight: what another XCD wrote comes from memory, and a row has
// up to 64 of them
template <int HD>
__global__ void __launch_bounds__(256) decode_reduce_kernel(u16* __restrict__ out,
                                                            const float* __restrict__ ws_o,
                                                            const float* __restrict__ ws_ml,
                                                            int B, int hq, int num_splits) {
  constexpr int E = HD / 64;                      // dims per lane
  const int lane = threadIdx.x & 63;
  const long bh = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (bh >= (long)B * hq) return;
  const float* ml = ws_ml + bh * num_splits * 2;
  float M = -INFINITY, den = 0.f, acc[E];
#pragma unroll
  for (int j = 0; j < E; ++j) acc[j] = 0.f;
  for (int s0 = 0; s0 < num_splits; s0 += 64) {
    float m = -INFINITY, l = -1.f;
    if (s0 + lane < num_splits) { m = ml[2 * (s0 + lane)]; l = ml[2 * (s0 + lane) + 1]; }
    const unsigned long long end = __ballot(l == -1.f);
    const int ns = end ? __ffsll(end) - 1 : 64;
    if (ns == 0) {
      if (s0 == 0) return;
      break;
    }
    if (lane >= ns) m = -INFINITY;
    float top = m;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) top = fmaxf(top, __shfl_xor(top, o, 64));
    top = fmaxf(top, M);
    const float old = top == -INFINITY ? 1.f : exp2f(M - top);
    den *= old;
#pragma unroll
    for (int j = 0; j < E; ++j) acc[j] *= old;
    M = top;
    const float w = lane >= ns || l == 0.f ? 0.f : exp2f(m - M) * l;
    const float* o = ws_o + (bh * num_splits + s0) * HD + lane * E;
    const auto batch = [&](auto depth, int s) {
      constexpr int U = decltype(depth)::value;
      float v[U][E];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int j = 0; j < E; ++j) v[u][j] = o[(long)min(s + u, ns - 1) * HD + j];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float ws = s + u < ns ? __shfl(w, (s + u) & 63, 64) : 0.f;
        den += ws;
#pragma unroll
        for (int j = 0; j < E; ++j) acc[j] += s + u < ns ? ws * v[u][j] : 0.f;   // (0 x inf is NaN)
      }
      return s + U;
    };
    for (int s = 0; s < ns;)
      s = ns - s > 4 ? batch(std::integral_constant<int, 16>{}, s)
                     : batch(std::integral_constant<int, 4>{}, s);
    if (ns < 64) break;
  }
  const float inv = den > 0.f ? 1.f / den : 0.f;
#pragma unroll
  for (int j = 0; j < E; ++j) out[bh * HD + lane * E + j] = f2bf(acc[j] * inv);
}

// a workgroup per (sequence, kv head) item while the items alone would leave most CUs idle
// (<= 256 items: B <= 32 at 8 kv heads), else a wave per item; tests force either form with
// dli_decode_set_form(1 = wave per item, DEC_WAVES = workgroup per item, 0 = automatic)
static int g_decode_form = 0;
extern "C" int dli_decode_set_form(int v) {
  const int old = g_decode_form;
  g_decode_form = v;
  return old;
}
static bool wg_form(long items) {
  return g_decode_form == DEC_WAVES || (g_decode_form != 1 && items <= 256);
}

extern "C" int dli_decode_attention(void* out, const void* q, int q_stride, const void* k_cache,
                                    const void* v_cache, const int* block_tables, int max_blocks,
                                    const int* context_lens, int B, int hq, int hkv, int hd,
                                    int block_size, float scale, int max_context, int num_splits,
                                    void* workspace, hipStream_t st) {
  if (B <= 0) return 0;
  if (hq % hkv || hq / hkv > 16 || block_size % 16 || (hd != 64 && hd != 128))
    return (int)hipErrorInvalidValue;
  if (num_splits < 1) num_splits = 1;
  if (num_splits > 1 && workspace == nullptr) return (int)hipErrorInvalidValue;
  int split_tokens = (max_context + num_splits - 1) / num_splits;
  split_tokens = ((split_tokens + DEC_TILE - 1) / DEC_TILE) * DEC_TILE;
  if (split_tokens <= 0) split_tokens = DEC_TILE;
  float* ws_o = (float*)workspace;
  float* ws_ml = ws_o ? ws_o + (long)B * hq * num_splits * hd : nullptr;
  const float scale_log2 = scale * 1.4426950408889634f;
  const long items = (long)B * hkv * num_splits;
  if (hd == 128 && num_splits == 1 && wg_form(items)) {
    decode_attn_wg_kernel<<<(int)items, 64 * DEC_WAVES, 0, st>>>(
        (u16*)out, (const u16*)q, q_stride, (const u16*)k_cache, (const u16*)v_cache,
        block_tables, max_blocks, context_lens, B, hq, hkv, block_size, scale_log2);
  } else if (hd == 128 && num_splits > 1) {
    decode_attn_split_kernel<-1, false><<<(int)decode_split_items<DEC_WAVES>(B * hkv, num_splits), 256, 0, st>>>(
        (u16*)out, q, q_stride, nullptr, nullptr, nullptr, (u16*)k_cache, (u16*)v_cache, block_tables,
        max_blocks, context_lens, B, hq, hkv, block_size, scale_log2, num_splits, ws_o, ws_ml);
  } else {
    const long listed = num_splits > 1 ? decode_split_items<1>(B * hkv, num_splits) : items;
    dim3 grid((int)((listed + DEC_WAVES - 1) / DEC_WAVES));
    if (hd == 128)
      decode_attn_kernel<128, 4, false><<<grid, 64 * DEC_WAVES, 0, st>>>(
          (u16*)out, (const u16*)q, q_stride, (const u16*)k_cache, (const u16*)v_cache,
          block_tables, max_blocks, context_lens, B, hq, hkv, block_size, scale_log2, num_splits,
          split_tokens, ws_o, ws_ml);
    else
      decode_attn_kernel<64, 1, true><<<grid, 64 * DEC_WAVES, 0, st>>>(
          (u16*)out, (const u16*)q, q_stride, (const u16*)k_cache, (const u16*)v_cache,
          block_tables, max_blocks, context_lens, B, hq, hkv, block_size, scale_log2, num_splits,
          split_tokens, ws_o, ws_ml);
  }
  if (num_splits > 1) {
    const int blocks = (int)(((long)B * hq + 3) / 4);
    if (hd == 128)
      decode_reduce_kernel<128><<<blocks, 256, 0, st>>>((u16*)out, ws_o, ws_ml, B, hq, num_splits);
    else
      decode_reduce_kernel<64><<<blocks, 256, 0, st>>>((u16*)out, ws_o, ws_ml, B, hq, num_splits);
  }
  DLI_RETURN_LAUNCH();
}

// Fused split-K QKV reduce + RoPE + KV-cache write + decode attention (head dim 128, RoPE models; workspace
// as dli_decode_attention's where num_splits > 1, apart from ws): one launch, and the splits' merge where
// there are some. ws = the QKV GEMM's fp32 slabs [splits, B, (hq + 2 hkv) * 128], or with splits == 0 the bf16 QKV rows [B, (hq + 2 hkv) * 128] of an unsplit GEMM.
// fmt: 0 = fp32 slabs (or the bf16 rows when splits == 0), 1 = fp16 x 1/16 slabs (EPI_SLAB16)
extern "C" int dli_decode_attention_fused(void* out, const void* ws, int splits,
                                          const int* positions, const int* slot_mapping,
                                          const float* cos_sin, void* k_cache, void* v_cache,
                                          const int* block_tables, int max_blocks,
                                          const int* context_lens, int B, int hq, int hkv,
                                          int hd, int block_size, float scale, int fmt,
                                          int num_splits, void* workspace, hipStream_t st) {
  if (B <= 0) return 0;
  if (hd != 128 || hq % hkv || hq / hkv > 16 || block_size % 16 ||
      (splits != 0 && splits != 2 && splits != 4) || fmt < 0 || fmt > 1 ||
      (fmt == 1 && splits == 0) || num_splits < 1 || (num_splits > 1 && workspace == nullptr))
    return (int)hipErrorInvalidValue;
  const int N = (hq + 2 * hkv) * hd;
  const float scale_log2 = scale * 1.4426950408889634f;
  const long items = (long)B * hkv;
  if (num_splits > 1) {
    float* ws_o = (float*)workspace;
    float* ws_ml = ws_o + (long)B * hq * num_splits * hd;
    const dim3 gs((int)decode_split_items<DEC_WAVES>(B * hkv, num_splits));
#define DLI_DAS(S, F) decode_attn_split_kernel<S, F><<<gs, 64 * DEC_WAVES, 0, st>>>(     \
      (u16*)out, ws, N, positions, slot_mapping, cos_sin, (u16*)k_cache, (u16*)v_cache,      \
      block_tables, max_blocks, context_lens, B, hq, hkv, block_size, scale_log2, num_splits,  \
      ws_o, ws_ml)
    if (splits == 0) DLI_DAS(0, false);
    else if (splits == 2) { if (fmt) DLI_DAS(2, true); else DLI_DAS(2, false); }
    else { if (fmt) DLI_DAS(4, true); else DLI_DAS(4, false); }
#undef DLI_DAS
    decode_reduce_kernel<128><<<(int)(((long)B * hq + 3) / 4), 256, 0, st>>>(
        (u16*)out, ws_o, ws_ml, B, hq, num_splits);
    DLI_RETURN_LAUNCH();
  }
  const bool per_wg = wg_form(items);
  dim3 grid((int)(per_wg ? items : (items + DEC_WAVES - 1) / DEC_WAVES));
#define DLI_DAF(S, W, F) decode_attn_fused_kernel<S, W, F><<<grid, 64 * DEC_WAVES, 0, st>>>(   \
      (u16*)out, ws, N, positions, slot_mapping, cos_sin, (u16*)k_cache, (u16*)v_cache,      \
      block_tables, max_blocks, context_lens, B, hq, hkv, block_size, scale_log2)
  if (per_wg) {
    if (splits == 0) DLI_DAF(0, DEC_WAVES, false);
    else if (splits == 2) { if (fmt) DLI_DAF(2, DEC_WAVES, true); else DLI_DAF(2, DEC_WAVES, false); }
    else { if (fmt) DLI_DAF(4, DEC_WAVES, true); else DLI_DAF(4, DEC_WAVES, false); }
  } else {
    if (splits == 0) DLI_DAF(0, 1, false);
    else if (splits == 2) { if (fmt) DLI_DAF(2, 1, true); else DLI_DAF(2, 1, false); }
    else { if (fmt) DLI_DAF(4, 1, true); else DLI_DAF(4, 1, false); }
  }
#undef DLI_DAF
  DLI_RETURN_LAUNCH();
}

extern "C" long dli_decode_attention_workspace_bytes(int B, int hq, int hd, int num_splits) {
  if (num_splits <= 1) return 0;
  return (long)B * hq * num_splits * (hd + 2) * (long)sizeof(float);
}
