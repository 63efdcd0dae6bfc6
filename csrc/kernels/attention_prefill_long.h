// Causal GQA prefill attention of long sequences, head_dim 128: one wave a SIMD, 64 query rows a wave, the softmax
// of a key tile beside the matrix products of the next (attention_prefill.hip has the others and chooses).
//
// Swapped products, so that no value but a row's maximum moves between lanes (v_mfma_f32_32x32x16_bf16):
//   S^T[key, q] = K . Q^T     A: K rows from LDS, B: Q^T in registers; a lane owns the queries qc and 32 + qc and half
//                             of a tile's 64 keys of each
//   O^T[d, q] += V^T . P^T    P^T is S^T's accumulator rounded to bf16; V^T by transposing LDS reads
//
// What bounds it: the power budget (8000 tokens: 1.67 GHz, 3400 cycles a tile, of which 2048 are MFMAs) and one wave's
// issue of what stands beside the MFMAs (a tile's 64 exponentials with their fma, add and half a packing each, 32
// max3, 48 LDS reads, 8 LDS-DMA pieces; none alone is worth more than 10 %). The kernel of 8 waves of 32 rows, which
// met at a barrier a tile, read K and V from LDS twice as often and did products and softmax by turns. Here the
// products S(t + 1) run beside the exponentials of tile t, the products with V(t) beside the last of them and the
// maxima of t + 1. 32 heads on 8, us, that kernel / this one: 3000 tokens 97 / 87, 7993 516 / 471 (1.11 PFLOP/s), 16000 1930 / 1718, 4
// x 4096 577 / 525; on another card 4096 of 8192 cached 416 / 389. Outputs are equal to the bit.
//
// A workgroup's fixed cost was 11 k cycles ahead of the first product and 6 k behind the last: queries read a row a
// lane, outputs stored 8 bytes a row, 32 rows a request. Both go through a tile image a wave in LDS now, in whole rows;
// and a cached tile's 130 scalar instructions (four cycles each beside the products) are 40 and 24 lane reads: 4 x 2048
// tokens 160 -> 150 us, 8000 473 -> 460, 2 x 2048 of 4096 cached 208 -> 193, 4096 of 8192 384 -> 367.
//
// PAIRED (launches of up to a workgroup a CU): a wave's 64 rows are 32 of a half block counted from a sequence's start and
// 32 of its counterpart from the end. Once the former see no more keys the wave goes on with the latter alone, an iteration
// of half the products (2.1 k cycles a tile, 3.2 k with both): the workgroups' work is nearly equal, where whole
// blocks would wait for the last. 32 heads on 8, us, the other kernel's pairs / these: 1024 tokens 30.1 / 25.0, 2048 51.9
// / 44.7, 512 of 2560 cached 77.8 / 66.0, 2048 of 4096 121 / 106, 8 heads and 8000 tokens 163 / 139. Equal to the bit.
//
// K and V tiles come by LDS-DMA into rings of three slots, rows past the keys as zeros (range-checked descriptors).
// In iteration t K(t + 1) and V(t) are read, K(t + 2) and V(t + 1) land, K(t + 3) and V(t + 2) are requested; the
// only barrier, once the last of V(t) is read, ends all three. Causal: a workgroup's tiles stop at its last row's
// bound, a wave's at its own; only tiles that cross a wave's diagonal or the last key are masked.
#pragma once
#include "lds_dma.h"

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef const __attribute__((address_space(3))) bf16x8 lds_frag;

__device__ __forceinline__ float max3_raw(float a, float b, float c) {  // no canonicalise
  float r;
  asm volatile("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

constexpr int HD = 128, KT = 64, ROWS = 256;
constexpr int SLOT = KT * HD * 2;                  // bytes of a K (or V) tile
constexpr float RESCALE_THR = 8.f;                 // log2 units: a running max is raised only by more than this

// Where keys and values are: the activation's rows, or blocks of the paged cache, of a power of two of at least 16
// tokens (others take the kernel of 8 waves).
enum { ROWS_OF_QKV = 0, BLOCKS_OF_16 = 1 };

template <int SRC, bool PAIRED>
__global__ void __launch_bounds__(256, 1) prefill_long_kernel(
    u16* __restrict__ out, int out_stride, const u16* __restrict__ qkv, int row_stride,
    const int* __restrict__ cu_seqlens, int hq, int hkv, float scale_log2,
    const int* __restrict__ ctx_lens, const u16* __restrict__ k_cache,
    const u16* __restrict__ v_cache, const int* __restrict__ block_tables, int bt_stride,
    int block_size, int block_shift) {
  extern __shared__ __attribute__((aligned(16))) char smem[];        // 3 K slots, 3 V slots, from address 0; a tile image a wave
  // Workgroups of a sequence: key heads fastest (round-robin over the XCDs: with 8 of them one L2
  // holds one head's K and V), then the query heads of a group, then row blocks, longest first over
  // all heads. Up to 4 heads leave too few of a sequence's blocks in flight before its empty ones come; there a
  // head's blocks of all sequences follow each other.
  const bool by_head = gridDim.z > 1;
  const int seq = blockIdx.y, G = hq / hkv;
  const int h = by_head ? blockIdx.z : blockIdx.x % hkv * G + blockIdx.x / hkv % G, kvh = h / G;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qc = lane & 31, hi = lane >> 5;
  const int s0 = __builtin_amdgcn_readfirstlane(cu_seqlens[seq]);
  const int len = __builtin_amdgcn_readfirstlane(cu_seqlens[seq + 1]) - s0;
  const int nblk = (len + ROWS - 1) / ROWS;
  const int blk = (int)((gridDim.x - 1 - blockIdx.x) / (by_head ? 1 : hq));
  if (blk >= nblk) return;                                           // workgroup-uniform
  const int nkeys = SRC ? __builtin_amdgcn_readfirstlane(ctx_lens[seq]) : len;
  const int qoff = nkeys - len;
  // this wave's two blocks of 32 rows: their first rows, and the tiles that both take part in, and one of them. Paired,
  // they are of a half block counted from the start and its counterpart from the end (the middle one of an odd number alone)
  const int nhalf = (len + ROWS / 2 - 1) / (ROWS / 2), front = nblk - 1 - blk, back = nhalf - 1 - front;
  const int row0[2] = {PAIRED ? front * (ROWS / 2) + wid * 32 : blk * ROWS + wid * 64,
                       PAIRED ? back * (ROWS / 2) + wid * 32 : blk * ROWS + wid * 64 + 32};
  const bool has0 = (!PAIRED || front != back) && row0[0] < len, active = has0 || (PAIRED && row0[1] < len);
  const int end1 = (qoff + min(row0[1] + 32, len) - 1) / KT + 1;     // (unpaired, a wave's last block is behind its first)
  const int both = !has0 ? 0 : PAIRED ? (qoff + min(row0[0] + 32, len) - 1) / KT + 1 : end1;
  const int mine = PAIRED && row0[1] < len ? max(both, end1) : both;
  const int kend = min(nkeys, qoff + min(PAIRED ? (back + 1) * (ROWS / 2) : (blk + 1) * ROWS, len));
  const int ntiles = (kend + KT - 1) / KT;

  // ---- staging: a tile is 16 pieces of 1 KiB (two of the 8-row x 32-column subtiles of 512 B, the XOR image
  // of attention_prefill.hip's pl_off); wave w moves pieces w + 4 j of K and of V, j = 0..3: rows 16 j + rw
  const int rw = 8 * (wid >> 1) + ((lane & 31) >> 2);
  const int cw = 4 * (2 * (wid & 1) + (lane >> 5)) + ((lane & 3) ^ ((rw >> 2) & 3));
  const int stride = SRC ? HD * 2 : row_stride * 2;                  // bytes of a row
  const int voff = rw * stride + cw * 16;
  const int* btab = SRC ? block_tables + (long)seq * bt_stride : nullptr;
  // where K's and V's rows of this head begin
  const u16* const first_k = SRC ? k_cache + (long)kvh * block_size * HD : qkv + (long)s0 * row_stride + (long)(hq + kvh) * HD;
  const u16* const first_v = SRC ? v_cache + (long)kvh * block_size * HD : first_k + hkv * HD;
  // (in scalar registers from here on: a descriptor formed beside its request from vector ones would need wait states
  // that nobody puts ahead of an asm statement)
  auto uniform = [](const u16* p) __attribute__((always_inline)) -> uintptr_t {
    return (uintptr_t)scalar((uint32_t)(uintptr_t)p) | (uintptr_t)scalar((uint32_t)((uintptr_t)p >> 32)) << 32;
  };
  const uintptr_t heads[2] = {uniform(first_k), uniform(first_v)};
  // Rows: one descriptor a sequence and operand, the tile in the scalar offset. Blocks: a descriptor a piece, of sixteen
  // rows; a lane holds those of a sixteen (scalar arithmetic costs issue cycles beside the MFMAs), for 15 tiles at a time
  // and the one before them, which V's pieces are of
  const int total = __builtin_amdgcn_readfirstlane((nkeys - 1) * stride + HD * 2);                   // (the launcher keeps a sequence's below 2^31)
  int row_at[2] = {0, 0};                                            // [K's tile, V's tile]
  int held = 0, place = 0, held_bytes = 0;                           // lane 0's sixteen, the lane of the first of K's tile
  uint32_t held_lo[2] = {0, 0}, held_hi[2] = {0, 0};
  auto hold = [&](int from) __attribute__((always_inline)) {
    held = from;
    const int first = 16 * (held + lane);
    const int id = btab[min(first, nkeys - 1) >> block_shift];
    const long at = (long)id * ((long)hkv * block_size * HD * 2) + (first & (block_size - 1)) * (HD * 2);
#pragma unroll
    for (int kv = 0; kv < 2; ++kv) {
      held_lo[kv] = (uint32_t)(heads[kv] + at);
      held_hi[kv] = (uint32_t)((heads[kv] + at) >> 32) & 0xffff;
    }
    held_bytes = min(max(nkeys - first, 0), 16) * (HD * 2);
  };
  // the tile that K's pieces are of next; V's are of the one before
  auto find = [&](int t) __attribute__((always_inline)) {
    if constexpr (SRC == BLOCKS_OF_16) {
      if (4 * t + 4 - held > 64) hold(4 * t - 4);                    // wave-uniform
      place = 4 * t - held;
    } else {
      row_at[1] = row_at[0];
      row_at[0] = t * (KT * stride);
    }
  };
  // (inline asm: behind the builtin hipcc waits for every LDS-DMA in flight ahead of a transposing read. It has no
  // result, and what it has written is read behind counted waits and a barrier)
  // (beside the products every scalar instruction costs; elsewhere the wait states of a descriptor out of vector registers)
  auto dma = [&](auto BESIDE, uint32_t dst, auto FURTHER, int lane_at, const u32x4& r, uint32_t so) __attribute__((always_inline)) {
    if constexpr (decltype(BESIDE)::value)
      asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, %4 offen lds"
                   :: "s"(dst), "i"(decltype(FURTHER)::value), "v"(lane_at), "s"(r), "s"(so) : "memory", "m0", "scc");
    else
      asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 4\n\tbuffer_load_dwordx4 %2, %3, %4 offen lds"
                   :: "s"(dst), "i"(decltype(FURTHER)::value), "v"(lane_at), "s"(r), "s"(so) : "memory", "m0", "scc");
  };
  // a piece's descriptor, and the piece to the slot at dst - wid KiB
  auto where = [&](auto J, auto KV) __attribute__((always_inline)) -> u32x4 {
    constexpr int j = decltype(J)::value, kv = decltype(KV)::value;
    if constexpr (SRC == BLOCKS_OF_16) {
      const int l = place - 4 * kv + j;
      return u32x4{(uint32_t)__builtin_amdgcn_readlane((int)held_lo[kv], l), (uint32_t)__builtin_amdgcn_readlane((int)held_hi[kv], l),
                   (uint32_t)__builtin_amdgcn_readlane(held_bytes, l), 0x00020000};
    } else {
      return bytes_at(heads[kv], total);
    }
  };
  auto piece = [&](auto J, auto KV, auto BESIDE, uint32_t dst, const u32x4& r) __attribute__((always_inline)) {
    constexpr int j = decltype(J)::value, kv = decltype(KV)::value;
    dma(BESIDE, dst, int_c<4096 * j>{}, voff, r,
        SRC == BLOCKS_OF_16 ? 0 : scalar((uint32_t)(row_at[kv] + j * 16 * stride)));
  };
  using K_ = int_c<0>;
  using V_ = int_c<1>;
  constexpr uint32_t V0 = 3 * SLOT, Q0 = 6 * SLOT;
  auto stage = [&](auto KV, uint32_t slot) __attribute__((always_inline)) {
    const uint32_t dst = scalar(slot + wid * 1024);
    unroll<4>([&](auto J) __attribute__((always_inline)) { piece(J, KV, int_c<0>{}, dst, where(J, KV)); });
  };
  if constexpr (SRC == BLOCKS_OF_16) hold(0);
  find(0);
  stage(K_{}, 0);
  // this wave's queries, to a tile image of their own (a row a lane would take 32 rows a request)
  const uint32_t mine_at = scalar(Q0 + wid * SLOT);
  unroll<2>([&](auto QB) __attribute__((always_inline)) {
    constexpr int qb = decltype(QB)::value;
    const int left = min(max(len - row0[qb], 0), 32), rl = (lane & 31) >> 2;
    const u32x4 r = bytes_at((uintptr_t)(qkv + (long)(s0 + row0[qb]) * row_stride + (long)h * HD),
                               left > 0 ? (left - 1) * row_stride * 2 + HD * 2 : 0);
    const int at = rl * row_stride * 2 + 64 * (lane >> 5);
    const int even = at + 16 * ((lane & 3) ^ (rl >> 2)), odd = at + 16 * ((lane & 3) ^ (2 + (rl >> 2)));
    unroll<8>([&](auto I) __attribute__((always_inline)) {
      constexpr int i = decltype(I)::value;
      dma(int_c<0>{}, mine_at, int_c<8192 * qb + 1024 * i>{}, (i >> 1) & 1 ? odd : even, r,
          scalar((uint32_t)((i >> 1) * 8 * row_stride * 2 + 128 * (i & 1))));
    });
  });
  find(1);
  stage(V_{}, V0);
  stage(K_{}, SLOT);
  find(2);
  stage(V_{}, V0 + SLOT);
  stage(K_{}, 2 * SLOT);
  asm volatile("s_waitcnt vmcnt(16)" ::: "memory");                  // K(0) and Q landed
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");

  // LDS read bases: K row reads of row 32 sub + qc, chunk 2 c + hi; transposed V reads by 16-lane group g16, lane
  // (q4, p4) of the group: rows 16 ks + 4 hi + q4 (+ 8)
  const int g16 = lane >> 4, q4 = (lane >> 2) & 3, p4 = lane & 3;
  uint32_t kb[2], vb[2];
#pragma unroll
  for (int par = 0; par < 2; ++par)
    kb[par] = 2048 * (qc >> 3) + 64 * (qc & 7) + 16 * ((2 * par + hi) ^ ((qc >> 2) & 3));
  {
    const int cl = 2 * (g16 & 1) + (p4 >> 1);
    vb[0] = V0 + 64 * (4 * hi + q4) + 16 * (cl ^ hi) + 8 * (p4 & 1);
    vb[1] = V0 + 2048 + 64 * (4 * hi + q4) + 16 * (cl ^ (hi ^ 2)) + 8 * (p4 & 1);
  }
  // Q^T operand: lane (query qc, half hi) holds Q[q][16 c + 8 hi .. + 7]
  bf16x8 qf[2][8];
#pragma unroll
  for (int qb = 0; qb < 2; ++qb)
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const bf16x8 v = *(lds_frag*)(kb[c & 1] + mine_at + 8192 * qb + 512 * (c >> 1));
      asm volatile("" : "=a"(qf[qb][c]) : "0"(v));
    }
  // the slots of tiles t, t + 1 and t + 2: K(t + 3) goes to the first, V(t + 2) to the last
  uint32_t slot[3] = {0, SLOT, 2 * SLOT};
  auto turn = [&]() {
    const uint32_t x = slot[0];
    slot[0] = slot[1];
    slot[1] = slot[2];
    slot[2] = x;
  };
  uint32_t ka[2], va[2];                                 // the read bases in the slots read
  auto k_base = [&](uint32_t slot) {
    ka[0] = kb[0] + slot, ka[1] = kb[1] + slot;
    asm volatile("" : "+v"(ka[0]), "+v"(ka[1]));
  };
  auto v_base = [&](uint32_t slot) {
    va[0] = vb[0] + slot, va[1] = vb[1] + slot;
    asm volatile("" : "+v"(va[0]), "+v"(va[1]));
  };
  auto kfrag = [&](auto F) __attribute__((always_inline)) -> bf16x8 {
    constexpr int f = decltype(F)::value, c = f >> 1, sub = f & 1;
    return *(lds_frag*)(ka[c & 1] + 8192 * sub + 512 * (c >> 1));
  };
  auto vfrag = [&](auto F) __attribute__((always_inline)) -> bf16x8 {
    constexpr int f = decltype(F)::value, ks = f >> 2, db = f & 3;
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) s16x4*)(va[0] + 4096 * ks + 512 * db));
    const s16x4 up = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) s16x4*)(va[1] + 4096 * ks + 512 * db));
    const s16x8 w = {lo[0], lo[1], lo[2], lo[3], up[0], up[1], up[2], up[3]};
    return __builtin_bit_cast(bf16x8, w);
  };
  auto fence = [&]() __attribute__((always_inline)) { __builtin_amdgcn_sched_barrier(0); };

  f32x16 o[2][4];
#pragma unroll
  for (int qb = 0; qb < 2; ++qb)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f32x16 zero = {};
      asm volatile("" : "=a"(o[qb][i]) : "0"(zero));
    }
  f32x16 s[2][2][2];                               // [tile parity][sub][qb]
  float m_run[2] = {-INFINITY, -INFINITY}, l_run[2] = {0.f, 0.f}, alpha[2] = {1.f, 1.f}, mc[2] = {0.f, 0.f};
  float top[2];

  // The products are inline asm, O and Q in the AGPR file; what reads their results stands many MFMAs behind them or
  // behind a pad of wait states, and fences keep it there
  auto mma_s = [&](f32x16& d, const bf16x8& a, const bf16x8& b, auto FIRST, auto FROM) __attribute__((always_inline)) {
    if constexpr (decltype(FIRST)::value && decltype(FROM)::value)     // (its registers may have been written just before)
      asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "a"(b));
    else if constexpr (decltype(FIRST)::value)
      asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "a"(b));
    else
      asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(d) : "v"(a), "a"(b));
  };
  auto pad = [&]() __attribute__((always_inline)) {
    fence();
    asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");
    fence();
  };
  // scores of keys that a lane's queries (from query block FROM on) do not see
  auto mask = [&](auto P, auto FROM, int t) __attribute__((always_inline)) {
    constexpr int p = decltype(P)::value, from = decltype(FROM)::value;
    const int k0 = t * KT;
    if (k0 + KT - 1 > qoff + row0[from] || k0 + KT > nkeys) {
      unroll<2 - from>([&](auto QB) __attribute__((always_inline)) {
        constexpr int qb = from + decltype(QB)::value;
        const int last = min(qoff + row0[qb] + qc, nkeys - 1) - k0 - 4 * hi;   // in steps of this lane's keys
        unroll<32>([&](auto R) __attribute__((always_inline)) {
          constexpr int sub = decltype(R)::value >> 4, r = decltype(R)::value & 15;
          if (32 * sub + (r & 3) + 8 * (r >> 2) > last) s[p][sub][qb][r] = -INFINITY;
          if constexpr (r % 4 == 3) fence();
        });
      });
    }
  };
  // step i of 32 of the maxima over a tile's scores, the two query blocks' chains in turn
  auto max_step = [&](auto P, auto I) __attribute__((always_inline)) {
    constexpr int p = decltype(P)::value, i = decltype(I)::value >> 1, qb = decltype(I)::value & 1;
    const f32x16 &a = s[p][0][qb], &b = s[p][1][qb];
    if constexpr (i == 0) top[qb] = max3_raw(a[0], a[1], a[2]);
    else if constexpr (i < 7) top[qb] = max3_raw(top[qb], a[2 * i + 1], a[2 * i + 2]);
    else if constexpr (i == 7) top[qb] = max3_raw(top[qb], a[15], b[0]);
    else if constexpr (i < 15) top[qb] = max3_raw(top[qb], b[2 * i - 15], b[2 * i - 14]);
    else top[qb] = max3_raw(top[qb], b[15], b[15]);
  };
  // the running maximum, in five steps: it moves only when the tile's exceeds it by more than 2^RESCALE_THR, so that
  // P <= 2^8 and O^T is rescaled for few tiles
  float rise[2];
  bool up[2];
  auto running_max = [&](auto I, auto FROM) __attribute__((always_inline)) {
#pragma unroll
    for (int qb = decltype(FROM)::value; qb < 2; ++qb) {
      constexpr int i = decltype(I)::value;
      if constexpr (i == 0) {
        const auto w = __builtin_amdgcn_permlane32_swap(__float_as_uint(top[qb]), __float_as_uint(top[qb]), false, false);
        top[qb] = max3_raw(__uint_as_float(w[0]), __uint_as_float(w[1]), __uint_as_float(w[1]));
      } else if constexpr (i == 1) {
        rise[qb] = (top[qb] - m_run[qb]) * scale_log2;
      } else if constexpr (i == 2) {
        up[qb] = rise[qb] > RESCALE_THR;
        alpha[qb] = __builtin_amdgcn_exp2f(-rise[qb]);
      } else if constexpr (i == 3) {
        alpha[qb] = up[qb] && m_run[qb] != -INFINITY ? alpha[qb] : 1.f;   // (nothing to rescale in the first tile)
        m_run[qb] = up[qb] ? top[qb] : m_run[qb];
      } else {
        mc[qb] = m_run[qb] == -INFINITY ? 0.f : m_run[qb] * scale_log2;
      }
    }
  };

  constexpr int DEEP = 4;                          // fragments read ahead of their products
  bf16x8 kf[DEEP], vf[DEEP];

  // S(0) and its maximum
  if (mine > 0) {
    k_base(0);
    unroll<16>([&](auto F) __attribute__((always_inline)) {
      constexpr int f = decltype(F)::value;
      const bf16x8 a = kfrag(F);
      mma_s(s[0][f & 1][0], a, qf[0][f >> 1], std::integral_constant<bool, (f < 2)>{}, int_c<0>{});
      mma_s(s[0][f & 1][1], a, qf[1][f >> 1], std::integral_constant<bool, (f < 2)>{}, int_c<0>{});
    });
    pad();
    mask(int_c<0>{}, int_c<0>{}, 0);
    unroll<32>([&](auto I) __attribute__((always_inline)) { max_step(int_c<0>{}, I); });
    unroll<5>([&](auto I) __attribute__((always_inline)) { running_max(I, int_c<0>{}); });
  }
  // every wave has read K(0), whose slot K(3) takes; V(0) and K(1) landed
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);
  asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  k_base(SLOT);
  unroll<DEEP>([&](auto F) __attribute__((always_inline)) { kf[decltype(F)::value] = kfrag(F); });

  int t = 0;
  // iteration t of parity P (the last one's scores and maxima are of no tile and no use: one code path), of the query
  // blocks from FROM on
  auto iteration = [&](auto P, auto FROM) __attribute__((always_inline)) {
    constexpr int p = decltype(P)::value, from = decltype(FROM)::value, blocks = 2 - from;
    float sum[2] = {0.f, 0.f}, e_even = 0.f;
    uint32_t pw[2][16];
    // element e: 16 (or 8) a k-step of 16 keys, 8 a query block of these (pinned: hipcc sinks all of it past the
    // branches below, to where it is used)
    auto element = [&](auto E) __attribute__((always_inline)) {
      constexpr int e = decltype(E)::value, ks = e / (8 * blocks), qb = from ? 1 : (e >> 3) & 1, j = e & 7;
      float x = __builtin_amdgcn_exp2f(fmaf(s[p][ks >> 1][qb][8 * (ks & 1) + j], scale_log2, -mc[qb]));
      sum[qb] += x;
      asm volatile("" : "+v"(x), "+v"(sum[qb]));
      if constexpr (j & 1) {
        pw[qb][4 * ks + (j >> 1)] = pack2bf(e_even, x);
        asm volatile("" : "+v"(pw[qb][4 * ks + (j >> 1)]));
      } else {
        e_even = x;
      }
    };
    const uint32_t k_to = scalar(slot[0] + wid * 1024), v_to = scalar(V0 + slot[2] + wid * 1024);
    u32x4 from_where;
    constexpr int ALL = 32 * blocks, FRONT = 20 * blocks;              // elements, those beside the products with K
    // ---- S(t + 1), elements 0..FRONT - 1
    unroll<32>([&](auto Q) __attribute__((always_inline)) {
      constexpr int q = decltype(Q)::value, f = q >> 1;
      if constexpr ((q & 1) >= from)
        mma_s(s[1 - p][f & 1][q & 1], kf[f % DEEP], qf[q & 1][f >> 1], std::integral_constant<bool, (f < 2)>{}, FROM);
      if constexpr (q % 2 == 1 && f + DEEP < 16) kf[f % DEEP] = kfrag(int_c<(f + DEEP < 16 ? f + DEEP : 0)>{});
      if constexpr (q == 1) {
        if (__ballot((from == 0 && alpha[0] != 1.f) || alpha[1] != 1.f)) {
          pad();
#pragma unroll
          for (int qb = from; qb < 2; ++qb)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              f32x16 v;
              asm volatile("" : "=v"(v) : "0"(o[qb][i]));
#pragma unroll
              for (int r = 0; r < 16; ++r) v[r] *= alpha[qb];
              asm volatile("" : "=a"(o[qb][i]) : "0"(v));
            }
          pad();
        }
      }
      if constexpr (q == 31 - DEEP) v_base(slot[0]);
      if constexpr (q == 2) find(t + 3);
      if constexpr (q >= 5 && q < 30) {                        // a piece, and two steps ahead of it where it is from
        constexpr int n = (q + 1) / 3 - 2;
        using KV = int_c<n / 4>;
        if constexpr (q % 3 == 2 && n < 8) {
          from_where = where(int_c<n % 4>{}, KV{});
          if constexpr (SRC == BLOCKS_OF_16) asm volatile("" : "+s"(from_where));
        }
        if constexpr (q % 3 == 0) piece(int_c<n % 4>{}, KV{}, int_c<1>{}, n < 4 ? k_to : v_to, from_where);
      }
      if constexpr (q >= 32 - DEEP) vf[q - 32 + DEEP] = vfrag(int_c<(q >= 32 - DEEP ? q - 32 + DEEP : 0)>{});
      constexpr int e0 = q * FRONT / 32, e1 = (q + 1) * FRONT / 32;
      unroll<e1 - e0>([&](auto I) __attribute__((always_inline)) { element(int_c<e0 + decltype(I)::value>{}); });
      fence();
    });
    // ---- O += V(t)^T P(t)^T, the other elements, the maxima of S(t + 1)
    const float alpha_t[2] = {alpha[0], alpha[1]};
    unroll<32>([&](auto Q) __attribute__((always_inline)) {
      constexpr int q = decltype(Q)::value, f = q >> 1, ks = f >> 2, qb = q & 1;
      if constexpr (qb >= from) {
        const u32x4 w = {pw[qb][4 * ks], pw[qb][4 * ks + 1], pw[qb][4 * ks + 2], pw[qb][4 * ks + 3]};
        asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0"
                     : "+a"(o[qb][f & 3]) : "v"(vf[f % DEEP]), "v"(w));
      }
      if constexpr (q % 2 == 1 && f + DEEP < 16) vf[f % DEEP] = vfrag(int_c<(f + DEEP < 16 ? f + DEEP : 0)>{});
      if constexpr (q < ALL - FRONT) element(int_c<(q < ALL - FRONT ? FRONT + q : 0)>{});
      constexpr int M = 4 * (1 + from);                        // (four products behind the last of S(t + 1))
      if constexpr (q == M) mask(int_c<1 - p>{}, FROM, t + 1);
      if constexpr (q >= M && q < M + 16) {
        if constexpr (from == 0) max_step(int_c<1 - p>{}, int_c<2 * (q - M)>{});
        max_step(int_c<1 - p>{}, int_c<2 * (q - M) + 1>{});
      }
      if constexpr (q >= M + 16 && q < M + 21) running_max(int_c<q - M - 16>{}, FROM);
      if constexpr (q == 24) {
        turn();
        __builtin_amdgcn_s_waitcnt(0xC07F);        // lgkmcnt(0): V(t) is read
        asm volatile("s_waitcnt vmcnt(8)" ::: "memory");   // K(t + 2) and V(t + 1), requested an iteration ago, landed
        fence();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        k_base(slot[1]);
      }
      if constexpr (q > 24 && q <= 24 + DEEP) kf[q - 25] = kfrag(int_c<(q > 24 && q <= 24 + DEEP ? q - 25 : 0)>{});
      fence();
    });
    static_assert(24 + DEEP < 32 && 2 * (15 - DEEP) + 1 < 24);
#pragma unroll
    for (int qb = from; qb < 2; ++qb) l_run[qb] = l_run[qb] * alpha_t[qb] + sum[qb];
    ++t;
  };
  using TWO = int_c<0>;
  using LAST = int_c<1>;
  // (with an exit between the two hipcc moves O between register files on the way round)
  while (t + 1 < both) {
    iteration(int_c<0>{}, TWO{});
    iteration(int_c<1>{}, TWO{});
  }
  // (what follows reads O, hipcc's copies of it where these paths meet included: the wait states on each of them)
  if (t < both) {
    iteration(int_c<0>{}, TWO{});
    pad();
    if (PAIRED && t < mine) {
      iteration(int_c<1>{}, LAST{});
      pad();
    }
  } else {
    pad();
  }
  if constexpr (PAIRED) {                          // t is even, or all of them
    while (t + 1 < mine) {
      iteration(int_c<0>{}, LAST{});
      iteration(int_c<1>{}, LAST{});
    }
    if (t < mine) {
      iteration(int_c<0>{}, LAST{});
      pad();
    } else {
      pad();
    }
  }
  // the workgroup's other tiles: this wave's share of the staging, and the barriers
  for (; t < ntiles; ++t) {
    find(t + 3);
    stage(K_{}, slot[0]);
    stage(V_{}, V0 + slot[2]);
    turn();
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // no LDS-DMA outlives the workgroup
  if (!active) return;
  // O through the queries' image, 256-byte rows whose 16-byte chunk c lies at c ^ (row & 15): stores of whole rows (8
  // bytes a lane, of 32 rows a store, took 6 k cycles)
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    const auto w = __builtin_amdgcn_permlane32_swap(__float_as_uint(l_run[qb]), __float_as_uint(l_run[qb]), false, false);
    const float l = __uint_as_float(w[0]) + __uint_as_float(w[1]);
    const float inv = l > 0.f ? 1.f / l : 0.f;
    const uint32_t to = mine_at + 8192 * qb + 256 * qc + 8 * hi;
#pragma unroll
    for (int db = 0; db < 4; ++db) {
      f32x16 v;
      asm volatile("" : "=v"(v) : "0"(o[qb][db]));
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *(__attribute__((address_space(3))) u32x2*)(to + 16 * ((4 * db + g) ^ (qc & 15))) =
            u32x2{pack2bf(v[4 * g] * inv, v[4 * g + 1] * inv), pack2bf(v[4 * g + 2] * inv, v[4 * g + 3] * inv)};
    }
  }
  asm volatile("" ::: "memory");
  const int r4 = lane >> 4, c16 = lane & 15;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int qb = i >> 3, row = 4 * (i & 7) + r4, qr = row0[qb] + row;
    const u32x4 x = *(const __attribute__((address_space(3))) u32x4*)(mine_at + 8192 * qb + 256 * row + 16 * (c16 ^ (row & 15)));
    if (qr < len && (qb == 1 || has0))
      *reinterpret_cast<u32x4*>(out + (long)(s0 + qr) * out_stride + (long)h * HD + 8 * c16) = x;
  }
}

template <int SRC, bool PAIRED>
static int launch_src(dim3 grid, void* out, int out_stride, const void* qkv, int row_stride, const int* cu_seqlens,
                      int hq, int hkv, float scale_log2, const int* ctx_lens, const void* k_cache, const void* v_cache,
                      const int* block_tables, int bt_stride, int block_size, int shift, hipStream_t st) {
  constexpr int lds = 10 * SLOT;
  static bool raised = false;
  if (!raised) {
    hipFuncSetAttribute((const void*)prefill_long_kernel<SRC, PAIRED>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    raised = true;
  }
  prefill_long_kernel<SRC, PAIRED><<<grid, 256, lds, st>>>((u16*)out, out_stride, (const u16*)qkv, row_stride, cu_seqlens,
                                                           hq, hkv, scale_log2, ctx_lens, (const u16*)k_cache,
                                                           (const u16*)v_cache, block_tables, bt_stride, block_size, shift);
  DLI_RETURN_LAUNCH();
}

// What both launches take. ctx_lens null: keys and values in the activation's rows. scale_log2: the scores' scale times log2 e
#define DLI_LONG_ARGS void *out, int out_stride, const void *qkv, int row_stride, const int *cu_seqlens, int num_seqs,      \
                      int max_seqlen, int hq, int hkv, float scale_log2, const int *ctx_lens, const void *k_cache,          \
                      const void *v_cache, const int *block_tables, int bt_stride, int block_size, hipStream_t st

template <bool PAIRED>
static int launch_rows(DLI_LONG_ARGS) {
  const int blocks = (max_seqlen + ROWS - 1) / ROWS;
  const dim3 grid = hq <= 4 ? dim3(blocks, num_seqs, hq) : dim3(blocks * hq, num_seqs);
#define DLI_ARGS out, out_stride, qkv, row_stride, cu_seqlens, hq, hkv, scale_log2, ctx_lens, k_cache, v_cache, \
                 block_tables, bt_stride, block_size
  if (ctx_lens == nullptr) return launch_src<ROWS_OF_QKV, PAIRED>(grid, DLI_ARGS, 0, st);
  if (block_size < 16 || (block_size & (block_size - 1))) return (int)hipErrorInvalidValue;
  return launch_src<BLOCKS_OF_16, PAIRED>(grid, DLI_ARGS, __builtin_ctz(block_size), st);
#undef DLI_ARGS
}
