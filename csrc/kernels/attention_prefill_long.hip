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
// K and V tiles come by LDS-DMA into rings of three slots, rows past the keys as zeros (range-checked descriptors).
// In iteration t K(t + 1) and V(t) are read, K(t + 2) and V(t + 1) land, K(t + 3) and V(t + 2) are requested; the
// only barrier, once the last of V(t) is read, ends all three. Causal: a workgroup's tiles stop at its last row's
// bound, a wave's at its own; only tiles that cross a wave's diagonal or the last key are masked.
#include "common.h"

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(1))) void gbl_void;
typedef const __attribute__((address_space(3))) bf16x8 lds_frag;

__device__ __forceinline__ float max3_raw(float a, float b, float c) {  // no canonicalise
  float r;
  asm volatile("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// a value that is the same in all lanes, in a scalar register
__device__ __forceinline__ uint32_t scalar(uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); }

constexpr int HD = 128, KT = 64, ROWS = 256;
constexpr int SLOT = KT * HD * 2;                  // bytes of a K (or V) tile
constexpr float RESCALE_THR = 8.f;                 // log2 units: a running max is raised only by more than this

// Where keys and values are: the activation's rows, or blocks of the paged cache, of a power of two of at least 16
// tokens (others take the kernel of 8 waves).
enum { ROWS_OF_QKV = 0, BLOCKS_OF_16 = 1 };

template <int SRC>
__global__ void __launch_bounds__(256, 1) prefill_long_kernel(
    u16* __restrict__ out, int out_stride, const u16* __restrict__ qkv, int row_stride,
    const int* __restrict__ cu_seqlens, int hq, int hkv, float scale_log2,
    const int* __restrict__ ctx_lens, const u16* __restrict__ k_cache,
    const u16* __restrict__ v_cache, const int* __restrict__ block_tables, int bt_stride,
    int block_size, int block_shift) {
  extern __shared__ __attribute__((aligned(16))) char smem[];        // 3 K slots, 3 V slots, from address 0
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
  const int q0 = blk * ROWS + wid * 64;                              // this wave's first row
  const bool active = q0 < len;
  const int wq_lo = qoff + q0, wq_hi = qoff + min(q0 + 64, len) - 1; // its first and last position
  const int kend = min(nkeys, qoff + min((blk + 1) * ROWS, len));
  const int ntiles = (kend + KT - 1) / KT, mine = active ? wq_hi / KT + 1 : 0;

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
  // Rows: one descriptor a sequence and operand, the tile in the scalar offset. Blocks: a descriptor a piece, whose
  // place and bytes V's piece, staged an iteration after K's, takes over
  const int total = __builtin_amdgcn_readfirstlane((nkeys - 1) * stride + HD * 2);                   // (the launcher keeps a sequence's below 2^31)
  int row_at[2] = {0, 0};                                            // [K's tile, V's tile]
  long at[2][4] = {};
  int bytes[2][4] = {};
  // the tile that K's pieces are of next, V's that which K's were of last
  auto find = [&](int t) __attribute__((always_inline)) {
    if constexpr (SRC == BLOCKS_OF_16) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        at[1][j] = at[0][j];
        bytes[1][j] = bytes[0][j];
        const int first = t * KT + 16 * j;
        const int id = __builtin_amdgcn_readfirstlane(btab[min(first, nkeys - 1) >> block_shift]);
        bytes[0][j] = __builtin_amdgcn_readfirstlane(min(max(nkeys - first, 0), 16) * (HD * 2));
        at[0][j] = (long)id * ((long)hkv * block_size * HD * 2) + (first & (block_size - 1)) * (HD * 2);
      }
    } else {
      row_at[1] = row_at[0];
      row_at[0] = t * (KT * stride);
    }
  };
  // (inline asm: behind the builtin hipcc waits for every LDS-DMA in flight ahead of a transposing read. It has no
  // result, and what it has written is read behind counted waits and a barrier)
  auto piece = [&](auto J, auto KV, uint32_t slot) __attribute__((always_inline)) {
    constexpr int j = decltype(J)::value, kv = decltype(KV)::value;
    const uintptr_t base = SRC == BLOCKS_OF_16 ? heads[kv] + at[kv][j] : heads[kv];
    // (a row past the last is out of range whatever its columns: rows are at least 256 bytes apart)
    const u32x4 r = {scalar((uint32_t)base), scalar((uint32_t)(base >> 32) & 0xffff),
                     scalar((uint32_t)(SRC == BLOCKS_OF_16 ? bytes[kv][j] : total)), 0x00020000};
    const uint32_t dst = scalar(slot + (wid + 4 * j) * 1024);
    const uint32_t so = SRC == BLOCKS_OF_16 ? 0 : scalar((uint32_t)(row_at[kv] + j * 16 * stride));
    const int lane_at = voff;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :: "s"(dst), "v"(lane_at), "s"(r), "s"(so) : "memory", "m0");
  };
  using K_ = int_c<0>;
  using V_ = int_c<1>;
  constexpr uint32_t V0 = 3 * SLOT;
  auto stage = [&](auto KV, uint32_t slot) __attribute__((always_inline)) {
    unroll<4>([&](auto J) __attribute__((always_inline)) { piece(J, KV, slot); });
  };
  // Q^T operand: lane (query qc, half hi) holds Q[q][16 c + 8 hi .. + 7]
  bf16x8 qf[2][8];
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    const u16* qp = qkv + (long)(s0 + min(q0 + 32 * qb + qc, len - 1)) * row_stride + (long)h * HD + 8 * hi;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const uint4 v = *reinterpret_cast<const uint4*>(qp + 16 * c);
      asm volatile("" : "=a"(qf[qb][c]) : "0"(__builtin_bit_cast(bf16x8, v)));
    }
  }
  find(0);
  stage(K_{}, 0);
  find(1);
  stage(V_{}, V0);
  stage(K_{}, SLOT);
  find(2);
  stage(V_{}, V0 + SLOT);
  stage(K_{}, 2 * SLOT);
  asm volatile("s_waitcnt vmcnt(8)" ::: "memory");                   // K(0), V(0) and K(1) landed
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
  auto mma_s = [&](f32x16& d, const bf16x8& a, const bf16x8& b, auto FIRST) __attribute__((always_inline)) {
    if constexpr (decltype(FIRST)::value)
      asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "a"(b));
    else
      asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(d) : "v"(a), "a"(b));
  };
  auto pad = [&]() __attribute__((always_inline)) {
    fence();
    asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");
    fence();
  };
  // scores of keys that a lane's queries do not see
  auto mask = [&](auto P, int t) __attribute__((always_inline)) {
    constexpr int p = decltype(P)::value;
    const int k0 = t * KT;
    if (k0 + KT - 1 > wq_lo || k0 + KT > nkeys) {
      unroll<2>([&](auto QB) __attribute__((always_inline)) {
        constexpr int qb = decltype(QB)::value;
        const int last = min(wq_lo + 32 * qb + qc, nkeys - 1) - k0 - 4 * hi;   // in steps of this lane's keys
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
  auto running_max = [&](auto I) __attribute__((always_inline)) {
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
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
      mma_s(s[0][f & 1][0], a, qf[0][f >> 1], std::integral_constant<bool, (f < 2)>{});
      mma_s(s[0][f & 1][1], a, qf[1][f >> 1], std::integral_constant<bool, (f < 2)>{});
    });
    pad();
    mask(int_c<0>{}, 0);
    unroll<32>([&](auto I) __attribute__((always_inline)) { max_step(int_c<0>{}, I); });
    unroll<5>(running_max);
    k_base(SLOT);
    unroll<DEEP>([&](auto F) __attribute__((always_inline)) { kf[decltype(F)::value] = kfrag(F); });
  }
  // every wave has read K(0), whose slot K(3) takes
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");

  int t = 0;
  // iteration t of parity P (the last one's scores and maxima are of no tile and no use: one code path)
  auto iteration = [&](auto P) __attribute__((always_inline)) {
    constexpr int p = decltype(P)::value;
    float sum[2] = {0.f, 0.f}, e_even = 0.f;
    uint32_t pw[2][16];
    // element e: 16 a k-step of 16 keys, 8 a query block of these (pinned: hipcc sinks all of it past the branches
    // below, to where it is used)
    auto element = [&](auto E) __attribute__((always_inline)) {
      constexpr int e = decltype(E)::value, ks = e >> 4, qb = (e >> 3) & 1, j = e & 7;
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
    constexpr int FRONT = 40;                      // elements beside the products with K
    // ---- S(t + 1), elements 0..39
    unroll<32>([&](auto Q) __attribute__((always_inline)) {
      constexpr int q = decltype(Q)::value, f = q >> 1;
      mma_s(s[1 - p][f & 1][q & 1], kf[f % DEEP], qf[q & 1][f >> 1], std::integral_constant<bool, (f < 2)>{});
      if constexpr (q % 2 == 1 && f + DEEP < 16) kf[f % DEEP] = kfrag(int_c<(f + DEEP < 16 ? f + DEEP : 0)>{});
      if constexpr (q == 1) {
        if (__ballot(alpha[0] != 1.f || alpha[1] != 1.f)) {
          pad();
#pragma unroll
          for (int qb = 0; qb < 2; ++qb)
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
      if constexpr (q >= 6 && q < 30 && q % 3 == 0) {
        constexpr int n = q / 3 - 2;
        if constexpr (n < 4) piece(int_c<n>{}, K_{}, slot[0]);
        else piece(int_c<n - 4>{}, V_{}, V0 + slot[2]);
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
      const u32x4 w = {pw[qb][4 * ks], pw[qb][4 * ks + 1], pw[qb][4 * ks + 2], pw[qb][4 * ks + 3]};
      asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0"
                   : "+a"(o[qb][f & 3]) : "v"(vf[f % DEEP]), "v"(w));
      if constexpr (q % 2 == 1 && f + DEEP < 16) vf[f % DEEP] = vfrag(int_c<(f + DEEP < 16 ? f + DEEP : 0)>{});
      if constexpr (q < 64 - FRONT) element(int_c<(q < 64 - FRONT ? FRONT + q : 0)>{});
      if constexpr (q == 4) mask(int_c<1 - p>{}, t + 1);       // (four products behind the last of S(t + 1))
      if constexpr (q >= 4 && q < 20) {
        max_step(int_c<1 - p>{}, int_c<2 * (q - 4)>{});
        max_step(int_c<1 - p>{}, int_c<2 * (q - 4) + 1>{});
      }
      if constexpr (q >= 20 && q < 25) running_max(int_c<q - 20>{});
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
    for (int qb = 0; qb < 2; ++qb) l_run[qb] = l_run[qb] * alpha_t[qb] + sum[qb];
    ++t;
  };
  // (with an exit between the two hipcc moves O between register files on the way round)
  while (t + 1 < mine) {
    iteration(int_c<0>{});
    iteration(int_c<1>{});
  }
  // (what follows reads O, hipcc's copies of it where these paths meet included: the wait states on each of them)
  if (t < mine) {
    iteration(int_c<0>{});
    pad();
  } else {
    pad();
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
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    const auto w = __builtin_amdgcn_permlane32_swap(__float_as_uint(l_run[qb]), __float_as_uint(l_run[qb]), false, false);
    const float l = __uint_as_float(w[0]) + __uint_as_float(w[1]);
    const float inv = l > 0.f ? 1.f / l : 0.f;
    const int qr = q0 + 32 * qb + qc;
    u16* op = out + (long)(s0 + qr) * out_stride + (long)h * HD;
#pragma unroll
    for (int db = 0; db < 4; ++db) {
      f32x16 v;
      asm volatile("" : "=v"(v) : "0"(o[qb][db]));
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const uint2 x = {pack2bf(v[4 * g] * inv, v[4 * g + 1] * inv), pack2bf(v[4 * g + 2] * inv, v[4 * g + 3] * inv)};
        if (qr < len) *reinterpret_cast<uint2*>(op + 32 * db + 8 * g + 4 * hi) = x;
      }
    }
  }
}

template <int SRC>
static int launch_src(dim3 grid, void* out, int out_stride, const void* qkv, int row_stride, const int* cu_seqlens,
                      int hq, int hkv, float scale_log2, const int* ctx_lens, const void* k_cache, const void* v_cache,
                      const int* block_tables, int bt_stride, int block_size, int shift, hipStream_t st) {
  constexpr int lds = 6 * SLOT;
  static bool raised = false;
  if (!raised) {
    hipFuncSetAttribute((const void*)prefill_long_kernel<SRC>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    raised = true;
  }
  prefill_long_kernel<SRC><<<grid, 256, lds, st>>>((u16*)out, out_stride, (const u16*)qkv, row_stride, cu_seqlens, hq,
                                                   hkv, scale_log2, ctx_lens, (const u16*)k_cache, (const u16*)v_cache,
                                                   block_tables, bt_stride, block_size, shift);
  DLI_RETURN_LAUNCH();
}

// ctx_lens null: keys and values in the activation's rows. scale_log2: the scores' scale times log2 e
int launch_prefill_long(void* out, int out_stride, const void* qkv, int row_stride, const int* cu_seqlens, int num_seqs,
                        int max_seqlen, int hq, int hkv, float scale_log2, const int* ctx_lens, const void* k_cache,
                        const void* v_cache, const int* block_tables, int bt_stride, int block_size, hipStream_t st) {
  const int blocks = (max_seqlen + ROWS - 1) / ROWS;
  const dim3 grid = hq <= 4 ? dim3(blocks, num_seqs, hq) : dim3(blocks * hq, num_seqs);
#define DLI_ARGS out, out_stride, qkv, row_stride, cu_seqlens, hq, hkv, scale_log2, ctx_lens, k_cache, v_cache, \
                 block_tables, bt_stride, block_size
  if (ctx_lens == nullptr) return launch_src<ROWS_OF_QKV>(grid, DLI_ARGS, 0, st);
  if (block_size < 16 || (block_size & (block_size - 1))) return (int)hipErrorInvalidValue;
  return launch_src<BLOCKS_OF_16>(grid, DLI_ARGS, __builtin_ctz(block_size), st);
#undef DLI_ARGS
}
