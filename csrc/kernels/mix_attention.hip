// Windowed attention whose heads' softmax weights are mixed before the value sum (talk [H, H]):
//   W'_h = sum_g talk[h, g] softmax_g,   out_h = W'_h . v_{group of h}
// the portions' form for 32 heads of 128 channels over at most 8 key / value heads; other sizes and
// short steps run window_attention_mfma.hip, whose arguments and roundings (normalised weights, the
// mixing matrix and the mixed weights in bf16, everything else fp32) this shares.
//
// Two launches: the softmax's (max, 1 / sum) per head and query, then the outputs. A workgroup is 8
// waves over 16 queries, a wave 4 heads of one key head, in tiles of 32 keys. Per tile
//   S^T = K . Q^T   K rows from the cache to registers, requested as soon as the last tile's are
//                   used and shared by the wave's 4 heads; the queries stay in registers
//   w = exp2(s - m) / l -> LDS [(key, query)][head]
//   W' = talk . w   each wave mixes 4 keys of all heads and queries -> LDS [head][query][key]
//   O^T += V^T . W' the wave's own value head, LDS-DMA a tile ahead, read transposed
// with two barriers. The outputs of 4 heads by 128 channels, the queries and a key tile are more
// registers than a wave has: a workgroup takes 64 of the channels, and the pair of workgroups repeats
// the scores. A tile takes some 7000 cycles: scores 1600, key loads 800 (a wave's are 8 KB through an
// L1 of 64 B a cycle), softmax 1300, mixing 800, values 600 and 1900 at the barriers, where the two
// waves of a SIMD, in the same phase, wait for each other; the registers allow no third.
// 4 x 2048 tokens, window 1024: the general form, which stages all heads' keys behind barriers, loads
// the queries for every tile and transposes the values by 2-byte stores, 2264 us; this 147 + 496.
// 8000 tokens, window 4096: 8141 -> 2052 us; 64 single ones at 1000 keys 306 -> 167. Since then a tile's values are
// requested a whole tile ahead (they were just ahead of the wait for the next keys, which hipcc makes a wait for both):
// both launches 562 -> 540, 8000 tokens, window 4000, 1787 -> 1704, the single ones 152 -> 135, to the bit.
#include "lds_dma.h"

typedef short mix_s16x4 __attribute__((ext_vector_type(4)));
typedef short mix_s16x8 __attribute__((ext_vector_type(8)));

namespace {

constexpr int TQ = 16, TK = 32, NW = 8, HW = 4, H = NW * HW, HD = 128, DVW = 64;
constexpr int PROW = H + 8;        // padded row of the weights [(key, query)][head]
constexpr int WROW = TK + 8;       // padded row of the mixed weights [(head, query)][key]
constexpr int SLOTS_MAX = 4096;    // keys a query tile may see: their cache rows are kept in LDS
constexpr float LOG2E = 1.4426950408889634f;
// Fewest query tiles; the general form splits a step of fewer over the keys. This / the general form, us,
// at ~1000 visible keys: 8 tiles 159 / 151, 16 160 / 157, 20 158 / 238, 32 163 / 304; of single rows 20 at
// 500, 1000, 2000, 4000 keys 103 / 99, 193 / 203, 290 / 319, 590 / 602, 32 at 4000 612 / 605, 64 630 / 1093.
constexpr int MIX_MIN_TILES = 20;

struct MixArgs {
  const u16* q; int ldq;
  const u16* k; long k_stride;
  const u16* v; long v_stride;
  u16* out; int ldo;
  const float* gate; int ldg;
  const float* slopes;
  const float* talk;
  const int* cu; const int* positions;
  const int* block_tables; int bt_stride; int block_size;
  int G, window, qtiles;
  float scale, out_scale;
  int head_gate;
  float* stats;                    // [T][H][2]
};

// 16-byte chunk of row r's values at c ^ swz(r): the transposed reads take 32 bytes of 4 rows
__device__ __forceinline__ int swz(int r) { return ((r >> 1) & 3) << 1; }

// NV: value tiles of a wave in LDS
template <bool STATS, int NV>
__global__ void __launch_bounds__(STATS ? 256 : 512) mix_attention_kernel(MixArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  u16* Vt = (u16*)smem;                            // [NW][NV][TK][DVW]
  u16* Pm = Vt + (STATS ? 0 : NW * NV * TK * DVW); // [TK * TQ][PROW]
  u16* Wm = Pm + (STATS ? 0 : TK * TQ * PROW);     // [H * TQ][WROW]
  int* slot = (int*)(Wm + (STATS ? 0 : H * TQ * WROW));
  const int tid = threadIdx.x, lane = tid & 63;
  const int fr = lane & 15, fq = lane >> 4;
  // consecutive tiles (and both halves of the channels) on one XCD: their windows overlap
  const int nb = gridDim.x, per = (nb + 7) / 8;
  int id = blockIdx.x;
  if (nb % 8 == 0) id = (id % 8) * per + id / 8;
  const int dvo = (id & 1) * DVW;                  // the pair: channels, or (statistics) heads
  const int wave = (tid >> 6) + (STATS ? (id & 1) * (NW / 2) : 0);
  id >>= 1;
  const int s = id / a.qtiles;
  const int t0 = a.cu[s] + (id % a.qtiles) * TQ, t_end = a.cu[s + 1];
  if (t0 >= t_end) return;
  const int nq = min(TQ, t_end - t0);
  const int p0 = a.positions[t0], p_last = p0 + nq - 1;      // positions of a portion are consecutive
  const int lo = max(0, p0 - a.window + 1);
  const int n = p_last - lo + 1, ntiles = (n + TK - 1) / TK;
  const bool my_q = fr < nq;
  const int my_p = p0 + fr;
  const int h0 = wave * HW, grp = h0 / (H / a.G);
  {
    const int* bt = a.block_tables + (long)s * a.bt_stride;
    for (int i = tid; i < ntiles * TK; i += blockDim.x) {
      const int j = min(lo + i, p_last);           // keys past the end are masked: any row will do
      slot[i] = bt[j / a.block_size] * a.block_size + j % a.block_size;
    }
  }
  bf16x8 qf[HW][HD / 32];
  float slope2[HW], m[HW], l[HW];
#pragma unroll
  for (int h = 0; h < HW; ++h) {
    const u16* qr = a.q + (long)(t0 + (my_q ? fr : 0)) * a.ldq + (h0 + h) * HD + fq * 8;
#pragma unroll
    for (int kk = 0; kk < HD / 32; ++kk) qf[h][kk] = *reinterpret_cast<const bf16x8*>(qr + kk * 32);
    slope2[h] = a.slopes ? a.slopes[h0 + h] * LOG2E : 0.f;
    m[h] = STATS ? -INFINITY : 0.f;
    l[h] = 0.f;                                    // output launch: 1 / sum
    if (!STATS && my_q) {
      const float* st = a.stats + ((long)(t0 + fr) * H + h0 + h) * 2;
      m[h] = st[0];
      l[h] = st[1];
    }
  }
  const float scale2 = a.scale * LOG2E;
  bf16x8 tk[2];
  f32x4 o[HW][DVW / 16];
  if constexpr (!STATS) {
#pragma unroll
    for (int hb = 0; hb < 2; ++hb)
#pragma unroll
      for (int j = 0; j < 8; ++j)
        tk[hb][j] = (__bf16)a.talk[(hb * 16 + fr) * H + fq * 8 + j];
#pragma unroll
    for (int h = 0; h < HW; ++h)
#pragma unroll
      for (int b = 0; b < DVW / 16; ++b) o[h][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  __syncthreads();                                 // slot table
  bf16x8 kf[2][HD / 32];
  const auto load_k = [&](int tile, int kb) {
    const u16* kr = a.k + (long)slot[tile * TK + kb * 16 + fr] * a.k_stride + grp * HD + fq * 8;
#pragma unroll
    for (int kk = 0; kk < HD / 32; ++kk) kf[kb][kk] = *reinterpret_cast<const bf16x8*>(kr + kk * 32);
  };
  const u16* const vts = Vt + wave * NV * TK * DVW;
  const auto load_v = [&](int tile) {              // 8 rows of 128 bytes an instruction
    const uint32_t to = lds_address(vts + tile % NV * TK * DVW);
#pragma unroll
    for (int p = 0; p < TK / 8; ++p) {
      const int r = p * 8 + (lane >> 3), c = (lane & 7) ^ swz(r);
      dma_lanes(to + p * 8 * DVW * 2, a.v + (long)slot[tile * TK + r] * a.v_stride + grp * HD + dvo + c * 8);
    }
  };
  // With two value tiles a tile's values are requested a whole tile ahead, ahead of its keys; with one, behind the next
  // keys. hipcc waits for the keys, and does not count the values: the loop waits for both itself, where it needs the
  // keys and nothing else is in flight
  if constexpr (!STATS) load_v(0);
  load_k(0, 0);
  load_k(0, 1);

  for (int tile = 0; tile < ntiles; ++tile) {
    const int j0 = lo + tile * TK;
    // (rows past the last query keep m = l = 0 or are not stored: whatever they hold stays theirs)
    const bool interior = j0 + TK - 1 <= p0 && j0 > p_last - a.window;
    if constexpr (!STATS) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // keys and values of this tile landed
    if constexpr (!STATS && NV == 2) {             // (behind hipcc's wait for the keys, which would be for these too)
#pragma unroll
      for (int kk = 0; kk < HD / 32; ++kk) asm volatile("" : "+v"(kf[0][kk]), "+v"(kf[1][kk]));
      if (tile + 1 < ntiles) load_v(tile + 1);
    }
    f32x4 sc[2][HW];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
      for (int h = 0; h < HW; ++h) sc[kb][h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < HD / 32; ++kk)
#pragma unroll
        for (int h = 0; h < HW; ++h)
          sc[kb][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[kb][kk], qf[h][kk], sc[kb][h], 0, 0, 0);
      if (tile + 1 < ntiles) load_k(tile + 1, kb);
    }
    // lane: query fr, keys j0 + 16 kb + 4 fq + r; scores in the log2 domain
    //   x = s * scale2 + slope2 * (key - position)      (output launch: less the row's m)
    const float dist = (float)(j0 + fq * 4 - my_p);
#pragma unroll
    for (int h = 0; h < HW; ++h) {
      const float base = fmaf(slope2[h], dist, STATS ? 0.f : -m[h]);
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          sc[kb][h][r] = fmaf(sc[kb][h][r], scale2, fmaf(slope2[h], (float)(kb * 16 + r), base));
    }
    if (!interior) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int d = my_p - (j0 + kb * 16 + fq * 4 + r);
          const bool out = !my_q || d < 0 || d >= a.window;
#pragma unroll
          for (int h = 0; h < HW; ++h) sc[kb][h][r] = out ? -INFINITY : sc[kb][h][r];
        }
    }
    if constexpr (STATS) {
      // every lane its own running pair over its 8 keys of a tile; combined at the end
#pragma unroll
      for (int h = 0; h < HW; ++h) {
        float top = m[h];
#pragma unroll
        for (int i = 0; i < 8; ++i) top = fmaxf(top, sc[i >> 2][h][i & 3]);
        const float mm = top == -INFINITY ? 0.f : top;
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) sum += __builtin_amdgcn_exp2f(sc[i >> 2][h][i & 3] - mm);
        l[h] = l[h] * __builtin_amdgcn_exp2f(m[h] - mm) + sum;
        m[h] = top;
      }
    } else {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float w[HW];
#pragma unroll
          for (int h = 0; h < HW; ++h) w[h] = __builtin_amdgcn_exp2f(sc[kb][h][r]) * l[h];
          uint2 pk;
          pk.x = pack2bf(w[0], w[1]);
          pk.y = pack2bf(w[2], w[3]);
          *reinterpret_cast<uint2*>(Pm + ((kb * 16 + fq * 4 + r) * TQ + fr) * PROW + h0) = pk;
        }
      __syncthreads();                             // all heads' weights; the last mixed ones are read
      {
        // this wave's keys 4 wave .. + 3 (rows of 16 queries): lane gets heads 16 hb + 4 fq + r of
        // query fr. Kept where the transposed value read has those keys: 8 (w & 3) + 4 (w >> 2)
        f32x4 mix[2][4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const bf16x8 pf = *reinterpret_cast<const bf16x8*>(
              Pm + ((wave * 4 + i) * TQ + fr) * PROW + fq * 8);
#pragma unroll
          for (int hb = 0; hb < 2; ++hb)
            mix[hb][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(tk[hb], pf, f32x4{0.f, 0.f, 0.f, 0.f},
                                                                 0, 0, 0);
        }
#pragma unroll
        for (int hb = 0; hb < 2; ++hb)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            uint2 pk;
            pk.x = pack2bf(mix[hb][0][r], mix[hb][1][r]);
            pk.y = pack2bf(mix[hb][2][r], mix[hb][3][r]);
            *reinterpret_cast<uint2*>(Wm + ((hb * 16 + fq * 4 + r) * TQ + fr) * WROW +
                                      (wave & 3) * 8 + (wave >> 2) * 4) = pk;
          }
      }
      __syncthreads();                             // mixed weights; the weights are read
      const u16* vt = vts + tile % NV * TK * DVW;
      bf16x8 wf[HW];
#pragma unroll
      for (int h = 0; h < HW; ++h)
        wf[h] = *reinterpret_cast<const bf16x8*>(Wm + ((h0 + h) * TQ + fr) * WROW + fq * 8);
      const int qrow = (lane >> 2) & 3, pcol = lane & 3;
#pragma unroll
      for (int b = 0; b < DVW / 16; ++b) {
        const int r0 = 4 * fq + qrow, r1 = 16 + r0, c = 2 * b + (pcol >> 1);
        const mix_s16x4 x0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) mix_s16x4*)(vt + r0 * DVW + (c ^ swz(r0)) * 8 +
                                                           4 * (pcol & 1)));
        const mix_s16x4 x1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) mix_s16x4*)(vt + r1 * DVW + (c ^ swz(r1)) * 8 +
                                                           4 * (pcol & 1)));
        const mix_s16x8 x = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
        const bf16x8 vf = *reinterpret_cast<const bf16x8*>(&x);
#pragma unroll
        for (int h = 0; h < HW; ++h)
          o[h][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, wf[h], o[h][b], 0, 0, 0);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // reads done before the tile is replaced
      if (NV == 1 && tile + 1 < ntiles) load_v(tile + 1);
    }
  }

  if constexpr (STATS) {
#pragma unroll
    for (int h = 0; h < HW; ++h) {
      float top = fmaxf(m[h], __shfl_xor(m[h], 16, 64));
      top = fmaxf(top, __shfl_xor(top, 32, 64));
      const float mm = top == -INFINITY ? 0.f : top;
      float sum = l[h] * __builtin_amdgcn_exp2f(m[h] - mm);
      sum += __shfl_xor(sum, 16, 64);
      sum += __shfl_xor(sum, 32, 64);
      if (fq == 0 && my_q) {
        float* st = a.stats + ((long)(t0 + fr) * H + h0 + h) * 2;
        st[0] = mm;
        st[1] = sum > 0.f ? 1.f / sum : 0.f;
      }
    }
  } else if (my_q) {
    const float* gr = a.gate ? a.gate + (long)(t0 + fr) * a.ldg : nullptr;
#pragma unroll
    for (int h = 0; h < HW; ++h) {
      const int col0 = (h0 + h) * HD + dvo + fq * 4;
      float g[DVW / 16][4];
      if (gr != nullptr) {
#pragma unroll
        for (int b = 0; b < DVW / 16; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r) g[b][r] = gr[a.head_gate ? h0 + h : col0 + b * 16 + r];
#pragma unroll
        for (int b = 0; b < DVW / 16; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r) o[h][b][r] *= 1.f / (1.f + expf(-g[b][r]));
      }
#pragma unroll
      for (int b = 0; b < DVW / 16; ++b) {
        uint2 pk;
        pk.x = pack2bf(o[h][b][0] * a.out_scale, o[h][b][1] * a.out_scale);
        pk.y = pack2bf(o[h][b][2] * a.out_scale, o[h][b][3] * a.out_scale);
        *reinterpret_cast<uint2*>(a.out + (long)(t0 + fr) * a.ldo + col0 + b * 16) = pk;
      }
    }
  }
}

}  // namespace

extern "C" long dli_mix_attention_workspace_bytes(int T) { return (long)T * H * 2 * 4; }

// Returns hipErrorNotSupported (801) for sizes it does not take; nothing was launched then.
extern "C" int dli_mix_attention(const void* q, int ldq, const void* k, long k_stride, const void* v,
                                 long v_stride, void* out, int ldo, const float* gate, int ldg,
                                 const float* slopes, const float* talk, const int* cu,
                                 const int* positions, const int* block_tables, int bt_stride,
                                 int block_size, int num_seqs, int max_seqlen, int heads, int G,
                                 int dq, int dv, int window, float scale, void* ws, int head_gate,
                                 float out_scale, hipStream_t st) {
  if (num_seqs <= 0 || max_seqlen <= 0) return 0;
  const int qtiles = (max_seqlen + TQ - 1) / TQ;
  // the general form splits a step of few query tiles over the keys
  if (talk == nullptr || heads != H || G < 1 || H % G || (H / G) % HW || dq != HD || dv != HD ||
      window < 1 || block_size < 1 || (long)qtiles * num_seqs < MIX_MIN_TILES ||
      (long)qtiles * num_seqs > (1 << 28))
    return (int)hipErrorNotSupported;
  const int slots = ((window < SLOTS_MAX ? window : SLOTS_MAX) + TQ - 1 + TK - 1) / TK * TK;
  if (window > SLOTS_MAX || ws == nullptr || (uintptr_t)q % 16 || (uintptr_t)k % 16 ||
      (uintptr_t)v % 16 || (uintptr_t)out % 8 || (uintptr_t)ws % 4 || ldq % 8 || k_stride % 8 ||
      v_stride % 8 || ldo % 4)
    return (int)hipErrorNotSupported;
  MixArgs a{(const u16*)q, ldq, (const u16*)k, k_stride, (const u16*)v, v_stride, (u16*)out, ldo, gate,
            ldg, slopes, talk, cu, positions, block_tables, bt_stride, block_size, G, window, qtiles,
            scale, out_scale, head_gate, (float*)ws};
  const size_t tables = (size_t)slots * 4;
  const size_t vts = (size_t)NW * TK * DVW * 2, sh = vts + (TK * TQ * PROW + H * TQ * WROW) * 2 + tables;
  // (two value tiles a wave to windows of 4081)
  const bool two = sh + vts <= 160 * 1024;
  static const hipError_t raised = [] {
    const hipError_t e = hipFuncSetAttribute((const void*)mix_attention_kernel<false, 1>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    return e != hipSuccess ? e : hipFuncSetAttribute((const void*)mix_attention_kernel<false, 2>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  }();
  if (raised != hipSuccess) return (int)raised;
  mix_attention_kernel<true, 1><<<2 * qtiles * num_seqs, 256, tables, st>>>(a);
  if (two) mix_attention_kernel<false, 2><<<2 * qtiles * num_seqs, 512, sh + vts, st>>>(a);
  else mix_attention_kernel<false, 1><<<2 * qtiles * num_seqs, 512, sh, st>>>(a);
  DLI_RETURN_LAUNCH();
}
