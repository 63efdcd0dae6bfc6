// Grouped-query sliding-window attention with kept first tokens over token-major paged caches
// (ops.hybrid.window_attention: bf16, the key / value widths in SWA_WIDTHS, an optional gate on the
// output, elementwise or one number a head, an optional sink logit a head, an output scale; no bias or
// mixing — those run window_attention_mfma.hip). The sink and the head's gate only touch the epilogue
// and cost nothing: 5 prompts of 900 to 2601 tokens, 32 heads of 128 on 8 kv heads, took 2.12 ms in
// window_attention_mfma.hip (16 queries x 8 heads a workgroup, barrier-separated phases) and take
// 0.2 ms here; decode of 64 rows at 984 keys 59 us instead of 252.
// Position i sees j <= i with i - j < window or j < keep.
//
// The keys that a group of queries can see are at most two runs, [0, kf) and [lo, last], walked
// as one list: list index x is key x for x < kf and key x + skip from there on. Everything below
// tiles that list, so kept tokens cost what they are and nothing between them and the window is
// read.
//
//  * swa_prefill32  8 waves x 32 query rows of one head: v_mfma_f32_32x32x16_bf16 on swapped
//                   products (S^T = K . Q^T, O^T = V^T . P^T), so that a lane owns one query and
//                   the softmax is lane-local but for one exchange; K / V tiles of 64 keys by
//                   LDS-DMA into three buffers, one barrier a tile; the list's cache rows (of
//                   every sixteenth, where 16 lie together) looked up once (LDS). The structure of attention_prefill.hip's long-prompt kernel.
//                   Latent attention runs it too, expanded: [k_h | shared rotated key] rows of 192.
//  * swa_prefill16  4 waves x 16 query rows: portions shorter than the above is worth
//  * swa_decode     one query token a sequence: a workgroup per (sequence, kv head, key split).
//                   Scores on the matrix cores with K rows straight from the cache (the heads
//                   of the group are the columns); the value sum in fp32 FMAs, a lane owning 8
//                   dims of every head of the group: at one row per head it is far below the
//                   time the bytes take, and V needs no transpose.
#include "lds_dma.h"

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef const __attribute__((address_space(1))) void gbl_void;

namespace {

constexpr float LOG2E = 1.4426950408889634f;

struct SwaArgs {
  const u16* q; int ldq;
  const u16* k; long k_stride;         // cache rows
  const u16* v; long v_stride;
  u16* out; int ldo;
  const float* gate; int ldg;          // null, or [T, H*dv]: the output times its sigmoid
  bool head_gate;                      // the gate is [T, H]: one number a head
  const float* sink;                   // null, or [H]: exp(sink) joins a head's softmax denominator
  float out_scale;
  const int* cu; const int* positions;
  const int* block_tables; int bt_stride; int block_size;
  int H, G, window, keep;
  float scale_log2;
  int block_shift;                     // log2 of a block's rows, where they are a power of two
  int nsplit;                          // decode: key splits
  float* ws;                           // decode, nsplit > 1: [nsplit][S][H][2], [nsplit][S][H][HD]
  // shared tail of queries and keys (prefill32 with DR > 0): head h of token t has its DR dims at q2 +
  // t * ldq2 + h * q2_head, a key row has them once for all heads; the key and value rows of sequence
  // s are then rows [cu_ctx[s], cu_ctx[s + 1]) of plain matrices, its last positions in order
  const u16* q2; long ldq2; int q2_head;
  const u16* k2; long k2_stride;
  const int* cu_ctx;
};

// floats of the decode splits' (max, sum) pairs, in front of their partial sums
__host__ __device__ inline long stat_floats(int nsplit, int S, int H) {
  return ((long)nsplit * S * H * 2 + 3) & ~3L;
}

// factor of un-normalised sums with maximum M (log2 units) and weight sum L, the sink included
__device__ __forceinline__ float norm_factor(const float* sink, int h, float M, float L) {
  if (sink == nullptr) return L > 0.f ? 1.f / L : 0.f;
  const float s = sink[h] * LOG2E, top = fmaxf(M, s), e = __builtin_amdgcn_exp2f(M - top);
  return e / (L * e + __builtin_amdgcn_exp2f(s - top));
}
// a head's share of the epilogue: its gate and the scale
__device__ __forceinline__ float head_factor(const SwaArgs& a, long t, int h) {
  return a.head_gate ? a.out_scale / (1.f + expf(-a.gate[t * a.ldg + h])) : a.out_scale;
}
__device__ __forceinline__ float sigmoid32(float g) { return 1.f / (1.f + __expf(-g)); }

// the key list of queries at positions [first, last]
struct KeyList {
  int kf, skip, n;
  __device__ KeyList(int first, int last, int window, int keep) {
    const int lo = max(0, first - window + 1);
    kf = min(keep, lo);
    skip = lo - kf;
    n = last - skip + 1;
  }
  __device__ int key(int x) const { return x < kf ? x : x + skip; }
  // The same with both runs widened to whole groups of 16 keys, whose rows lie in one cache block each; the keys
  // that no query sees are masked as those of other queries are
  __device__ void widen(int last) {
    const int lo = kf + skip & ~15;
    kf = kf + 15 & ~15;
    skip = kf < lo ? lo - kf : 0;
    if (skip == 0) kf = 0;
    n = last - skip + 1;
  }
};

__device__ __forceinline__ float max3(float a, float b, float c) {
  return fmaxf(fmaxf(a, b), c);
}

constexpr int KT = 64;                 // keys a tile
constexpr int LROWS = 256;             // query rows of a long-form workgroup
constexpr float RESCALE_THR = 8.f;     // log2 units: the running max moves only by more than this

// One tile of rows (D wide) by LDS-DMA: 1-KiB pieces of two subtiles in a row, wave w of 8 takes
// pieces w, w + 8, ... The DMA writes lane-linearly, so each lane loads the logical chunk that
// lands at its place. Columns from D1 on come from a second matrix (its rows alike).
template <int D, int D1, typename RowOf>
__device__ __forceinline__ void stage_rows(const u16* src, long stride, const u16* src2, long stride2,
                                           char* dst, int x0, int wid, int lane, const RowOf& row_of) {
  constexpr int NP = D / 8;
#pragma unroll
  for (int j = 0; j < (NP + 7) / 8; ++j) {
    const int piece = wid + 8 * j;
    if (NP % 8 != 0 && piece >= NP) break;                     // wave-uniform
    const int b = piece * 1024 + lane * 16;
    const int rg = b / (D * 16), in = b % (D * 16);
    const int r = 8 * rg + ((lane & 31) >> 2);
    const int c = 4 * (in / 512) + ((lane & 3) ^ ((r >> 2) & 3));
    const long row = row_of(x0 + r);
    const u16* p = D1 < D && c * 8 >= D1 ? src2 + row * stride2 + (c * 8 - D1) : src + row * stride + c * 8;
    __builtin_amdgcn_global_load_lds((gbl_void*)p, (lds_void*)(dst + piece * 1024), 16, 0, 0);
  }
}

// The same tile from rows that lie together, by sixteens (TOGETHER = 16) or all 64 of it: a lane's offset (voff, of each
// piece) is its place among those rows, and rows past the last land as zeros. rows: the descriptor of sixteen g's (tail:
// of the second matrix's)
template <int D, int D1, typename Rows>
__device__ __forceinline__ void stage_together(uint32_t dst, int wid, const int (&voff)[(D / 8 + 7) / 8], const Rows& rows) {
  constexpr int NP = D / 8;
#pragma unroll
  for (int j = 0; j < (NP + 7) / 8; ++j) {
    const int piece = wid + 8 * j;
    if (NP % 8 != 0 && piece >= NP) break;                     // wave-uniform
    const bool tail = D1 < D && piece * 1024 % (D * 16) / 16 >= D1;
    dma_piece(dst + piece * 1024, voff[j], rows(piece * 64 / D >> 1, tail));
  }
}
template <int D, int D1, int TOGETHER>
__device__ __forceinline__ void piece_offsets(int (&voff)[(D / 8 + 7) / 8], long stride, long stride2, int wid, int lane) {
#pragma unroll
  for (int j = 0; j < (D / 8 + 7) / 8; ++j) {
    const int b = (wid + 8 * j) * 1024 + lane * 16, in = b % (D * 16);
    const int r = 8 * (b / (D * 16)) + ((lane & 31) >> 2), c = 4 * (in / 512) + ((lane & 3) ^ ((r >> 2) & 3));
    const bool tail = D1 < D && c * 8 >= D1;
    voff[j] = r % TOGETHER * (int)(tail ? stride2 : stride) * 2 + (tail ? c * 8 - D1 : c * 8) * 2;
  }
}

// Tile image: 8-row x 32-column subtiles of 512 B with the chunks of a row rotated by its row
// group: conflict-free for row reads and for transposed reads. DK, DR, DV: multiples of 32.
// How a tile's rows are found: SIXTEENS, cache blocks are powers of two of at least 16 rows (or the rows a plain matrix's), staged by
// stage_together; ROWS, a table in LDS of the list's cache rows; BLOCKS, by the block table (or a plain matrix's first row).
// Each a kernel of its own: with the choice between the latter two and both masks in one, it spilled registers at 128 + 256
// wide. In BLOCKS, whose waves wait for the block table, the mask is key by key alone. 16 heads on 4, 8-row blocks, us, one
// kernel / these: 128 + 256 4000 tokens 294 / 193, 513 of 6513 422 / 294, 96 + 192 the latter 325 / 271; in ROWS 2 to 7 % less
enum { BLOCKS = 0, ROWS = 1, SIXTEENS = 2 };
template <int DK, int DR, int DV, int FOUND>
__global__ void __launch_bounds__(512) swa_prefill32_kernel(SwaArgs a) {
  constexpr bool GROUPS = FOUND == SIXTEENS;
  constexpr int KW = DK + DR, KC = KW / 16, DBK = DV / 32;
  constexpr int RGK = KW * 16, RGV = DV * 16;                  // bytes of an 8-row group
  constexpr int TILE_K = KT * KW * 2, TILE_B = KT * (KW + DV) * 2, NBUF = 3;
  constexpr int NPK = KW / 8, NPV = DV / 8;                    // 1-KiB pieces of a tile
  extern __shared__ __attribute__((aligned(16))) char lds[];   // [NBUF][K tile | V tile], slot table
  int* table = (int*)(lds + NBUF * TILE_B);
  // key heads fastest, then the query heads of a group, then row blocks, longest lists first
  // (attention_prefill.hip's order): 5 prompts of 900 to 2601 tokens, 32 heads of 128 on 8 kv heads,
  // 339 -> 250 us; expanded latent heads, 6 prompts of 301 to 3000, 416 -> 278
  const bool by_head = gridDim.z > 1;                          // (up to 4 heads, as there)
  const int s = blockIdx.y, rep = a.H / a.G;
  const int h = by_head ? blockIdx.z : blockIdx.x % a.G * rep + blockIdx.x / a.G % rep, kvh = h / rep;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qc = lane & 31, hi = lane >> 5;
  const int t0 = a.cu[s], len = a.cu[s + 1] - t0;
  const int blk = (int)((gridDim.x - 1 - blockIdx.x) / (by_head ? 1 : a.H));
  const int wg_q0 = blk * LROWS;
  if (wg_q0 >= len) return;                                    // workgroup-uniform
  const int p0 = a.positions[t0];
  const int q0 = wg_q0 + wid * 32;
  const bool active = q0 < len;
  const int last = p0 + min(wg_q0 + LROWS, len) - 1;
  KeyList kl(p0 + wg_q0, last, a.window, a.keep);
  if (GROUPS && !DR) kl.widen(last);           // (a plain matrix has no row ahead of the first key)
  const int ntiles = (kl.n + KT - 1) / KT;
  const int* bt = DR ? nullptr : a.block_tables + (long)s * a.bt_stride;
  const int base = DR ? a.cu_ctx[s + 1] - (p0 + len) : 0;
  const auto row_of = [&](int x) {
    const int j = kl.key(x);
    return DR ? base + j : bt[j / a.block_size] * a.block_size + j % a.block_size;
  };
  // the list's cache rows (GROUPS: of every sixteenth)
  if (FOUND == ROWS)
    for (int x = tid; x < kl.n; x += 512) table[x] = row_of(x);
  if (GROUPS && !DR)
    for (int x = tid; x < 4 * ntiles; x += 512) {
      const int j = kl.key(min(16 * x, kl.n - 1 & ~15));
      table[x] = (bt[j >> a.block_shift] << a.block_shift) + (j & (a.block_size - 1));
    }

  bf16x8 qf[KC];
  {
    const long qt = t0 + min(q0 + qc, len - 1);
    const u16* qp = a.q + qt * a.ldq + (long)h * DK + 8 * hi;
    const u16* qp2 = DR ? a.q2 + qt * a.ldq2 + (long)h * a.q2_head + 8 * hi : nullptr;
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      const uint4 v = *reinterpret_cast<const uint4*>(16 * c < DK ? qp + 16 * c : qp2 + (16 * c - DK));
      qf[c] = *reinterpret_cast<const bf16x8*>(&v);
    }
  }
  const int qpos = p0 + q0 + qc;
  const int wq_lo = p0 + q0, wq_hi = p0 + min(q0 + 32, len) - 1;
  f32x16 o[DBK];
#pragma unroll
  for (int i = 0; i < DBK; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[i][r] = 0.f;
  float m_run = -INFINITY, l_part = 0.f;
  __syncthreads();

  const auto row_in_list = [&](int x) -> long {
    x = min(x, kl.n - 1);
    return FOUND == ROWS ? table[x] : row_of(x);
  };
  int vk[(KW / 8 + 7) / 8], vv[(DV / 8 + 7) / 8];
  if constexpr (GROUPS) {
    piece_offsets<KW, DK, DR ? KT : 16>(vk, a.k_stride, a.k2_stride, wid, lane);
    piece_offsets<DV, DV, DR ? KT : 16>(vv, a.v_stride, 0, wid, lane);
  }
  // GROUPS: where the next tile's rows begin (of a plain matrix; else the cache's first), and the bytes of a row
  const uint32_t lds0 = lds_address(lds);
  const int row_k = (int)a.k_stride * 2, row_v = (int)a.v_stride * 2, row_k2 = (int)a.k2_stride * 2;
  const long row0 = DR ? base + kl.skip : 0;
  uintptr_t at_k = (uintptr_t)(a.k + kvh * DK) + row0 * row_k, at_v = (uintptr_t)(a.v + kvh * DV) + row0 * row_v,
            at_k2 = (uintptr_t)a.k2 + row0 * row_k2;
  const auto stage = [&](int buf, int x0) {
    if constexpr (GROUPS) {
      const uint32_t to = lds0 + buf * TILE_B;
      const int left = kl.n - x0;                              // (only the last tile's are fewer than its rows)
      if constexpr (DR != 0) {
        const int n = left < KT ? left : KT;
        const u32x4 head = bytes_at(at_k, n * row_k), tail = bytes_at(at_k2, n * row_k2), vals = bytes_at(at_v, n * row_v);
        stage_together<KW, DK>(to, wid, vk, [&](int, bool t) { return t ? tail : head; });
        stage_together<DV, DV>(to + TILE_K, wid, vv, [&](int, bool) { return vals; });
        at_k += KT * row_k, at_k2 += KT * row_k2, at_v += KT * row_v;
      } else {
        const int rows4 = table[(x0 >> 4) + (lane & 3)];
        const auto rows = [&](uintptr_t m, int row, int g) {
          const int n = left - 16 * g;
          return bytes_at(m + (long)__builtin_amdgcn_readlane(rows4, g) * row, n >= 16 ? 16 * row : n > 0 ? n * row : 0);
        };
        stage_together<KW, DK>(to, wid, vk, [&](int g, bool) { return rows(at_k, row_k, g); });
        stage_together<DV, DV>(to + TILE_K, wid, vv, [&](int g, bool) { return rows(at_v, row_v, g); });
      }
      return;
    }
    char* kd = lds + buf * TILE_B;
    stage_rows<KW, DK>(a.k + kvh * DK, a.k_stride, a.k2, a.k2_stride, kd, x0, wid, lane, row_in_list);
    stage_rows<DV, DV>(a.v + kvh * DV, a.v_stride, nullptr, 0, kd + TILE_K, x0, wid, lane, row_in_list);
  };
  const auto wait_one_tile = [&]() {                           // all but the youngest tile landed
    constexpr int LO = NPK / 8 + NPV / 8, RK = NPK % 8, RV = NPV % 8;
    static_assert(LO + 2 < 16, "vmcnt field");
    const int extra = (wid < RK) + (wid < RV);                 // wave-uniform
    constexpr int BASE = (7 << 4) | (15 << 8);                 // other counters at their maxima
    if (extra == 0) __builtin_amdgcn_s_waitcnt(LO | BASE);
    else if (extra == 1) __builtin_amdgcn_s_waitcnt((LO + 1) | BASE);
    else __builtin_amdgcn_s_waitcnt((LO + 2) | BASE);
    asm volatile("" ::: "memory");
  };
  stage(0, 0);
  // the queries are there from here on: hipcc would wait for them where it first uses them, in every tile, and so for the
  // DMA in flight, which it does not count
  if constexpr (GROUPS)
#pragma unroll
    for (int c = 0; c < KC; ++c) asm volatile("" : "+v"(qf[c]));
  if (ntiles > 1) {
    stage(1, KT);
    wait_one_tile();
  } else {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  __syncthreads();
  const int g16 = lane >> 4, q4 = (lane >> 2) & 3, p4 = lane & 3;
  int kbase[2], vbase[2];
#pragma unroll
  for (int par = 0; par < 2; ++par)
    kbase[par] = RGK * (qc >> 3) + 64 * (qc & 7) + 16 * ((2 * par + hi) ^ ((qc >> 2) & 3));
  {
    const int cl = 2 * (g16 & 1) + (p4 >> 1);
    vbase[0] = 64 * (4 * hi + q4) + 16 * (cl ^ hi) + 8 * (p4 & 1);
    vbase[1] = RGV + 64 * (4 * hi + q4) + 16 * (cl ^ (hi ^ 2)) + 8 * (p4 & 1);
  }
  f32x16 sacc[2];
  int cur = 0;
  for (int t = 0; t < ntiles; ++t) {
    const int x0 = t * KT;
    if (t + 2 < ntiles) stage(cur == 0 ? 2 : cur - 1, x0 + 2 * KT);
    const int kt0 = kl.key(x0), kt1 = kl.key(x0 + KT - 1);     // the tile's first and last key
    // tiles above this wave's rows, or all of them past its window and not kept, are skipped
    if (active && kt0 <= wq_hi && (kt1 > wq_lo - a.window || kt0 < a.keep)) {
      const char* kt = lds + cur * TILE_B;
#pragma unroll
      for (int sub = 0; sub < 2; ++sub) {
#pragma unroll
        for (int r = 0; r < 16; ++r) sacc[sub][r] = 0.f;
#pragma unroll
        for (int c = 0; c < KC; ++c) {
          const bf16x8 kf = *reinterpret_cast<const bf16x8*>(
              kt + kbase[c & 1] + 4 * RGK * sub + 512 * (c >> 1));
          sacc[sub] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[c], sacc[sub], 0, 0, 0);
        }
      }
      // only tiles that cross this wave's diagonal or the window's far edge are masked
      if (FOUND != BLOCKS && kt0 >= a.keep && (kt1 > wq_lo || wq_hi - kt0 >= a.window)) {
        // (one run of keys: those seen are the window's that end at the query)
        const int first = kt0 + 4 * hi - (qpos - a.window + 1);
#pragma unroll
        for (int sub = 0; sub < 2; ++sub)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            sacc[sub][r] = (unsigned)(first + 32 * sub + (r & 3) + 8 * (r >> 2)) < (unsigned)a.window ? sacc[sub][r]
                                                                                                     : -INFINITY;
      } else if (kt1 > wq_lo || wq_hi - kt0 >= a.window) {
#pragma unroll
        for (int sub = 0; sub < 2; ++sub)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int key = kl.key(x0 + 32 * sub + (r & 3) + 8 * (r >> 2) + 4 * hi);
            if (key > qpos || (qpos - key >= a.window && key >= a.keep)) sacc[sub][r] = -INFINITY;
          }
      }
      float mloc = max3(sacc[0][0], sacc[0][1], sacc[0][2]);
#pragma unroll
      for (int r = 3; r < 15; r += 2) mloc = max3(mloc, sacc[0][r], sacc[0][r + 1]);
      mloc = max3(mloc, sacc[0][15], sacc[1][0]);
#pragma unroll
      for (int r = 1; r < 15; r += 2) mloc = max3(mloc, sacc[1][r], sacc[1][r + 1]);
      mloc = fmaxf(mloc, sacc[1][15]);
      mloc = fmaxf(mloc, __shfl_xor(mloc, 32, 64));
      float alpha = 1.f;
      if ((mloc - m_run) * a.scale_log2 > RESCALE_THR) {
        alpha = m_run == -INFINITY ? 0.f
                                   : __builtin_amdgcn_exp2f((m_run - mloc) * a.scale_log2);
        m_run = mloc;
      }
      const float mc = (m_run == -INFINITY ? 0.f : m_run) * a.scale_log2;
      float psum = 0.f;
#pragma unroll
      for (int sub = 0; sub < 2; ++sub)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float e = __builtin_amdgcn_exp2f(fmaf(sacc[sub][r], a.scale_log2, -mc));
          sacc[sub][r] = e;
          psum += e;
        }
      l_part = l_part * alpha + psum;
      if (__ballot(alpha != 1.f)) {
#pragma unroll
        for (int i = 0; i < DBK; ++i)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[i][r] *= alpha;
      }
      const char* vt = kt + TILE_K;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const int sub = ks >> 1, hs = ks & 1;
        bf16x8 pb;
#pragma unroll
        for (int j = 0; j < 8; ++j) pb[j] = (__bf16)sacc[sub][8 * hs + j];
#pragma unroll
        for (int db = 0; db < DBK; ++db) {
          const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) s16x4*)(vt + vbase[0] + 2 * RGV * ks + 512 * db));
          const s16x4 up = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) s16x4*)(vt + vbase[1] + 2 * RGV * ks + 512 * db));
          const s16x8 w = {lo[0], lo[1], lo[2], lo[3], up[0], up[1], up[2], up[3]};
          o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8*>(&w),
                                                         pb, o[db], 0, 0, 0);
        }
      }
    }
    if (t + 2 < ntiles) wait_one_tile();
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);                          // lgkmcnt(0): own reads done
    __builtin_amdgcn_s_barrier();
    cur = (cur == 2) ? 0 : cur + 1;
  }
  if (!active) return;
  const float l_tot = l_part + __shfl_xor(l_part, 32, 64);
  const int qr = q0 + qc;
  if (qr < len) {
    const float inv = norm_factor(a.sink, h, m_run * a.scale_log2, l_tot) * head_factor(a, t0 + qr, h);
    u16* op = a.out + (long)(t0 + qr) * a.ldo + (long)h * DV;
    const float* gp = a.gate && !a.head_gate ? a.gate + (long)(t0 + qr) * a.ldg + (long)h * DV : nullptr;
#pragma unroll
    for (int db = 0; db < DBK; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f32x4 w = {1.f, 1.f, 1.f, 1.f};
        if (gp != nullptr) {
          w = *reinterpret_cast<const f32x4*>(gp + 32 * db + 8 * g + 4 * hi);
#pragma unroll
          for (int r = 0; r < 4; ++r) w[r] = sigmoid32(w[r]);
        }
        U16x4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v.v[r] = f2bf(o[db][4 * g + r] * inv * w[r]);
        *reinterpret_cast<U16x4*>(op + 32 * db + 8 * g + 4 * hi) = v;
      }
  }
}

// 4 waves x 16 query rows of one head
template <int DK, int DV>
__global__ void __launch_bounds__(256) swa_prefill16_kernel(SwaArgs a) {
  constexpr int KK = DK / 32, DB = DV / 16, ROWK = DK + 16, ROWV = DV + 16;
  constexpr int CHK = DK / 8, CHV = DV / 8, PK = KT * CHK / 256, PV = KT * CHV / 256;
  __shared__ __attribute__((aligned(16))) u16 ktile[KT * ROWK];
  __shared__ __attribute__((aligned(16))) u16 vtile[KT * ROWV];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int s = blockIdx.y, h = blockIdx.z;
  const int col = lane & 15, grp = lane >> 4;
  const int t0 = a.cu[s], len = a.cu[s + 1] - t0;
  const int wg_q0 = blockIdx.x * 64;
  if (wg_q0 >= len) return;                                      // workgroup-uniform
  const int p0 = a.positions[t0];
  const int q0 = wg_q0 + wid * 16;
  const bool active = q0 < len;
  const int kvh = h / (a.H / a.G);
  const KeyList kl(p0 + wg_q0, p0 + min(wg_q0 + 64, len) - 1, a.window, a.keep);
  const int* bt = a.block_tables + (long)s * a.bt_stride;
  bf16x8 qf[KK];
  {
    const u16* qp = a.q + (long)(t0 + min(q0 + col, len - 1)) * a.ldq + (long)h * DK;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      const uint4 v = *reinterpret_cast<const uint4*>(qp + kk * 32 + grp * 8);
      qf[kk] = *reinterpret_cast<const bf16x8*>(&v);
    }
  }
  const int my_q = p0 + q0 + col, wq_lo = p0 + q0, wq_hi = p0 + min(q0 + 16, len) - 1;
  float m_run = -INFINITY, l_part = 0.f;
  f32x4 o_acc[DB];
#pragma unroll
  for (int i = 0; i < DB; ++i) o_acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  // the next tile in flight in registers (of a native vector type: arrays of
  // HIP's uint4 would be kept in memory)
  u32x4 kr[PK], vr[PV];
  const auto row_at = [&](int x) {
    const int key = kl.key(min(x, kl.n - 1));
    return (long)bt[key / a.block_size] * a.block_size + key % a.block_size;
  };
  const auto load_tile = [&](int x0) {
#pragma unroll
    for (int j = 0; j < PK; ++j) {
      const int i = tid + 256 * j;
      kr[j] = *reinterpret_cast<const u32x4*>(a.k + row_at(x0 + i / CHK) * a.k_stride + kvh * DK +
                                              (i % CHK) * 8);
    }
#pragma unroll
    for (int j = 0; j < PV; ++j) {
      const int i = tid + 256 * j;
      vr[j] = *reinterpret_cast<const u32x4*>(a.v + row_at(x0 + i / CHV) * a.v_stride + kvh * DV +
                                              (i % CHV) * 8);
    }
  };
  load_tile(0);
  const int qrow = (lane >> 2) & 3, pcol = lane & 3;
  for (int x0 = 0; x0 < kl.n; x0 += KT) {
    __syncthreads();                                             // previous tile fully read
#pragma unroll
    for (int j = 0; j < PK; ++j) {
      const int i = tid + 256 * j;
      *reinterpret_cast<u32x4*>(ktile + i / CHK * ROWK + i % CHK * 8) = kr[j];
    }
#pragma unroll
    for (int j = 0; j < PV; ++j) {
      const int i = tid + 256 * j;
      *reinterpret_cast<u32x4*>(vtile + i / CHV * ROWV + i % CHV * 8) = vr[j];
    }
    __syncthreads();
    if (x0 + KT < kl.n) load_tile(x0 + KT);                      // in flight during compute
    const int kt0 = kl.key(x0), kt1 = kl.key(x0 + KT - 1);
    if (!active || kt0 > wq_hi || (kt1 <= wq_lo - a.window && kt0 >= a.keep)) continue;
    f32x4 s_acc[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const u16* kp = ktile + (16 * u + col) * ROWK;
      s_acc[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < KK; ++kk)
        s_acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            *reinterpret_cast<const bf16x8*>(kp + kk * 32 + grp * 8), qf[kk], s_acc[u], 0, 0, 0);
    }
    float p[16], tmax = -INFINITY;
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int key = kl.key(x0 + 16 * u + 4 * grp + r);
        const bool seen = key <= my_q && (my_q - key < a.window || key < a.keep);
        const float v = seen ? s_acc[u][r] * a.scale_log2 : -INFINITY;
        p[u * 4 + r] = v;
        tmax = fmaxf(tmax, v);
      }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
    const float m_new = fmaxf(m_run, tmax);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;        // nothing seen yet: keep it finite
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_use);
    m_run = m_new;
    float psum = 0.f;
#pragma unroll
    for (int j = 0; j < 16; ++j) { p[j] = __builtin_amdgcn_exp2f(p[j] - m_use); psum += p[j]; }
    l_part = l_part * alpha + psum;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float al = __shfl(alpha, 4 * grp + r, 64);
#pragma unroll
      for (int i = 0; i < DB; ++i) o_acc[i][r] *= al;
    }
    // O += P . V, two 32-key halves; B operand rows: keys 32 hh + 4 grp + q and 16 further on
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      bf16x8 pa;
#pragma unroll
      for (int j = 0; j < 8; ++j) pa[j] = (__bf16)p[8 * hh + j];
#pragma unroll
      for (int i = 0; i < DB; ++i) {
        const u16* a0 = vtile + (32 * hh + 4 * grp + qrow) * ROWV + 16 * i + 4 * pcol;
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4*)(a0));
        const s16x4 up = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4*)(a0 + 16 * ROWV));
        const s16x8 w = {lo[0], lo[1], lo[2], lo[3], up[0], up[1], up[2], up[3]};
        o_acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            pa, *reinterpret_cast<const bf16x8*>(&w), o_acc[i], 0, 0, 0);
      }
    }
  }
  if (!active) return;
  float l_tot = l_part + __shfl_xor(l_part, 16, 64);
  l_tot += __shfl_xor(l_tot, 32, 64);
  const float inv = norm_factor(a.sink, h, m_run, l_tot) * head_factor(a, t0 + min(q0 + col, len - 1), h);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float iv = __shfl(inv, 4 * grp + r, 64);
    const int qr = q0 + 4 * grp + r;
    if (qr < len) {
      u16* op = a.out + (long)(t0 + qr) * a.ldo + (long)h * DV;
      const float* gp = a.gate && !a.head_gate ? a.gate + (long)(t0 + qr) * a.ldg + (long)h * DV : nullptr;
#pragma unroll
      for (int i = 0; i < DB; ++i) {
        float v = o_acc[i][r] * iv;
        if (gp != nullptr) v *= sigmoid32(gp[16 * i + col]);
        op[16 * i + col] = f2bf(v);
      }
    }
  }
}

// One query token a sequence. Workgroup = 4 waves of one (sequence, kv head, chunk of HP heads,
// key split); a wave takes every fourth 32-key tile of the split. PAST: what it reads past the caches (0
// nothing, 1 the values, 2 the keys too), see launch_swa.
template <int DK, int DV, int HP, int PAST>
__global__ void __launch_bounds__(256) swa_decode_kernel(SwaArgs a) {
  constexpr int KK = DK / 32, LPR = DV / 8;        // lanes that cover a V row with 16 bytes each
  constexpr int KPI = 64 / LPR, NV = 32 / KPI;     // keys per V load of a wave, V loads per tile
  static_assert(32 % KPI == 0, "V loads tile 32 keys");
  __shared__ __attribute__((aligned(16))) float pl[4][32][HP];
  __shared__ __attribute__((aligned(16))) float ol[4][HP][DV];
  __shared__ float ml[4][HP][2];
  const int rep = a.H / a.G, nhc = (rep + HP - 1) / HP;
  const int s = blockIdx.y, split = blockIdx.z;
  const int kvh = blockIdx.x / nhc, h0 = kvh * rep + (blockIdx.x % nhc) * HP;
  const int nh = min(HP, (kvh + 1) * rep - h0);
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int fr = lane & 15, fq = lane >> 4;
  const int t = a.cu[s];
  if (a.cu[s + 1] <= t) return;
  const int p = a.positions[t];
  const KeyList kl(p, p, a.window, a.keep);
  const int* bt = a.block_tables + (long)s * a.bt_stride;
  const int ntiles = (kl.n + 31) / 32, per = (ntiles + a.nsplit - 1) / a.nsplit;
  const int tile_hi = min(ntiles, (split + 1) * per);
  bf16x8 qf[KK];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) {
    uint4 v = uint4{0u, 0u, 0u, 0u};
    if (fr < nh)
      v = *reinterpret_cast<const uint4*>(a.q + (long)t * a.ldq + (long)(h0 + fr) * DK + kk * 32 +
                                          fq * 8);
    qf[kk] = *reinterpret_cast<const bf16x8*>(&v);
  }
  float m_run = -INFINITY, l_run = 0.f;            // of head fr
  float acc[HP][8];
#pragma unroll
  for (int h = 0; h < HP; ++h)
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[h][i] = 0.f;
  for (int tile = split * per + wid; tile < tile_hi; tile += 4) {
    const int x0 = tile * 32;
    const int key = kl.key(min(x0 + (lane & 31), kl.n - 1));
    const int row = bt[key / a.block_size] * a.block_size + key % a.block_size;
    bf16x8 kf[2][KK];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const long r = __shfl(row, 16 * u + fr, 64);
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        const uint4 v = load16<(PAST > 1)>(a.k + r * a.k_stride + kvh * DK + kk * 32 + fq * 8);
        kf[u][kk] = *reinterpret_cast<const bf16x8*>(&v);
      }
    }
    uint4 vv[NV];
    // (widths whose rows do not tile a wave leave its last lanes to repeat the last key's row)
    const int vk = min(lane / LPR, KPI - 1);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const long r = __shfl(row, i * KPI + vk, 64);
      vv[i] = load16<(PAST > 0)>(a.v + r * a.v_stride + kvh * DV + (lane % LPR) * 8);
    }
    f32x4 sa[2];
    float tmax = -INFINITY;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      sa[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < KK; ++kk)
        sa[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[u][kk], qf[kk], sa[u], 0, 0, 0);
      // lane: head fr, keys x0 + 16 u + 4 fq + r; every listed key is seen
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        sa[u][r] = x0 + 16 * u + 4 * fq + r < kl.n ? sa[u][r] * a.scale_log2 : -INFINITY;
        tmax = fmaxf(tmax, sa[u][r]);
      }
    }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
    const float m_new = fmaxf(m_run, tmax);        // finite: a tile holds at least one key
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
    m_run = m_new;
    float psum = 0.f;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float e = __builtin_amdgcn_exp2f(sa[u][r] - m_new);
        psum += e;
        if (fr < HP) pl[wid][16 * u + 4 * fq + r][fr] = e;
      }
    l_run = l_run * alpha + psum;                  // this lane's keys only
    if (__ballot(fr < nh && alpha != 1.f)) {
#pragma unroll
      for (int h = 0; h < HP; ++h) {
        const float al = __shfl(alpha, h, 64);
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[h][i] *= al;
      }
    }
    // the wave's own weights, written above by its own lanes: in order in the LDS pipe
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      float v8[8];
      unpack8bf(vv[i], v8);
      const float* pr = pl[wid][i * KPI + vk];
#pragma unroll
      for (int h = 0; h < HP; ++h) {
        const float w = pr[h];
#pragma unroll
        for (int c = 0; c < 8; ++c) acc[h][c] += w * v8[c];
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  l_run += __shfl_xor(l_run, 16, 64);
  l_run += __shfl_xor(l_run, 32, 64);
  if (lane < HP) { ml[wid][lane][0] = m_run; ml[wid][lane][1] = l_run; }
#pragma unroll
  for (int h = 0; h < HP; ++h)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float v = acc[h][i];
      if constexpr ((LPR & (LPR - 1)) == 0) {
#pragma unroll
        for (int o = LPR; o < 64; o <<= 1) v += __shfl_xor(v, o, 64);
      } else {                                     // lanes below LPR gather their column's sums
        const float own = v;
#pragma unroll
        for (int k = 1; k < KPI; ++k) v += __shfl(own, (lane + k * LPR) & 63, 64);
      }
      acc[h][i] = v;
    }
  if (lane < LPR) {
#pragma unroll
    for (int h = 0; h < HP; ++h) {
      *reinterpret_cast<f32x4*>(&ol[wid][h][lane * 8]) =
          f32x4{acc[h][0], acc[h][1], acc[h][2], acc[h][3]};
      *reinterpret_cast<f32x4*>(&ol[wid][h][lane * 8 + 4]) =
          f32x4{acc[h][4], acc[h][5], acc[h][6], acc[h][7]};
    }
  }
  __syncthreads();
  const int S = gridDim.y;
  float* stats = a.ws;
  float* part = a.ws + stat_floats(a.nsplit, S, a.H);
  for (int i = tid; i < nh * DV; i += 256) {
    const int h = i / DV, c = i % DV;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < 4; ++w) M = fmaxf(M, ml[w][h][0]);
    float L = 0.f, o = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      if (ml[w][h][0] == -INFINITY) continue;      // a wave without tiles
      const float e = __builtin_amdgcn_exp2f(ml[w][h][0] - M);
      L += ml[w][h][1] * e;
      o += ol[w][h][c] * e;
    }
    if (a.nsplit == 1) {
      const int oc = (h0 + h) * DV + c;
      float v = o * norm_factor(a.sink, h0 + h, M, L) * head_factor(a, t, h0 + h);
      if (a.gate != nullptr && !a.head_gate) v *= sigmoid32(a.gate[(long)t * a.ldg + oc]);
      a.out[(long)t * a.ldo + oc] = f2bf(v);
    } else {
      const long b = ((long)split * S + s) * a.H + h0 + h;
      part[b * DV + c] = o;
      if (c == 0) { stats[2 * b] = M; stats[2 * b + 1] = L; }
    }
  }
}

// out = the splits' un-normalised partial sums, weighed by their (max, sum); 4 columns a thread
template <int DV>
__global__ void __launch_bounds__(256) swa_reduce_kernel(SwaArgs a, int S) {
  const long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int w4 = a.H * DV / 4;
  if (gid >= (long)S * w4) return;
  const int s = (int)(gid / w4), c = (int)(gid % w4) * 4, h = c / DV;
  if (a.cu[s + 1] <= a.cu[s]) return;
  const float* stats = a.ws;
  const float* part = a.ws + stat_floats(a.nsplit, S, a.H);
  float M = -INFINITY;
  for (int k = 0; k < a.nsplit; ++k) M = fmaxf(M, stats[2 * (((long)k * S + s) * a.H + h)]);
  float L = 0.f;
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
  for (int k = 0; k < a.nsplit; ++k) {
    const long b = ((long)k * S + s) * a.H + h;
    if (stats[2 * b] == -INFINITY) continue;       // a split without keys
    const float e = __builtin_amdgcn_exp2f(stats[2 * b] - M);
    L += stats[2 * b + 1] * e;
    o += e * *reinterpret_cast<const f32x4*>(part + b * DV + c % DV);
  }
  o *= norm_factor(a.sink, h, M, L) * head_factor(a, a.cu[s], h);
  if (a.gate != nullptr && !a.head_gate) {
    const f32x4 g = *reinterpret_cast<const f32x4*>(a.gate + (long)a.cu[s] * a.ldg + c);
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] *= sigmoid32(g[i]);
  }
  uint2 pk;
  pk.x = pack2bf(o[0], o[1]);
  pk.y = pack2bf(o[2], o[3]);
  *reinterpret_cast<uint2*>(a.out + (long)a.cu[s] * a.ldo + c) = pk;
}

int decode_splits(int num_seqs, int H, int G, long keys) {
  const int rep = H / G, hp = rep <= 4 ? 4 : 8;
  const long base = (long)num_seqs * G * ((rep + hp - 1) / hp);
  const long keys_most = (keys + 127) / 128;       // a tile for each wave of a workgroup
  const int most = (int)(keys_most > 32 ? 32 : keys_most);
  // 256 units and more: to 1536 workgroups, so that long contexts among short ones are cut (contexts of
  // 64 to 2000 keys, 32 heads on 8: 32 sequences 45 us with 6 splits, 56 whole; 64 77 with 3, 84 whole).
  // Fewer: a CU's time goes with the keys that its workgroups read, so what counts is how evenly 512
  // workgroups or more fill 256 CUs: ceil(base n / 256) / n of a sequence for the fullest, and 0.004 of
  // one for every split's share of the merge. With 1536 before; us, 8 sequences of 4000 keys 53 -> 39,
  // 16 of 2000 44 -> 36, 24 of 2000 53 -> 48; 8 of 64 to 4000 45 -> 35, 24 of 64 to 2000 40 -> 34.
  if (base >= 256) {
    const long n = (1536 + base - 1) / base;
    return n > most ? most : (int)n;
  }
  int best = (int)((512 + base - 1) / base);
  if (best >= most) return most < 1 ? 1 : most;
  float least = 1e30f;
  for (int n = best; n <= most && base * n <= 1536; ++n) {
    const float cost = (float)((base * n + 255) / 256) / (float)n + 0.004f * (float)n;
    if (cost < least) { least = cost; best = n; }
  }
  return best;
}

// key / value widths this file is built for
#define SWA_WIDTHS(F) F(64, 64) F(128, 128) F(64, 128) F(96, 192) F(128, 256)

template <int DK, int DR, int DV, int FOUND>
int launch_prefill32(SwaArgs a, int sh, int num_seqs, int max_seqlen, hipStream_t st) {
  static bool raised = false;
  if (!raised) {
    const hipError_t e = hipFuncSetAttribute((const void*)swa_prefill32_kernel<DK, DR, DV, FOUND>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize,
                                             160 * 1024);
    if (e != hipSuccess) return (int)e;
    raised = true;
  }
  const int blocks = (max_seqlen + LROWS - 1) / LROWS;
  const dim3 grid = a.H <= 4 ? dim3(blocks, num_seqs, a.H) : dim3(blocks * a.H, num_seqs);
  swa_prefill32_kernel<DK, DR, DV, FOUND><<<grid, 512, sh, st>>>(a);
  DLI_RETURN_LAUNCH();
}

// How a launch's tiles are found, and its LDS
struct Form {
  int found, lds;
};
template <int DK, int DR, int DV>
Form portion_form(long k_stride, long v_stride, long k2_stride, int block_size, int window, int keep) {
  constexpr int TILES = 3 * KT * (DK + DR + DV) * 2, MOST = 160 * 1024;
  const long list = (long)window + LROWS + keep;
  // Rows that lie together, by 31-bit offsets, apart from one another, and a table of the list's sixteens beside the tiles
  // (at 128 + 128 wide it has room for 260 thousand keys, at 128 + 256 for 65 thousand). Row by row otherwise, the former way, through a table of rows
  // or the block table itself, whose loads wait for all DMA in flight. That way and its mask, by runs and key by key,
  // against this one and the mask of one run, us, 32 heads of 128 on 8 with a sink and a gate a head: 5 portions of
  // 900 to 2601 tokens 285 -> 203, in windows of 1024 217 -> 171, 8000 tokens 767 -> 567 (0.92 PFLOP/s); expanded latent
  // heads, 6 of 301 to 3000 222 -> 199, in windows of 1024 187 -> 158. The mask is 13 % of the first and all of the last
  const auto fits = [](long stride, int wide) { return stride >= wide && stride < (1l << 31) / (2 * (DR ? KT : 16)); };
  if (fits(k_stride, DK) && fits(v_stride, DV) && (DR == 0 || fits(k2_stride, DR))) {
    if (DR) return {SIXTEENS, TILES};
    const long sixteens = (list + 32 + 63) / KT * 4;
    if (block_size >= 16 && (block_size & (block_size - 1)) == 0 && TILES + sixteens * 4 <= MOST)
      return {SIXTEENS, TILES + (int)sixteens * 4};
  }
  if (DR == 0 && list <= 6144 && TILES + list * 4 <= MOST) return {ROWS, TILES + (int)list * 4};
  return {BLOCKS, TILES};
}

template <int DK, int DR, int DV>
int launch_prefill32(SwaArgs a, int num_seqs, int max_seqlen, hipStream_t st) {
  const Form f = portion_form<DK, DR, DV>(a.k_stride, a.v_stride, a.k2_stride, a.block_size, a.window, a.keep);
  if (f.found == SIXTEENS) {
    a.block_shift = __builtin_ctz(a.block_size);
    return launch_prefill32<DK, DR, DV, SIXTEENS>(a, f.lds, num_seqs, max_seqlen, st);
  }
  if constexpr (DR == 0)
    if (f.found == ROWS) return launch_prefill32<DK, DR, DV, ROWS>(a, f.lds, num_seqs, max_seqlen, st);
  return launch_prefill32<DK, DR, DV, BLOCKS>(a, f.lds, num_seqs, max_seqlen, st);
}

template <int DK, int DV>
int launch_swa(SwaArgs a, int num_seqs, int max_seqlen, hipStream_t st) {
  if (max_seqlen == 1) {
    const int rep = a.H / a.G, hp = rep <= 4 ? 4 : 8;
    dim3 grid(a.G * ((rep + hp - 1) / hp), num_seqs, a.nsplit);
    // Keys and values are read past the caches: 4 of 300 keys 12.0 -> 11.0 us, 32 of 64 7.3 -> 6.5. Not the keys of
    // few long sequences, whose rows arrive in two pieces and which the tail of a step of different lengths waits
    // for (8 kv heads of 128, 16 of 63 to 8000 keys 89 us, the keys through the caches 77, the values too 80); from
    // 192 (sequence, kv head) pairs on the whole chip reads, and what the keys push out of the caches costs the rest of the
    // step more (24 of 2083 keys on 8 kv heads, two such layers of a step: 660 us, 693). Not where several
    // workgroups read a kv head's keys and the second one would find them (16 heads a kv head: 128 of 8000 keys
    // 370 us, 308 through the caches; 16 heads on one of 128 and 256, 64 of 1000 keys, 49 MB, 33 and 30; 4 of 8000
    // on two, 33 MB, 36 and 45).
    const long keys = (long)a.window + a.keep, bytes = (long)num_seqs * a.G * keys * (DK + DV) * 2;
    const bool all = bytes <= 48l << 20 || ((long)num_seqs * a.G >= 192 && keys < 4096);
#define SWA_DECODE(HP, PAST) swa_decode_kernel<DK, DV, HP, PAST><<<grid, 256, 0, st>>>(a)
    if (rep > 8 && bytes > 36l << 20) SWA_DECODE(8, 0);
    else if (hp == 4) all ? (void)SWA_DECODE(4, 2) : (void)SWA_DECODE(4, 1);
    else all ? (void)SWA_DECODE(8, 2) : (void)SWA_DECODE(8, 1);
#undef SWA_DECODE
    if (a.nsplit > 1) {
      const long n = (long)num_seqs * a.H * DV / 4;
      swa_reduce_kernel<DV><<<(int)((n + 255) / 256), 256, 0, st>>>(a, num_seqs);
    }
    DLI_RETURN_LAUNCH();
  }
  if (max_seqlen < 192) {
    dim3 grid((max_seqlen + 63) / 64, num_seqs, a.H);
    swa_prefill16_kernel<DK, DV><<<grid, 256, 0, st>>>(a);
    DLI_RETURN_LAUNCH();
  }
  return launch_prefill32<DK, 0, DV>(a, num_seqs, max_seqlen, st);
}


// Rows [cu_ctx[s], cu_ctx[s + 1]) of out <- the cache rows of the last positions of sequence s, whose
// new tokens are rows [cu[s], cu[s + 1]), `chunks` 16-byte pieces each
__global__ void __launch_bounds__(256) gather_rows_kernel(uint4* out, const uint4* cache,
                                                          const int* cu_ctx, const int* cu,
                                                          const int* positions, const int* block_tables,
                                                          int bt_stride, int block_size, int chunks) {
  const int s = blockIdx.y, o0 = cu_ctx[s], n = cu_ctx[s + 1] - o0;
  const int* bt = block_tables + (long)s * bt_stride;
  const int j0 = blockIdx.x * 64, rows = min(64, n - j0);
  if (rows <= 0 || cu[s + 1] <= cu[s]) return;
  const int first = positions[cu[s + 1] - 1] + 1 - n;
  for (int i = threadIdx.x; i < rows * chunks; i += 256) {
    const int j = j0 + i / chunks, c = i % chunks, p = first + j;
    const long row = (long)bt[p / block_size] * block_size + p % block_size;
    out[(long)(o0 + j) * chunks + c] = cache[row * chunks + c];
  }
}

}  // namespace

// The cached rows (width bf16 elements, a multiple of 8) of every sequence's last cu_ctx[s + 1] -
// cu_ctx[s] <= max_rows positions, in order
extern "C" int dli_gather_context(void* out, const void* cache, int width, const int* cu_ctx,
                                  const int* cu, const int* positions, const int* block_tables,
                                  int bt_stride, int block_size, int num_seqs, int max_rows,
                                  hipStream_t st) {
  if (num_seqs <= 0 || max_rows <= 0) return 0;
  if (width < 8 || width % 8 || block_size < 1 || num_seqs > 65535 ||
      (((uintptr_t)out | (uintptr_t)cache) & 15))
    return (int)hipErrorInvalidValue;
  dim3 grid((max_rows + 63) / 64, num_seqs);
  gather_rows_kernel<<<grid, 256, 0, st>>>((uint4*)out, (const uint4*)cache, cu_ctx, cu, positions,
                                           block_tables, bt_stride, block_size, width / 8);
  DLI_RETURN_LAUNCH();
}

// Portions whose keys share their last dr dims (latent attention, expanded): q [T, H*dk] and its tail
// q2 (row stride ldq2, head stride q2_head); k and v are rows [cu_ctx[s], cu_ctx[s + 1]), a sequence's
// last positions (every one that a query sees), of matrices with one column block a head, k2 [.., dr] of a third. hipErrorNotSupported (801): widths or alignment that this
// form does not take.
extern "C" int dli_shared_tail_attention(const void* q, int ldq, const void* q2, long ldq2, int q2_head,
                                         const void* k, long k_stride, const void* k2, long k2_stride,
                                         const void* v, long v_stride, void* out, int ldo, const int* cu,
                                         const int* positions, const int* cu_ctx, int num_seqs,
                                         int max_seqlen, int H, int dk, int dr, int dv, int window,
                                         float scale, const float* gate, int ldg, hipStream_t st) {
  if (num_seqs <= 0 || max_seqlen <= 0) return 0;
  if (H < 1 || window < 1 || cu_ctx == nullptr) return (int)hipErrorInvalidValue;
  const bool aligned = (((uintptr_t)q | (uintptr_t)q2 | (uintptr_t)k | (uintptr_t)k2 | (uintptr_t)v) & 15) == 0 &&
                       (uintptr_t)out % 8 == 0 && ldq % 8 == 0 && ldq2 % 8 == 0 && q2_head % 8 == 0 &&
                       k_stride % 8 == 0 && k2_stride % 8 == 0 && v_stride % 8 == 0 && ldo % 4 == 0;
  if (!aligned || !(scale > 0.f) || num_seqs > 65535 || H > 65535 || dk != 128 || dr != 64 || dv != 128)
    return (int)hipErrorNotSupported;
  SwaArgs a{(const u16*)q, ldq, (const u16*)k, k_stride, (const u16*)v, v_stride, (u16*)out, ldo,
            gate, ldg, gate != nullptr, nullptr, 1.f, cu, positions, nullptr, 0, 1, H, H, window, 0,
            scale * LOG2E, 0, 1, nullptr, (const u16*)q2, ldq2, q2_head, (const u16*)k2, k2_stride, cu_ctx};
  return launch_prefill32<128, 64, 128>(a, num_seqs, max_seqlen, st);
}

// Workspace bytes of a decode step (0: not split over keys)
extern "C" long dli_swa_attention_workspace_bytes(int num_seqs, int max_seqlen, int H, int G,
                                                  int dv, int window, int keep) {
  if (max_seqlen != 1 || H < 1 || G < 1) return 0;
  const int n = decode_splits(num_seqs, H, G, (long)window + keep);
  return n == 1 ? 0 : (stat_floats(n, num_seqs, H) + (long)n * num_seqs * H * dv) * 4;
}

// Returns hipErrorNotSupported (801) for shapes this family does not take. A decode step
// (max_seqlen 1) gets the workspace its query asked for.
extern "C" int dli_swa_attention(const void* q, int ldq, const void* k, long k_stride,
                                 const void* v, long v_stride, void* out, int ldo, const int* cu,
                                 const int* positions, const int* block_tables, int bt_stride,
                                 int block_size, int num_seqs, int max_seqlen, int H, int G,
                                 int dk, int dv, int window, int keep, float scale,
                                 const float* gate, int ldg, int head_gate, const float* sink,
                                 float out_scale, void* ws, hipStream_t st) {
  if (num_seqs <= 0 || max_seqlen <= 0) return 0;
  if (H < 1 || G < 1 || H % G || window < 1 || keep < 0 || block_size < 1)
    return (int)hipErrorInvalidValue;
  head_gate = head_gate && gate != nullptr;
  const bool aligned = (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v) & 15) == 0 &&
                       (uintptr_t)out % 8 == 0 && ldq % 8 == 0 && k_stride % 8 == 0 &&
                       v_stride % 8 == 0 && ldo % 4 == 0 &&
                       (gate == nullptr || head_gate ||
                        ((uintptr_t)gate % 16 == 0 && ldg % 4 == 0));
  if (!aligned || !(scale > 0.f) || num_seqs > 65535 || H > 65535)
    return (int)hipErrorNotSupported;
  SwaArgs a{(const u16*)q, ldq, (const u16*)k, k_stride, (const u16*)v, v_stride, (u16*)out, ldo,
            gate, ldg, head_gate != 0, sink, out_scale, cu, positions, block_tables, bt_stride, block_size, H, G, window, keep,
            scale * LOG2E, 0, 1, (float*)ws, nullptr, 0, 0, nullptr, 0, nullptr};
  if (max_seqlen == 1) {
    a.nsplit = decode_splits(num_seqs, H, G, (long)window + keep);
    if (a.nsplit > 1 && ws == nullptr) return (int)hipErrorInvalidValue;
  }
#define SWA_TRY(K, V) if (dk == K && dv == V) return launch_swa<K, V>(a, num_seqs, max_seqlen, st);
  SWA_WIDTHS(SWA_TRY)
#undef SWA_TRY
  return (int)hipErrorNotSupported;
}

// How portions of 192 tokens and more find their tiles: 2 by sixteens of rows, 1 by a table of rows, 0 by the block table; -1 where
// other kernels take them
extern "C" int dli_swa_portion_form(int dk, int dv, long k_stride, long v_stride, int block_size, int window, int keep) {
#define SWA_FORM(K, V) if (dk == K && dv == V) return portion_form<K, 0, V>(k_stride, v_stride, 0, block_size, window, keep).found;
  SWA_WIDTHS(SWA_FORM)
#undef SWA_FORM
  return -1;
}
