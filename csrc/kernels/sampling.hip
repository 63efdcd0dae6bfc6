// On-device token sampling with HF `generate` semantics.
//
// HF warper order (transformers/generation/utils.py): Temperature -> TopK -> TopP -> softmax
// -> multinomial. One 512-thread workgroup per row (vocab up to ~256k), no full-vocab sort:
//   * greedy (temperature <= 0 or top_k == 1): block argmax (first index on ties, like torch).
//   * top_k <= 0 and top_p >= 1: exact Gumbel-max sampling over the whole row in one pass.
//   * otherwise the top-k set (ties with the k-th kept, as HF's `scores < kth` mask keeps them):
//     up to k = 256 from the elements above a bound on the k-th largest, found from per-thread
//     maxima; larger k and rows this does not take by radix select (8-bit digits, early exit) and
//     a gather of <= CAP elements. The set is sorted, then temperature-softmax, top-p truncation
//     (keep j while the mass of strictly larger tokens < top_p, i.e. HF's `cumsum_asc <=
//     1-top_p` removal) and an inverse-CDF draw.
// Where the LM head left the largest key of every block of columns (BlockMax in gemm_common.h), the
// bound comes from these, and only the blocks that reach it are read. top_k 50 of 128k fp32 logits with
// the head's product before them, us: 512 rows 503 -> 449, 64 212 -> 201, 24 196 -> 184; of 32k, 64
// rows 64 -> 59. Greedy 512 rows 488 -> 430. One row of 16-column blocks 179 -> 173, where the head
// takes a kernel of 4-column ones (which leaves none) two phases as before.
// top_k is capped at CAP (2048). Randomness: Philox4x32-10 keyed by a per-row 64-bit seed
// supplied by the engine (seed = f(request seed, output index)), so a request samples the
// same tokens regardless of how it is batched.
#include "common.h"

#define SMP_THREADS 512
#define SMP_CAP 2048
// candidates ranked by counting; more go through the bitonic sort
#define SMP_RANK_MAX 128

__device__ __forceinline__ float key2f(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// Philox4x32-10
__device__ __forceinline__ uint4 philox(uint2 key, uint4 ctr) {
  const uint32_t M0 = 0xD2511F53u, M1 = 0xCD9E8D57u, W0 = 0x9E3779B9u, W1 = 0xBB67AE85u;
#pragma unroll
  for (int i = 0; i < 10; ++i) {
    const uint32_t hi0 = __umulhi(M0, ctr.x), lo0 = M0 * ctr.x;
    const uint32_t hi1 = __umulhi(M1, ctr.z), lo1 = M1 * ctr.z;
    ctr = make_uint4(hi1 ^ ctr.y ^ key.x, lo1, hi0 ^ ctr.w ^ key.y, lo0);
    key.x += W0; key.y += W1;
  }
  return ctr;
}
__device__ __forceinline__ float u01(uint32_t x) {           // (0, 1)
  return ((x >> 8) + 0.5f) * (1.0f / 16777216.0f);
}

struct ArgMax { float v; int i; };
__device__ __forceinline__ ArgMax amax(ArgMax a, ArgMax b) {
  if (b.v > a.v || (b.v == a.v && b.i < a.i)) return b;
  return a;
}
__device__ ArgMax block_argmax(ArgMax a, float* sv, int* si) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    ArgMax b{__shfl_xor(a.v, o, 64), __shfl_xor(a.i, o, 64)};
    a = amax(a, b);
  }
  const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) { sv[w] = a.v; si[w] = a.i; }
  __syncthreads();
  ArgMax r{sv[0], si[0]};
  for (int i = 1; i < nw; ++i) r = amax(r, ArgMax{sv[i], si[i]});
  return r;
}

// inclusive block scan of one float per thread (512 threads)
__device__ float block_scan(float v, float* tmp) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float t = __shfl_up(v, o, 64);
    if (lane >= o) v += t;
  }
  __syncthreads();
  if (lane == 63) tmp[w] = v;
  __syncthreads();
  float add = 0.f;
  for (int i = 0; i < w; ++i) add += tmp[i];
  (void)nw;
  return v + add;
}

// Radix-select digit step: the largest bin d whose suffix count S(d) = sum_{b >= d} hist[b]
// reaches k_rem (bins walked from 255 down), as one block scan over the 256 bins instead of
// a serial walk by one thread (up to 256 dependent LDS reads per pass). sel = {digit, count
// strictly above the digit's bin, count in it}; with S(0) < k_rem (fewer than k_rem keys):
// {0, S(0), 0}, so sel[1] + sel[2] < k_rem tells that case apart.
// All threads call it (block_scan barriers).
__device__ __forceinline__ void find_digit(const uint32_t* hist, uint32_t k_rem, float* tmp,
                                           uint32_t* sel) {
  const int tid = threadIdx.x;
  const uint32_t h = tid < 256 ? hist[255 - tid] : 0u;
  const uint32_t S = (uint32_t)block_scan((float)h, tmp);     // exact: counts < 2^24
  if (tid < 256) {
    const bool hit = S >= k_rem && S - h < k_rem;
    if (hit || (tid == 255 && S < k_rem)) {
      sel[0] = 255u - (uint32_t)tid;
      sel[1] = hit ? S - h : S;
      sel[2] = hit ? h : 0u;
    }
  }
}

// k-th largest non-zero key of keys[0..n) (LDS), 8-bit digits. Key 0 (an all-ones NaN
// pattern) marks an empty slot and is never counted. Returns 0 when fewer than k keys exist.
__device__ uint32_t radix_kth(const uint32_t* keys, int n, uint32_t k, uint32_t* hist,
                              float* tmp, uint32_t* sel) {
  uint32_t prefix = 0, pmask = 0, k_rem = k;
  for (int pass = 0; pass < 4; ++pass) {
    const int shift = 24 - 8 * pass;
    for (int i = threadIdx.x; i < 256; i += blockDim.x) hist[i] = 0;
    __syncthreads();
    for (int e = threadIdx.x; e < n; e += blockDim.x) {
      const uint32_t key = keys[e];
      if (key != 0u && (key & pmask) == prefix) atomicAdd(&hist[(key >> shift) & 255u], 1u);
    }
    __syncthreads();
    find_digit(hist, k_rem, tmp, sel);
    __syncthreads();
    if (k_rem > sel[1] + sel[2]) return 0u;                    // fewer than k keys
    k_rem -= sel[1];
    prefix |= sel[0] << shift;
    pmask |= 255u << shift;
  }
  return prefix;
}

// A threshold t with at least k of the wave's 64 * NR keys at or above it, the largest one unless
// exactly k keys are: bit by bit, one ballot per register and bit, no LDS and no barrier. 0 when
// fewer than k keys are non-zero. low: every key but empty (0) ones is at least that, so the bits
// it shares with the largest key need no step. steps: bits to find; fewer leave a lower threshold.
// (512 keys by four histogram passes: some 4 us in 20 barriers; by some 12 bits of 8 ballots 1 us,
// every wave for itself.)
template <int NR>
__device__ __forceinline__ uint32_t wave_kth(const uint32_t (&keys)[NR], int k, uint32_t low = 0u,
                                              int steps = 32) {
  uint32_t t = 0u;
  int bit = 31;
  if (low != 0u) {
    uint32_t top = low;
#pragma unroll
    for (int j = 0; j < NR; ++j) top = max(top, keys[j]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) top = max(top, (uint32_t)__shfl_xor((int)top, o, 64));
    const uint32_t diff = top ^ low;
    if (diff == 0u) return low;
    bit = 31 - __builtin_clz(diff);
    t = bit == 31 ? 0u : low >> (bit + 1) << (bit + 1);
  }
  for (; bit >= 0 && steps > 0; --bit, --steps) {
    const uint32_t c = t | (1u << bit);
    int cnt = 0;
#pragma unroll
    for (int j = 0; j < NR; ++j) cnt += __popcll(__ballot(keys[j] >= c));
    if (cnt >= k) t = c;
    if (cnt == k) break;
  }
  return t;
}

// Logits arrive as fp32 or as bf16 (u16: the LM head's output in the model dtype, as HF's
// `lm_head(hidden).float()` produces them); every comparison runs on the exact fp32 value.
__device__ __forceinline__ float ldv(const float* x, int i) { return x[i]; }
__device__ __forceinline__ float ldv(const u16* x, int i) { return bf2f(x[i]); }

// Visit every element of a row with 16-B loads, 8 in flight per thread, the last partial round
// too (the sampler is one workgroup per row, so memory-level parallelism per CU comes from ILP,
// not occupancy).
template <typename F>
__device__ __forceinline__ void visit16(const uint4 v, int base, const u16*, F&& f) {
  f(__uint_as_float(v.x << 16), base);     f(__uint_as_float(v.x & 0xffff0000u), base + 1);
  f(__uint_as_float(v.y << 16), base + 2); f(__uint_as_float(v.y & 0xffff0000u), base + 3);
  f(__uint_as_float(v.z << 16), base + 4); f(__uint_as_float(v.z & 0xffff0000u), base + 5);
  f(__uint_as_float(v.w << 16), base + 6); f(__uint_as_float(v.w & 0xffff0000u), base + 7);
}
template <typename F>
__device__ __forceinline__ void visit16(const uint4 v, int base, const float*, F&& f) {
  f(__uint_as_float(v.x), base);     f(__uint_as_float(v.y), base + 1);
  f(__uint_as_float(v.z), base + 2); f(__uint_as_float(v.w), base + 3);
}

// with a floor: only groups holding an element that is not below it
template <typename F>
__device__ __forceinline__ void visit16(const uint4 v, int base, const u16* x, F&& f, float lo) {
  bool any = false;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t w = j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w;
    any |= !(__uint_as_float(w << 16) < lo) | !(__uint_as_float(w & 0xffff0000u) < lo);
  }
  if (any) visit16(v, base, x, f);
}
template <typename F>
__device__ __forceinline__ void visit16(const uint4 v, int base, const float* x, F&& f, float lo) {
  if (!(__uint_as_float(v.x) < lo) | !(__uint_as_float(v.y) < lo) |
      !(__uint_as_float(v.z) < lo) | !(__uint_as_float(v.w) < lo))
    visit16(v, base, x, f);
}

// Every step-th round of the workgroup over a row, from the first on (a sample leaves the row's last
// partial piece out)
template <int U, typename LT, typename F, typename... G>
__device__ __forceinline__ void row_rounds(const LT* __restrict__ x, int V, int step, F&& f, G... floor) {
  constexpr int E = 16 / sizeof(LT);
  const int tid = threadIdx.x, nt = blockDim.x * step;
  int done = 0;
  if ((reinterpret_cast<uintptr_t>(x) & 15) == 0) {
    const int VE = V / E;
    const uint4* xe = reinterpret_cast<const uint4*>(x);
    uint4 a[U];
    int i = tid;
    for (; i + (U - 1) * nt < VE; i += U * nt) {
#pragma unroll
      for (int u = 0; u < U; ++u) a[u] = xe[i + u * nt];
#pragma unroll
      for (int u = 0; u < U; ++u) visit16(a[u], E * (i + u * nt), x, f, floor...);
    }
    if (i < VE) {
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (i + u * nt < VE) a[u] = xe[i + u * nt];
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (i + u * nt < VE) visit16(a[u], E * (i + u * nt), x, f, floor...);
    }
    done = VE * E;
    if (step > 1) return;
  }
  for (int j = done + tid; j < V; j += nt) f(ldv(x, j), j);
}
template <typename LT, typename F, typename... G>
__device__ __forceinline__ void row_scan(const LT* __restrict__ x, int V, F&& f, G... floor) {
  row_rounds<8>(x, V, 1, f, floor...);
}

// The same over n listed blocks of bw columns (a multiple of 4; V is one too), 4 quads in flight a thread
template <typename LT, typename F>
__device__ __forceinline__ void block_scan_quads(const LT* __restrict__ x, int V, const int* blk, int n,
                                                 int bw, F&& f, float lo) {
  constexpr int U = 4;
  const int q = bw >> 2, total = n * q;
  for (int t0 = threadIdx.x; t0 < total; t0 += U * blockDim.x) {
    float v[U][4];
    int at[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int t = t0 + u * blockDim.x, b = t < total ? t / q : 0;
      at[u] = t < total ? blk[b] * bw + (t - b * q) * 4 : V;
      if (at[u] < V) {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[u][j] = ldv(x, at[u] + j);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (at[u] < V) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (!(v[u][j] < lo)) f(v[u][j], at[u] + j);
      }
  }
}

// ---------------------------------------------------------------------------------------
// Small batches (B <= SMP_SPLIT_MAX_B): one workgroup per row leaves ~255 CUs idle while it
// walks a 128k-entry row (23 us at batch 1; two phases 18). Two phases
// instead: sample_chunk_kernel splits each row into P chunks (P workgroups per row); a chunk
// keeps every logit >= its own Keff-th largest (16 keys a thread in registers, the threshold by
// ballots as in sample_kernel), in index order, in a CAPC-slot candidate list (pads: -inf). The row's top-Keff is contained in the union of the
// chunks' lists, which keep index order, so sample_kernel then runs its unchanged algorithm
// over the P*CAPC candidates (ties still break on the lower vocab index) and maps the pick
// back to a vocab id. Rows whose Keff exceeds CAPC, plain-temperature rows and rows where a
// chunk had more than CAPC ties at its threshold (overflow flag) read the full row as before.
#define SMP_CAPC 64
#define SMP_CHUNK_MAX 4096
#define SMP_SPLIT_MAX_B 8                       // default largest two-phase batch
#define SMP_SPLIT_CAP_B 1024                    // largest batch dli_sample_set_split_max_b takes
static int g_smp_max_b = SMP_SPLIT_MAX_B;

__device__ __forceinline__ bool smp_split_ok(float T, int K, float P) {
  const bool greedy = T <= 0.f || K == 1;
  return greedy || (K >= 1 && K <= SMP_CAPC);      // K <= 0 means 'no top-k': whole row
}

template <typename LT>
__global__ void __launch_bounds__(256) sample_chunk_kernel(
    float* __restrict__ cand_v, int* __restrict__ cand_i, int* __restrict__ overflow,
    const LT* __restrict__ logits, long row_stride, int V, int L,
    const float* __restrict__ temperature, const int* __restrict__ top_k,
    const float* __restrict__ top_p) {
  constexpr int NE = SMP_CHUNK_MAX / 256, LIST = 512;
  __shared__ uint32_t lk[LIST], s_tau[4];
  __shared__ int li[LIST], s_cnt;
  const int row = blockIdx.y, c = blockIdx.x, tid = threadIdx.x, P = gridDim.x;
  const float T = temperature[row];
  const int K = top_k[row];
  if (!smp_split_ok(T, K, top_p[row])) return;        // sample_kernel reads the full row
  const int keff = (T <= 0.f || K == 1) ? 1 : K;
  const int lo = c * L, n = max(0, min(V, lo + L) - lo);
  const LT* x = logits + (long)row * row_stride + lo;
  uint32_t key[NE];
  uint32_t mk[1] = {0u};
#pragma unroll
  for (int j = 0; j < NE; ++j) {
    const int e = tid + 256 * j;
    key[j] = e < n ? f2key(ldv(x, e)) : 0u;
  }
#pragma unroll
  for (int j = 0; j < NE; ++j) mk[0] = max(mk[0], key[j]);
  // a lower bound of the chunk's keff-th largest key, as in sample_kernel: the least of the
  // ceil(keff / waves)-th largest per-thread maxima of the waves that have elements
  const int nw = max(1, min(4, (n + 63) >> 6));
  const uint32_t tw = wave_kth(mk, (keff + nw - 1) / nw);
  if ((tid & 63) == 0) s_tau[tid >> 6] = (tid >> 6) < nw ? tw : 0xffffffffu;
  if (tid == 0) s_cnt = 0;
  __syncthreads();
  const uint32_t tau0 = max(min(min(s_tau[0], s_tau[1]), min(s_tau[2], s_tau[3])), 1u);
#pragma unroll
  for (int j = 0; j < NE; ++j)
    if (key[j] >= tau0) {
      const int pos = atomicAdd(&s_cnt, 1);
      if (pos < LIST) { lk[pos] = key[j]; li[pos] = lo + tid + 256 * j; }
    }
  __syncthreads();
  const int nc = s_cnt;
  if (nc > LIST) {                                     // ties by the hundred: the row's full scan
    if (tid == 0) overflow[row] = 1;
    return;
  }
  if (tid >= 64) return;                               // one wave orders what is left
  uint32_t ck[LIST / 64];
  int ci[LIST / 64];
#pragma unroll
  for (int j = 0; j < LIST / 64; ++j) {
    const int e = j * 64 + tid;
    ck[j] = e < nc ? lk[e] : 0u;
    ci[j] = e < nc ? li[e] : 0;
  }
  // (fewer than keff entries: keep them all)
  const uint32_t tau = nc > keff ? wave_kth(ck, keff, tau0) : 1u;
  int m = 0;
  const unsigned long long below = (1ull << tid) - 1ull;
#pragma unroll
  for (int j = 0; j < LIST / 64; ++j) {
    const unsigned long long keep = __ballot(ck[j] >= tau);
    const int pos = m + __popcll(keep & below);
    if (ck[j] >= tau) { lk[pos] = ck[j]; li[pos] = ci[j]; }   // every entry is in registers
    m += __popcll(keep);
  }
  if (m > SMP_CAPC) {
    if (tid == 0) overflow[row] = 1;                   // the row falls back to the full scan
    return;
  }
  __builtin_amdgcn_wave_barrier();
  const long base = ((long)row * P + c) * SMP_CAPC;
  if (tid < m) {
    const int id = li[tid];
    int rank = 0;                                      // index order within the chunk
    for (int j = 0; j < m; ++j) rank += li[j] < id;
    cand_v[base + rank] = key2f(lk[tid]);
    cand_i[base + rank] = id;
  } else {
    cand_v[base + tid] = -INFINITY;
    cand_i[base + tid] = 0;
  }
}

template <typename LT>
__global__ void __launch_bounds__(SMP_THREADS) sample_kernel(
    int* __restrict__ out_tokens, const LT* __restrict__ logits, long row_stride, int V,
    const float* __restrict__ temperature, const int* __restrict__ top_k,
    const float* __restrict__ top_p, const long long* __restrict__ seeds,
    const float* __restrict__ cand_v, const int* __restrict__ cand_i,
    int* __restrict__ overflow, int ncand, const uint32_t* __restrict__ maxima, int nblk, int bw) {
  __shared__ uint32_t hist[256];
  __shared__ uint32_t ckey[2 * SMP_CAP];      // fast path: the list of candidates
  __shared__ int cidx[2 * SMP_CAP];
  __shared__ uint32_t skey[512];
  __shared__ int sidx[512];
  __shared__ __attribute__((aligned(8))) float cprob[SMP_CAP];
  __shared__ float sv[16];
  __shared__ int si[16];
  __shared__ uint32_t s_sel[3], s_tau[SMP_THREADS / 64], s_cnt;
  constexpr int BLKS = 512;                      // blocks of columns that a pass lists
  __shared__ int s_blk[BLKS], s_nblk;
  const int row = blockIdx.x, tid = threadIdx.x;
  // largest key of every block of bw columns (null: none were formed)
  const uint32_t* mx = maxima == nullptr ? nullptr : maxima + (long)row * nblk;
  const LT* xl = logits + (long)row * row_stride;
  const float* xc = nullptr;                     // two-phase mode: the row's candidate list
  const float T = temperature[row];
  const int K = top_k[row];
  const float P = top_p[row];
  const unsigned long long sd = (unsigned long long)seeds[row];
  const uint2 key = make_uint2((uint32_t)sd, (uint32_t)(sd >> 32));
  // two-phase small-batch mode: read the row's candidate list unless a chunk overflowed
  const int Vfull = V;
  const int* map = nullptr;
  if (cand_v != nullptr && smp_split_ok(T, K, P)) {
    if (overflow[row] == 0) {
      xc = cand_v + (long)row * ncand;
      map = cand_i + (long)row * ncand;
      V = ncand;
    }
    __syncthreads();                                          // every thread read the flag
    if (tid == 0) overflow[row] = 0;                          // zero for the next call
  }
  auto vocab_id = [&](int j) { return map != nullptr ? map[j] : j; };
  // every pass over the row: the candidate list (fp32) or the logits row (fp32 / bf16)
  auto scan = [&](auto&& f) {
    if (xc != nullptr) row_scan(xc, V, f);
    else row_scan(xl, V, f);
  };

  if (T <= 0.f || K == 1) {                                  // greedy
    ArgMax a{-INFINITY, 0x7fffffff};
    const auto larger = [&](float v, int i) { a = amax(a, ArgMax{v, i}); };
    if (mx != nullptr) {
      // the first block of the largest value, then its first element (a block with a NaN, which never
      // is the largest but whose key hides the others, sends the row to the whole scan)
      int odd = 0;
      for (int i = tid; i < nblk; i += SMP_THREADS) {
        const uint32_t k = mx[i];
        odd |= k > 0xff800000u;
        a = amax(a, ArgMax{key2f(k), i});
      }
      if (!__syncthreads_or(odd)) {
        a = block_argmax(a, sv, si);
        if (a.i < nblk) {
          const int lo = a.i * bw, hi = min(V, lo + bw);
          a = ArgMax{-INFINITY, 0x7fffffff};
          for (int i = lo + tid; i < hi; i += SMP_THREADS) a = amax(a, ArgMax{ldv(xl, i), i});
          __syncthreads();                         // sv / si are written again
          a = block_argmax(a, sv, si);
        }
        if (tid == 0) out_tokens[row] = a.i < V ? a.i : 0;
        return;
      }
      a = ArgMax{-INFINITY, 0x7fffffff};
    }
    // (fewer loads in flight where more rows than CUs are walked: 512 rows of 128k bf16 logits 24 us, 27)
    if (xc != nullptr) row_scan(xc, V, larger);
    else if (sizeof(LT) == 2 || gridDim.x > 128) row_rounds<4>(xl, V, 1, larger);
    else row_scan(xl, V, larger);
    a = block_argmax(a, sv, si);
    if (tid == 0) out_tokens[row] = a.i < V ? vocab_id(a.i) : 0;
    return;
  }
  const float invT = 1.f / T;
  if (K <= 0 && P >= 1.f) {                                  // plain temperature: Gumbel-max
    ArgMax a{-INFINITY, 0x7fffffff};
    for (int base = tid * 4; base < V; base += blockDim.x * 4) {
      const uint4 r = philox(key, make_uint4((uint32_t)(base >> 2), 0u, 0x5a5a5a5au, 0u));
      const uint32_t rr[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = base + j;
        if (i < V) {
          const float g = -__logf(-__logf(u01(rr[j])));
          a = amax(a, ArgMax{(xc != nullptr ? xc[i] : ldv(xl, i)) * invT + g, i});
        }
      }
    }
    a = block_argmax(a, sv, si);
    if (tid == 0) out_tokens[row] = a.i < V ? a.i : 0;
    return;
  }
  int Keff = (K <= 0 || K > SMP_CAP) ? SMP_CAP : K;
  if (Keff > Vfull) Keff = Vfull;

  int n = 0;
  bool fast_ok = false, sorted = false;
  // ---- fast path, no full-row select:
  //  (1) tau0: each of the 8 waves takes the ceil(Keff / 8)-th largest of its 64 per-thread
  //      maxima over a sample of the row (fewer waves on a short row); the least of them,
  //      brought nearer to the Keff-th largest of all 512 by a few steps, is tau0. At least Keff elements are >= tau0, so
  //      tau0 <= the row's Keff-th largest. (Without the steps the list runs to 300 - 600.)
  //      The sample is spread over the row, which may rise or fall with the index, and larger for
  //      a larger Keff: the list takes -512 ln(1 - Keff / 512) times the row's part in it elements,
  //      211 for 50 of a quarter, 295 for 128 and 507 for 200 of a half, 355 for 256 of all; a quarter
  //      would take 1014 for 200, and some thread more than its slots.
  //  (2) one pass over the row; each thread keeps the elements >= tau0 it meets, a few hundred
  //      of 128k over all, in 8 slots of its own in LDS (a shared counter would cost a round trip
  //      per element). Where a thread needs more (many ties, a row with its large elements in one
  //      thread's columns) the Keff-th largest of what was kept is a nearer bound for a second pass;
  //      a row that needs more again goes through the full radix select.
  //  (3) the list's Keff-th largest key is the row's; what reaches it is ranked by counting.
  // 24 rows of 32k / 128k logits, top-k 50: 32 / 42 us with the 512 maxima and the list's 4096 slots
  // selected by histograms and a bitonic sort of the rest -> 16 / 25.
  if (Keff <= 256) {
    uint32_t mk = 0u;
    int step = Keff <= 64 ? 4 : Keff <= 208 ? 2 : 1;
    // (a short row whole: every thread needs elements)
    while (step > 1 && V < step * 16 * SMP_THREADS) step >>= 1;
    int pieces;                                   // of a first round over the row
    const auto sample = [&](auto* x) {
      row_rounds<8>(x, V, step, [&](float v, int) { mk = max(mk, f2key(v)); });
      pieces = (reinterpret_cast<uintptr_t>(x) & 15) ? V : V / (int)(16 / sizeof(*x));
    };
    const bool by_block = mx != nullptr && nblk >= 4 * Keff;   // (fewer blocks bound too loosely)
    if (by_block) {
      pieces = nblk;
#pragma unroll 4
      for (int i = tid; i < nblk; i += SMP_THREADS) mk = max(mk, mx[i]);
    } else if (xc != nullptr) sample(xc);
    else sample(xl);
    constexpr int NWV = SMP_THREADS / 64, SLOTS = 2 * SMP_CAP / SMP_THREADS;
    const uint32_t mk1[1] = {mk};
    // waves that met elements; of a few hundred blocks only whole ones (the 8th largest of a last wave's
    // 16 bounds too loosely: 256 rows of 400 blocks 30 us, so 18)
    const int nw = max(1, min(NWV, by_block ? pieces >> 6 : (pieces + 63) >> 6));
    const uint32_t tw = wave_kth(mk1, (Keff + nw - 1) / nw);
    if ((tid & 63) == 0) s_tau[tid >> 6] = (tid >> 6) < nw ? tw : 0xffffffffu;
    if (tid == 0) s_cnt = 0;
    skey[tid] = mk;
    __syncthreads();
    uint32_t tau0 = s_tau[0];
#pragma unroll
    for (int w = 1; w < NWV; ++w) tau0 = min(tau0, s_tau[w]);
    if (xc == nullptr) {                          // (a candidate list is short enough)
      uint32_t ck[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) ck[j] = skey[j * 64 + (tid & 63)];
      tau0 = max(tau0, wave_kth(ck, Keff, tau0, 7));
    }
    tau0 = max(tau0, 1u);                         // key 0 is no element
    int cnt;
    auto hit = [&](float v, int i) {
      const uint32_t k = f2key(v);
      if (k >= tau0) {
        if (cnt < SLOTS) {                        // thread-strided slots: no bank conflicts
          ckey[tid + SMP_THREADS * cnt] = k;
          cidx[tid + SMP_THREADS * cnt] = i;
        }
        ++cnt;
      }
    };
    uint32_t at, nc;
    int dropped;
    for (bool again = false;; again = true) {
      // !(v < tf) is true of every element with a key >= tau0 (and of NaNs and zeros below it): one
      // compare an element, the keys only where one of 16 bytes passes
      const float tf = key2f(tau0);
      cnt = 0;
      bool listed = by_block;
      if (by_block) {
        if (tid == 0) s_nblk = 0;
        __syncthreads();
#pragma unroll 4
        for (int i = tid; i < nblk; i += SMP_THREADS)
          if (mx[i] >= tau0) {
            const int pos = atomicAdd(&s_nblk, 1);
            if (pos < BLKS) s_blk[pos] = i;
          }
        __syncthreads();
        listed = s_nblk <= BLKS;                  // else ties by the hundred: the whole row
        if (listed) block_scan_quads(xl, V, s_blk, s_nblk, bw, hit, tf);
      }
      if (listed) {
      } else if (xc != nullptr) row_scan(xc, V, hit, tf);
      else row_scan(xl, V, hit, tf);
      at = cnt ? atomicAdd(&s_cnt, (uint32_t)cnt) : 0u;
      dropped = __syncthreads_or(cnt > SLOTS ? 1 : 0);
      nc = s_cnt;
      if (!dropped || again) break;
      for (int j = cnt; j < SLOTS; ++j) ckey[tid + SMP_THREADS * j] = 0u;
      __syncthreads();
      const uint32_t t = radix_kth(ckey, SLOTS * SMP_THREADS, (uint32_t)Keff, hist, sv, s_sel);
      if (t <= tau0) break;                       // (0: fewer than Keff were kept)
      __syncthreads();
      tau0 = t;
      if (tid == 0) s_cnt = 0;
      __syncthreads();
    }
    if (!dropped && nc >= (uint32_t)Keff) {
      if (nc <= 512) {
        for (int j = 0; j < cnt; ++j) {
          skey[at + j] = ckey[tid + SMP_THREADS * j];
          sidx[at + j] = cidx[tid + SMP_THREADS * j];
        }
      } else {
        for (int j = cnt; j < SLOTS; ++j) ckey[tid + SMP_THREADS * j] = 0u;
      }
      __syncthreads();
      if (nc <= 512) {
        // every wave holds the whole list and finds the threshold for itself; the first packs
        // and ranks what reaches it
        uint32_t ck[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const uint32_t e = j * 64 + (tid & 63);
          ck[j] = e < nc ? skey[e] : 0u;
        }
        const uint32_t(&half)[4] = *reinterpret_cast<const uint32_t(*)[4]>(ck);
        const uint32_t tau = nc <= 256 ? wave_kth(half, Keff, tau0) : wave_kth(ck, Keff, tau0);
#pragma unroll
        for (int j = 0; j < 8; ++j) n += __popcll(__ballot(ck[j] >= tau));
        sorted = n <= SMP_RANK_MAX;
        unsigned long long* both = reinterpret_cast<unsigned long long*>(cprob);
        if (tid < 64) {
          int m = 0;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const unsigned long long keep = __ballot(ck[j] >= tau);
            if (ck[j] >= tau) {
              const int pos = m + __popcll(keep & ((1ull << tid) - 1ull));
              const int id = sidx[j * 64 + tid];
              if (sorted) {
                both[pos] = (unsigned long long)ck[j] << 32 | (uint32_t)~id;
              } else {
                ckey[pos] = ck[j];
                cidx[pos] = id;
              }
            }
            m += __popcll(keep);
          }
          __builtin_amdgcn_wave_barrier();
          if (sorted) {
            for (int e = tid; e < n; e += 64) {
              const unsigned long long own = both[e];   // larger key first, then smaller index
              int rank = 0;
#pragma unroll 8
              for (int j = 0; j < n; ++j) rank += both[j] > own;
              ckey[rank] = (uint32_t)(own >> 32);
              cidx[rank] = ~(int)(uint32_t)own;
            }
          }
        }
        fast_ok = true;
      } else {
        const uint32_t tau = radix_kth(ckey, SLOTS * SMP_THREADS, (uint32_t)Keff, hist, sv, s_sel);
        if (tid == 0) s_cnt = 0;
        __syncthreads();
        for (int e = tid; e < SLOTS * SMP_THREADS; e += blockDim.x) {
          if (ckey[e] >= tau) {
            const uint32_t pos = atomicAdd(&s_cnt, 1u);
            if (pos < 512) { skey[pos] = ckey[e]; sidx[pos] = cidx[e]; }
          }
        }
        __syncthreads();
        fast_ok = s_cnt <= 512;                   // absurd tie count: take the slow path
        if (fast_ok) {
          n = (int)s_cnt;
          for (int e = tid; e < n; e += blockDim.x) { ckey[e] = skey[e]; cidx[e] = sidx[e]; }
        }
      }
      __syncthreads();
    }
  }
  if (!fast_ok) {
  // ---- radix select on order-preserving keys (largest first), 8-bit digits
  uint32_t prefix = 0, pmask = 0, k_rem = (uint32_t)Keff, above_total = 0;
  for (int pass = 0; pass < 4; ++pass) {
    const int shift = 24 - 8 * pass;
    for (int i = tid; i < 256; i += blockDim.x) hist[i] = 0;
    __syncthreads();
    scan([&](float v, int) {
      const uint32_t k = f2key(v);
      if ((k & pmask) == prefix) atomicAdd(&hist[(k >> shift) & 255u], 1u);
    });
    __syncthreads();
    find_digit(hist, k_rem, sv, s_sel);
    __syncthreads();
    k_rem -= s_sel[1];
    above_total += s_sel[1];
    prefix |= s_sel[0] << shift;
    pmask |= 255u << shift;
    if (above_total + s_sel[2] <= SMP_CAP) break;
  }
  // ---- gather everything at or above the boundary bin. When that is more than SMP_CAP
  // (the 4 passes ran out: prefix is the exact CAP-th key, and its ties overflow), keep every
  // key strictly above it and the lowest-index ties: a deterministic set, whatever the order
  // of the atomics below (bf16 logits tie often)
  const bool overflow_ties = above_total + s_sel[2] > SMP_CAP;
  if (tid == 0) s_cnt = 0;
  __syncthreads();
  scan([&](float v, int i) {
    const uint32_t k = f2key(v);
    if (overflow_ties ? k > prefix : (k & pmask) >= prefix) {
      const uint32_t pos = atomicAdd(&s_cnt, 1u);
      if (pos < SMP_CAP) { ckey[pos] = k; cidx[pos] = i; }
    }
  });
  __syncthreads();
  n = (int)min(s_cnt, (uint32_t)SMP_CAP);
  if (overflow_ties) {
    // ordered compaction of the ties over contiguous per-thread slices of the row
    const uint32_t need = (uint32_t)SMP_CAP - (uint32_t)n;
    const int per = (V + SMP_THREADS - 1) / SMP_THREADS;
    const int lo = min(V, tid * per), hi = min(V, lo + per);
    auto val = [&](int e) { return xc != nullptr ? xc[e] : ldv(xl, e); };
    uint32_t n_eq = 0;
    for (int e = lo; e < hi; ++e) n_eq += f2key(val(e)) == prefix;
    __syncthreads();                              // sv reuse by block_scan
    uint32_t before = (uint32_t)block_scan((float)n_eq, sv) - n_eq;   // exact: < 2^24
    for (int e = lo; e < hi && before < need; ++e) {
      if (f2key(val(e)) == prefix) {
        ckey[n + before] = prefix;
        cidx[n + before] = e;
        ++before;
      }
    }
    __syncthreads();
    n = SMP_CAP;
  }
  }
  int npow = 1;
  if (!sorted) {
    while (npow < n) npow <<= 1;
    for (int i = n + tid; i < npow; i += blockDim.x) { ckey[i] = 0u; cidx[i] = 0x7fffffff; }
    __syncthreads();
  }
  // ---- bitonic sort descending by key (ties: smaller index first)
  for (int size = 2; size <= npow; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int i = tid; i < npow / 2; i += blockDim.x) {
        const int lo = 2 * i - (i & (stride - 1));
        const int hi = lo + stride;
        const bool desc = ((lo & size) == 0);
        const uint32_t a = ckey[lo], b = ckey[hi];
        const int ia = cidx[lo], ib = cidx[hi];
        const bool a_first = (a > b) || (a == b && ia < ib);
        if (a_first != desc) {
          ckey[lo] = b; ckey[hi] = a; cidx[lo] = ib; cidx[hi] = ia;
        }
      }
      __syncthreads();
    }
  }
  // ---- top-k cut (ties with the k-th value kept)
  const int kk = min(Keff, n);
  const uint32_t tau = ckey[kk - 1];
  int m = kk;
  while (m < n && ckey[m] == tau) ++m;
  if (m <= 256) {
    // the first wave's entries are all there are: the sums below in the same order, in its
    // registers, and no barriers (7k -> 2k cycles)
    if (tid >= 64) return;
    const float xm = key2f(ckey[0]);
    float cp[4], ls = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int e = tid * 4 + j;
      cp[j] = e < m ? __expf((key2f(ckey[e]) - xm) * invT) : 0.f;
      ls += cp[j];
    }
    float inc = ls;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const float t = __shfl_up(inc, o, 64);
      if (tid >= o) inc += t;
    }
    float run = inc - ls;
#pragma unroll
    for (int j = 0; j < 4; ++j) { run += cp[j]; cp[j] = run; }
    auto at = [&](int e) {                        // e is the same in every lane
      const float v = (e & 2) ? ((e & 1) ? cp[3] : cp[2]) : ((e & 1) ? cp[1] : cp[0]);
      return __shfl(v, e >> 2, 64);
    };
    auto first = [&](int end, auto&& pass) {      // first e < end that passes, else end
      int e = end;
#pragma unroll
      for (int j = 3; j >= 0; --j)
        if (tid * 4 + j < end && pass(cp[j])) e = tid * 4 + j;
      const unsigned long long any = __ballot(e < end);
      return any ? __shfl(e, __ffsll(any) - 1, 64) : end;
    };
    const float lim = P * at(m - 1);
    const int c = first(m - 1, [&](float v) { return v >= lim; }) + 1;
    const uint4 r = philox(key, make_uint4(0xfffffffu, 1u, 0xa5a5a5a5u, 7u));
    const float u = u01(r.x) * at(c - 1);
    const int pick = first(c - 1, [&](float v) { return v > u; });
    if (tid == 0) out_tokens[row] = vocab_id(cidx[pick]);
    return;
  }
  // ---- temperature softmax over the m survivors, top-p, inverse CDF
  const float xmax = key2f(ckey[0]);
  constexpr int PER = SMP_CAP / SMP_THREADS;                 // 4 consecutive entries / thread
  float loc[PER], lsum = 0.f;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int e = tid * PER + j;
    loc[j] = e < m ? __expf((key2f(ckey[e]) - xmax) * invT) : 0.f;
    lsum += loc[j];
  }
  const float incl = block_scan(lsum, sv);
  float run = incl - lsum;
#pragma unroll
  for (int j = 0; j < PER; ++j) { run += loc[j]; cprob[tid * PER + j] = run; }
  __syncthreads();
  const float Z = cprob[m - 1];
  // keep entries whose exclusive prefix < P * Z: c = 1 + (first j < m-1 with cprob[j] >= lim,
  // else m-1); then the draw j = first j < c-1 with cprob[j] > u, else c-1. Both "first
  // index" searches run over all threads with an LDS atomicMin (was one thread's serial walk)
  const float lim = P * Z;
  if (tid == 0) s_cnt = (uint32_t)(m - 1);
  __syncthreads();
  for (int e = tid; e < m - 1; e += blockDim.x)
    if (cprob[e] >= lim) atomicMin(&s_cnt, (uint32_t)e);
  __syncthreads();
  const int c = (int)s_cnt + 1;
  const float zk = cprob[c - 1];
  const uint4 r = philox(key, make_uint4(0xfffffffu, 1u, 0xa5a5a5a5u, 7u));
  const float u = u01(r.x) * zk;
  __syncthreads();                                // s_cnt read by every thread
  if (tid == 0) s_cnt = (uint32_t)(c - 1);
  __syncthreads();
  for (int e = tid; e < c - 1; e += blockDim.x)
    if (cprob[e] > u) atomicMin(&s_cnt, (uint32_t)e);
  __syncthreads();
  if (tid == 0) out_tokens[row] = vocab_id(cidx[s_cnt]);
}

// Bytes of the two-phase workspace dli_sample takes for a batch of B rows (0: one phase).
extern "C" long dli_sample_workspace_bytes(int B, int V) {
  if (B <= 0 || B > g_smp_max_b) return 0;
  return (long)g_smp_max_b * 4 + (long)B * 64 * SMP_CAPC * 8;
}

// Largest batch that samples in two phases (default SMP_SPLIT_MAX_B = 8; A/B runs raise it:
// the workspace layout follows it, so set it before the first workspace is sized). Returns
// the previous value.
extern "C" int dli_sample_set_split_max_b(int b) {
  const int old = g_smp_max_b;
  if (b >= 1 && b <= SMP_SPLIT_CAP_B) g_smp_max_b = b;
  return old;
}

// ws: nullable; when given (>= dli_sample_workspace_bytes, its first g_smp_max_b ints
// zero before the first call — the kernels leave them zero), batches of B <= 8 rows sample in
// two phases (above).
template <typename LT>
static int launch_sample(int* out_tokens, const LT* logits, long row_stride, int B, int V,
                         const float* temperature, const int* top_k, const float* top_p,
                         const long long* seeds, void* ws, const uint32_t* maxima, int nblk,
                         int bw, hipStream_t st) {
  if (B <= 0) return 0;
  if (maxima != nullptr && (bw < 4 || bw % 4 || V % 4 || (long)nblk != ((long)V + bw - 1) / bw))
    return (int)hipErrorInvalidValue;
  if (maxima == nullptr && ws != nullptr && B <= g_smp_max_b) {
    // P chunks per row: >= 256 workgroups in all, each chunk <= SMP_CHUNK_MAX entries
    int P = 1;
    while (P < 64 && (B * P < 256 || (V + P - 1) / P > SMP_CHUNK_MAX)) P <<= 1;
    const int L = (((V + P - 1) / P) + 3) & ~3;
    if (L <= SMP_CHUNK_MAX) {
      int* overflow = static_cast<int*>(ws);
      float* cand_v = reinterpret_cast<float*>(overflow + g_smp_max_b);
      int* cand_i = reinterpret_cast<int*>(cand_v + (long)B * 64 * SMP_CAPC);
      sample_chunk_kernel<LT><<<dim3(P, B), 256, 0, st>>>(cand_v, cand_i, overflow, logits,
                                                          row_stride, V, L, temperature, top_k,
                                                          top_p);
      sample_kernel<LT><<<B, SMP_THREADS, 0, st>>>(out_tokens, logits, row_stride, V,
                                                  temperature, top_k, top_p, seeds, cand_v,
                                                  cand_i, overflow, P * SMP_CAPC, nullptr, 0, 0);
      DLI_RETURN_LAUNCH();
    }
  }
  sample_kernel<LT><<<B, SMP_THREADS, 0, st>>>(out_tokens, logits, row_stride, V, temperature,
                                              top_k, top_p, seeds, nullptr, nullptr, nullptr, 0, maxima,
                                              nblk, bw);
  DLI_RETURN_LAUNCH();
}

extern "C" int dli_sample(int* out_tokens, const float* logits, long row_stride, int B, int V,
                          const float* temperature, const int* top_k, const float* top_p,
                          const long long* seeds, void* ws, hipStream_t st) {
  return launch_sample(out_tokens, logits, row_stride, B, V, temperature, top_k, top_p, seeds,
                       ws, nullptr, 0, 0, st);
}

// the same with maxima uint32 [B, nblk]: the largest key of every bw columns of these logits, as
// dli_gemm_head leaves them
extern "C" int dli_sample_blocks(int* out_tokens, const float* logits, long row_stride, int B, int V,
                                 const float* temperature, const int* top_k, const float* top_p,
                                 const long long* seeds, const void* maxima, int nblk, int bw,
                                 hipStream_t st) {
  if (maxima == nullptr) return (int)hipErrorInvalidValue;
  return launch_sample(out_tokens, logits, row_stride, B, V, temperature, top_k, top_p, seeds,
                       nullptr, static_cast<const uint32_t*>(maxima), nblk, bw, st);
}

// the same over bf16 logits (row_stride in elements)
extern "C" int dli_sample_bf16(int* out_tokens, const void* logits, long row_stride, int B,
                               int V, const float* temperature, const int* top_k,
                               const float* top_p, const long long* seeds, void* ws,
                               hipStream_t st) {
  return launch_sample(out_tokens, static_cast<const u16*>(logits), row_stride, B, V,
                       temperature, top_k, top_p, seeds, ws, nullptr, 0, 0, st);
}

// ---------------------------------------------------------------------------------------
// Per-row top-c of fp32 logits (the vocab-parallel LM head's candidates,
// parallel/pipeline.py): one 512-thread workgroup per row.
//   1. radix select over the row in global memory (4 passes of 8-bit digits on order-
//      preserving keys): tau = key of the c-th largest element, n_gt = count above tau;
//   2. ordered compaction: thread t owns a contiguous slice of the row, so a block scan of
//      per-thread counts writes the winners (every key > tau, then the first c - n_gt keys
//      == tau in index order) already in ascending index order — the order the candidate
//      merge on rank 0 requires (ranks concatenate ascending vocab slices).
// Replaces torch.topk + torch.sort + gather on the pipeline's hot path.
template <typename T>
__global__ void __launch_bounds__(SMP_THREADS) topk_rows_kernel(
    float* __restrict__ out_v, int* __restrict__ out_i, const T* __restrict__ x,
    long row_stride, int V, int c, int id_offset) {
  __shared__ uint32_t hist[256];
  __shared__ float sv[16];
  __shared__ uint32_t s_sel[3];
  const int row = blockIdx.x, tid = threadIdx.x;
  const T* xr = x + (long)row * row_stride;
  uint32_t prefix = 0, pmask = 0, k_rem = (uint32_t)c;
  for (int pass = 0; pass < 4; ++pass) {
    const int shift = 24 - 8 * pass;
    for (int i = tid; i < 256; i += blockDim.x) hist[i] = 0;
    __syncthreads();
    row_scan(xr, V, [&](float v, int) {
      const uint32_t k = f2key(v);
      if ((k & pmask) == prefix) atomicAdd(&hist[(k >> shift) & 255u], 1u);
    });
    __syncthreads();
    find_digit(hist, k_rem, sv, s_sel);
    __syncthreads();
    k_rem -= s_sel[1];
    prefix |= s_sel[0] << shift;
    pmask |= 255u << shift;
    __syncthreads();
  }
  const uint32_t tau = prefix;                 // c-th largest key; k_rem of its ties are taken
  // ---- ordered compaction over contiguous per-thread slices
  const int per = (V + SMP_THREADS - 1) / SMP_THREADS;
  const int lo = min(V, tid * per), hi = min(V, lo + per);
  uint32_t n_gt = 0, n_eq = 0;
  for (int e = lo; e < hi; ++e) {
    const uint32_t k = f2key(ldv(xr, e));
    n_gt += k > tau;
    n_eq += k == tau;
  }
  const float gt_incl = block_scan((float)n_gt, sv);        // exact: counts < 2^24
  __syncthreads();
  const float eq_incl = block_scan((float)n_eq, sv);
  uint32_t eq_before = (uint32_t)eq_incl - n_eq;            // ties in earlier slices
  uint32_t before = (uint32_t)gt_incl - n_gt + min(eq_before, k_rem);
  for (int e = lo; e < hi && before < (uint32_t)c; ++e) {
    const float v = ldv(xr, e);
    const uint32_t k = f2key(v);
    bool take = k > tau;
    if (k == tau) { take = eq_before < k_rem; ++eq_before; }
    if (take) {
      out_v[(long)row * c + before] = v;
      out_i[(long)row * c + before] = e + id_offset;
      ++before;
    }
  }
}

extern "C" int dli_topk_rows(float* out_v, int* out_i, const float* x, long row_stride, int rows,
                             int V, int c, int id_offset, hipStream_t st) {
  if (rows <= 0) return 0;
  if (c < 1 || c > V || V > (1 << 24)) return (int)hipErrorInvalidValue;
  topk_rows_kernel<float><<<rows, SMP_THREADS, 0, st>>>(out_v, out_i, x, row_stride, V, c,
                                                         id_offset);
  DLI_RETURN_LAUNCH();
}

extern "C" int dli_topk_rows_bf16(float* out_v, int* out_i, const void* x, long row_stride,
                                  int rows, int V, int c, int id_offset, hipStream_t st) {
  if (rows <= 0) return 0;
  if (c < 1 || c > V || V > (1 << 24)) return (int)hipErrorInvalidValue;
  topk_rows_kernel<u16><<<rows, SMP_THREADS, 0, st>>>(out_v, out_i, static_cast<const u16*>(x),
                                                       row_stride, V, c, id_offset);
  DLI_RETURN_LAUNCH();
}
