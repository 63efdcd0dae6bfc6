// Portions of the linear recurrences, 16 tokens at a time on the fp32 matrix cores:
//     S_t = diag(a_t) S_{t-1} + k_t v_t^T,      o_t = S_t^T q_t        S [d, dv] per head, fp32
// with the decay a_t
//   HGRN2  a number per channel, lower + (1 - lower) sigmoid(fz_t + bias); k_t = 1 - a_t, q = silu(qz)
//   GLA    a number per channel, sigmoid(z_t + bias)^(1/tau); q times qscale
//   FIXED  one number per head; SiLU on q, k and v
//   MLSTM  a number per head and token, exp(f_t + m_{t-1} - m_t), m_t = max(f_t + m_{t-1}, i_t), with
//          b_t = exp(i_t - m_t) on k_t, a normaliser vector n_t beside S_t and q times d^(-1/2)
// (recurrent.hip and recurrent_scalar.hip state the four in full and hold the decode steps and the
// token-by-token walk for the sizes that this form does not take).
//
// With A_i = prod_{t <= i} a_t, B_j = prod_{t > j} a_t and G = prod a_t over a block of 16 tokens
//     o_i = (A_i q_i)^T S + sum_{j <= i} P_ij v_j,   P_ij = sum_c q_ic k_jc prod_{j < t <= i} a_tc
//     S  <- diag(G) S + sum_j (B_j k_j) v_j^T
// are four products of v_mfma_f32_16x16x4_f32. A block's 72 MFMAs of 32 cycles a wave at d = 128 are its
// floor (1.9 us with two waves a SIMD); it takes 4 to 6 us, the rest being the gates and the LDS image.
// The walk's floor is one token after another: 0.5 to 1.2 us each.
//
// A workgroup fills a CU, and there are as many as heads times sequences. Where that leaves CUs idle the
// portions are cut in segments: a first launch forms each segment's state from nothing (no read-outs:
// less than half the work), the second starts every segment from the fold of the states before it.
//
// d = dv = 128, HGRN2 / GLA / FIXED of 32 heads / MLSTM of 16, us; the walk, whole portions (before LONG), and what runs:
//   4 x 2048 tokens     1667  2342   976  1938     621   704   517   895     386   424   346   241
//   998 to 2601 (5)                                768   891   650  1133     461   503   410   305
//   1 x 8000                                      2325  2688  1972  3441     384   421   345   274
//   32 x 256 (not cut)   680   824   508   423     354   397   295   240     307   332   258   183
//
// One workgroup of 8 waves per (head, sequence, 128 state columns); a wave owns 16 columns and all d
// rows of S in its accumulators for the whole portion. The summation index of an MFMA may be permuted
// as long as both operands agree: register r of an accumulator tile holds rows 4 q + r (q = lane / 16),
// so it is, as it stands, the second operand of the read-out's MFMA over channels {4 q + r}, and the
// first operand is a 16-byte LDS read. P^T = K Q^T leaves P in the layout of the first operand of P V
// likewise. So neither S nor P is ever re-laid through LDS; only P's partial sums are (every wave
// takes 16 channels of P).
//
// Per-channel decays: P's terms factor as (A_i q_i) (k_j / A_j). Where a channel's decay over the block
// is below MIN_DECAY the quotient could overflow; such a channel is left out of the product and its 136
// terms are formed by multiplying the decays in between, as the walk does. Per-token decays scale the
// raw products k_j . q_i instead, by products of the decays in between.
//
// One barrier a block. Between two of them a wave stages block b + 1 (the LDS images are double
// buffered), requests the rows of block b + 2, runs block b's products, finishes block b - 1 (sums P,
// adds P V, squares for the norm), writes block b - 2 and forms the gates of block b + 2; half of the
// waves run the products before the finishing, half after it, so that a SIMD's two waves keep the
// matrix pipe and the vector unit busy at the same time (per-channel decays: the former ahead of the staging too).
//
// A step of the loop was up to 93 basic blocks (a bound a token, a head's widths) and waited for LDS at each of 8
// tiles' operands. LONG takes the steps whose blocks are full, of heads of 128 channels and columns, through a copy
// without bounds, with scalar row addresses; the next tile's operands are read ahead of a tile's products; with
// per-channel decays the wave that has products to issue goes first (the others lose 1 to 2 % by it). 4 x 2048 tokens
// without and with it, one card: HGRN2 441 / 382 us, GLA 501 / 424, FIXED 396 / 345, MLSTM 326 / 294. Equal to the bit.
#include "common.h"

namespace {

template <typename S> __device__ __forceinline__ float ldf(const S* p);
template <> __device__ __forceinline__ float ldf<u16>(const u16* p) { return bf2f(*p); }
template <> __device__ __forceinline__ float ldf<float>(const float* p) { return *p; }
template <typename S> __device__ __forceinline__ void stf(S* p, float v);
template <> __device__ __forceinline__ void stf<u16>(u16* p, float v) { *p = f2bf(v); }
template <> __device__ __forceinline__ void stf<float>(float* p, float v) { *p = v; }

// exp, reciprocal and sigmoid to about an ulp in a few instructions: 2^(x log2 e) with the product's
// rounding carried to first order, and one Newton step. Infinities saturate, NaN stays.
__device__ __forceinline__ float exp1(float x) {
  x = __builtin_elementwise_maximum(__builtin_elementwise_minimum(x, 88.f), -104.f);
  const float hi = x * 0x1.715476p+0f;
  const float lo = fmaf(x, 0x1.4ae0bfp-26f, fmaf(x, 0x1.715476p+0f, -hi));
  const float r = __builtin_amdgcn_exp2f(hi);
  return fmaf(r, lo * 0x1.62e430p-1f, r);
}
__device__ __forceinline__ float rcp1(float x) {                  // 0 < |x| < 2^126
  const float r = __builtin_amdgcn_rcpf(x);
  return fmaf(fmaf(-x, r, 1.f), r, r);
}
__device__ __forceinline__ float sigmoid1(float x) { return rcp1(1.f + exp1(-x)); }
__device__ __forceinline__ float silu1(float x) { return x * sigmoid1(x); }
// sigmoid(x)^(inv_tau); below -16 the sigmoid is e^x to fp32's precision. A slow channel remembers
// thousands of tokens, so its decay is rounded only once: 1 + y P(y) for 2^y near one.
__device__ __forceinline__ float decay_pow(float x, float inv_tau) {
  const float lg = x < -16.f ? x * 0x1.715476p+0f : __builtin_amdgcn_logf(sigmoid1(x));
  const float y = lg * inv_tau;
  float p = fmaf(y, 0x1.430912p-13f, 0x1.5d87fep-10f);            // ln2^k / k!, k = 6 .. 1
  p = fmaf(y, p, 0x1.3b2ab6p-7f);
  p = fmaf(y, p, 0x1.c6b08ep-5f);
  p = fmaf(y, p, 0x1.ebfbe0p-3f);
  p = fmaf(y, p, 0x1.62e430p-1f);
  return y > -0.25f ? fmaf(y, p, 1.f) : __builtin_amdgcn_exp2f(y);
}
__device__ __forceinline__ float logsigmoid32(float x) {          // stable on both sides
  return x > 0.f ? -log1pf(expf(-x)) : x - log1pf(expf(x));
}
__device__ __forceinline__ float from_lane(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
// LDS writes of all waves before it are visible after it; global loads and stores stay in flight
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
// lane i of a row of 16 takes lane i - n (CTRL 0x110 + n), i + n (0x100 + n) or (i + n) mod 16 (0x120 +
// 16 - n); lanes without a source take `other`
template <int CTRL> __device__ __forceinline__ float row(float other, float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(other), __float_as_int(v), CTRL, 0xf,
                                                    0xf, false));
}
__device__ __forceinline__ float row_sum(float v) {
  v += row<0x128>(0.f, v);
  v += row<0x124>(0.f, v);
  v += row<0x122>(0.f, v);
  return v + row<0x121>(0.f, v);
}
__device__ __forceinline__ f32x4 mfma4(const f32x4 a, const f32x4 b, f32x4 c) {
#pragma unroll
  for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], c, 0, 0, 0);
  return c;
}

enum { HGRN2 = 0, GLA = 1, FIXED = 2, MLSTM = 3 };
constexpr int TB = 16;              // tokens a block
constexpr int COLS = 128;           // state columns of a workgroup
constexpr int NTH = 512;
constexpr int LT = TB + 4;          // stride of the token-minor images
constexpr float MIN_DECAY = 1e-25f;

struct ChunkArgs {
  const float* proj; int ldp;
  const float* z; int ldz;                      // GLA
  const void* bias; const void* lower;          // [H*d] (HGRN2: both, GLA: bias)
  float inv_tau, qscale;
  const float* decays;                          // [H] (FIXED)
  const float* if_b; float cap;                 // [2H] (MLSTM)
  const void* norm_w; float eps;                // [dv] (HGRN2, GLA) or [H*dv] (MLSTM)
  float* state; float* nstate;
  const int* slots; const int* cu; const int* positions;
  void* out; int ldo; float out_scale;
  int H, d, dv;
  int min_len;                                  // sequences that bring fewer tokens are left alone
  const float* gates;                           // MLSTM: [T][H][4] = a, b, exp(-m)
  // nseg > 1: the portions are cut in segments of seg_tokens, (sequence s, segment k, head h) being
  // unit (s nseg + k) H + h of: the state after a segment, from nothing (from the portion's start for
  // k = 0); its decay (a number a channel, or the first); its normaliser (MLSTM). Segment nseg - 1
  // has no successor: its unit keeps the portion's first state.
  int seg_tokens, nseg;
  float* seg_state; float* seg_decay; float* seg_n;
};
constexpr int UNIT = 128;                       // floats of seg_decay and seg_n a unit

// scalar decays of a block: A_i, b_j B_j, exp(-m_i), G, and D_ij = b_j prod_{j < t <= i} a_t
struct Gates { float A[TB], kb[TB], em[TB], G[4], D[TB * LT]; };   // G as a sum of two floats

// STATE: the image of a launch that forms the segments' states only
template <int ND, bool STATE> struct Smem {
  static constexpr int DP = ND * 16, LQ = DP + 8;
  float Kb[2][DP * LT];             // B_j k_j, channel-major
  float V[2][COLS * LT];            // v, column-major
  float Q[2][STATE ? 4 : TB * LQ];  // q (per-channel decays: A_i q_i), token-major
  float K[2][STATE ? 4 : TB * LQ];  // k (per-channel decays: k_j / A_j), token-major
  float P[2][ND][STATE ? 4 : 256];  // partial sums of P^T, an accumulator a lane
  float ss[2][TB][8];               // partial sums of squares of a row
};
template <int ND, bool STATE> struct ChannelSmem {          // per-channel decays
  float G[2][ND * 16];              // over the block
  float part[17][ND * 16];          // over 4 tokens: rows 3 to 6 and 10 to 13, ones between and around them
  float raw[2][STATE ? 1 : ND * 16][3 * TB + 4];  // q, k and decays of a channel below MIN_DECAY
  float xP[2][STATE ? 2 : 256];     // such channels' share of P, [j][i]
  unsigned long long bad[2][2];     // which channels
};
template <int ND> struct ScalarSmem {           // one decay a token
  Gates g[4];
  float nq[2][ND][TB], n[ND * 16];  // MLSTM: n . q_i by 16 channels, n
};

// ND * 16 >= d
// STATE: only the states after the segments that have a successor
// LONG: with a loop for the full blocks of whole heads beside the general one, which pays from MIN_LONG tokens on
template <typename S, int ND, int MODE, bool STATE, bool LONG>
__global__ void __launch_bounds__(NTH) recurrence_chunk_kernel(ChunkArgs a) {
  constexpr bool CHANNEL = MODE == HGRN2 || MODE == GLA;
  constexpr int DP = ND * 16, LQ = DP + 8;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  using Image = Smem<ND, STATE>;
  using Channels = ChannelSmem<ND, STATE>;
  Image& sm = *reinterpret_cast<Image*>(smem_raw);
  Channels& cm = *reinterpret_cast<Channels*>(smem_raw + sizeof(Image));
  ScalarSmem<ND>& gm = *reinterpret_cast<ScalarSmem<ND>*>(smem_raw + sizeof(Image));
  const int H = a.H, d = a.d, dv = a.dv;
  const int segs = STATE ? a.nseg - 1 : a.nseg;
  const int h = blockIdx.x, s = blockIdx.y / segs, seg = blockIdx.y % segs, c0 = blockIdx.z * COLS;
  const int end = a.cu[s + 1], first = a.cu[s];
  const int slot = a.slots[s], t0 = first + seg * a.seg_tokens;
  if (end <= t0 || end - first < a.min_len) return;
  const int t1 = seg + 1 < a.nseg && end - t0 > a.seg_tokens ? t0 + a.seg_tokens : end;
  const bool last = t1 == end, cut = end - first > a.seg_tokens;
  if (STATE && (last || slot < 0)) return;
  const int tid = threadIdx.x, lane = tid & 63, w = MODE == MLSTM ? tid >> 6 : __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, q = lane >> 4;
  const int col = c0 + w * 16 + fr;             // this lane's state column
  const bool on = col < dv, wave_on = c0 + w * 16 < dv;
  S* out = (S*)a.out;
  float* outf = (float*)a.out;                  // FIXED: raw read-outs, fp32
  if (slot < 0) {                               // padding rows
    if (on)
      for (int t = t0 + q; t < t1; t += 4) {
        if (MODE == FIXED) outf[(long)t * a.ldo + h * dv + col] = 0.f;
        else stf(out + (long)t * a.ldo + h * dv + col, 0.f);
      }
    return;
  }
  const bool fresh = a.positions[first] == 0;
  float* sp = a.state + ((long)slot * H + h) * d * dv + col;
  float* np = MODE == MLSTM ? a.nstate + ((long)slot * H + h) * (d + 1) : nullptr;
  const auto unit = [&](int k) { return ((long)s * a.nseg + k) * H + h; };
  // Segments' states lie as the accumulators hold them, 8 requests of 1 KiB a wave; row by row a lane took 32, each a quarter
  // wave's 64 bytes, for every segment folded. us, row by row / so: GLA 301 to 3000 (6) 534 / 491, FIXED 900 to
  // 2601 (5) 445 / 395, MLSTM 322 / 289, 1 x 8000 FIXED 368 / 343, MLSTM 331 / 273
  const auto seg_st = [&](int k) {
    return (f32x4*)a.seg_state + ((unit(k) * gridDim.z + blockIdx.z) * 8 + w) * ND * 64 + lane;
  };
  f32x4 st[ND];
  const auto load_state = [&](const float* p) {
#pragma unroll
    for (int t = 0; t < ND; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int c = 16 * t + 4 * q + r;
        st[t][r] = p != nullptr && on && c < d ? p[(long)c * dv] : 0.f;
      }
  };
  const auto load_segment = [&](int k) __attribute__((always_inline)) {
    const f32x4* p = seg_st(k);
#pragma unroll
    for (int t = 0; t < ND; ++t) st[t] = p[t * 64];
  };
  const auto store_segment = [&](int k) __attribute__((always_inline)) {
    f32x4* p = seg_st(k);
#pragma unroll
    for (int t = 0; t < ND; ++t) p[t * 64] = st[t];
  };
  const auto store_state = [&](float* p) {
    if (on) {
#pragma unroll
      for (int t = 0; t < ND; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int c = 16 * t + 4 * q + r;
          if (c < d) p[(long)c * dv] = st[t][r];
        }
    }
  };
  // The first state. Where the portion is cut, the output launch's last segment replaces the state
  // that the first one starts from, in any order: the first reads the copy that the state launch
  // took. Later segments fold the states before them.
  const int nc = w * 16 + fr;                   // this lane's channel of the normaliser
  float n0 = 0.f;
  if (seg == 0) {
    const bool copied = !STATE && cut;
    if (copied && !fresh) load_segment(a.nseg - 1);
    else load_state(fresh ? nullptr : sp);
    if (MODE == MLSTM && !fresh && nc < d) n0 = copied ? a.seg_n[unit(a.nseg - 1) * UNIT + nc] : np[nc];
    if (STATE && !fresh) {
      store_segment(a.nseg - 1);
      if (MODE == MLSTM && q == 0 && nc < d) a.seg_n[unit(a.nseg - 1) * UNIT + nc] = n0;
    }
  } else {
    if (STATE) load_state(nullptr);
    else load_segment(0);
    if (!STATE) {
      if (MODE == MLSTM && nc < d) n0 = a.seg_n[unit(0) * UNIT + nc];
      float Gs = 0.f, Gl = 0.f;
      if (MODE == FIXED) {                      // a segment's decay, as in scalar_gates
        double p = 1.0, x = (double)a.decays[h];
        for (int e = a.seg_tokens; e; e >>= 1, x *= x)
          if (e & 1) p *= x;
        Gs = (float)p;
        Gl = (float)(p - (double)Gs);
      }
      for (int k = 1; k < seg; ++k) {
        const float* dec = a.seg_decay + unit(k) * UNIT;
        const f32x4* own = seg_st(k);
        if (MODE == MLSTM) {
          Gs = dec[0];
          if (nc < d) n0 = Gs * n0 + a.seg_n[unit(k) * UNIT + nc];
        }
#pragma unroll
        for (int t = 0; t < ND; ++t) {
          if (CHANNEL) st[t] *= *reinterpret_cast<const f32x4*>(dec + 16 * t + 4 * q);
          else if (MODE == FIXED) st[t] = st[t] * Gs + st[t] * Gl;
          else st[t] *= Gs;
          st[t] += own[t * 64];
        }
      }
    }
  }
  if (MODE == MLSTM && w < ND && q == 0) gm.n[nc] = n0;
  float G_seg = 1.f;                            // STATE: this thread's channel's, or the gate wave's
  // staging: thread = (channel sc and column sc of the block's 128, tokens 4 tg .. 4 tg + 3)
  const int sc = tid & 127, tg = w >> 1;
  const bool chan = sc < d, scol = c0 + sc < dv;
  float bias = 0.f, low = 0.f;
  if (CHANNEL && chan) {
    bias = ldf((const S*)a.bias + h * d + sc);
    if (MODE == HGRN2) low = ldf((const S*)a.lower + h * d + sc);
  }
  const int goff = 2 * H * d + H * dv + h * dv + min(col, dv - 1);   // output gate
  constexpr int GW = 7;                                         // the gate wave
  const int nb = (t1 - t0 + TB - 1) / TB;
  auto tokens = [&](int b) { return min(TB, t1 - t0 - b * TB); };
  // FULL: a head of 128 channels and columns, and blocks of 16 tokens (the loop says which). A lane's places in a
  // block of rows are then constant and the rows' start is scalar, without a bound or a branch a token
  const bool whole = ND == 8 && d == DP && c0 + COLS <= dv && a.ldp < 1 << 24 && a.ldz < 1 << 24 && a.ldo < 1 << 24;
  const uint32_t pat = 4u * (4 * tg * a.ldp + sc), zat = 4u * (4 * tg * a.ldz + sc);
  const uint32_t gat = 4u * (4 * q * a.ldp + w * 16 + fr);
  const uint32_t oat = sizeof(S) * (4 * q * a.ldo + w * 16 + fr);
  const auto at = [](const float* base, uint32_t bytes) { return *(const float*)((const char*)base + bytes); };
  float rq[4], rk[4], rz[4], rv[4], ra[4];
  f32x4 gin = {1.f, 0.f, 0.f, 0.f};
  auto load = [&](int b, auto FULL) __attribute__((always_inline)) {
    const int tc = t0 + b * TB, n = tokens(b);
    if constexpr (decltype(FULL)::value) {
      const float* rows = a.proj + (long)tc * a.ldp + h * d;
      const float* vals = a.proj + (long)tc * a.ldp + 2 * H * d + h * dv + c0;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint32_t ro = pat + 4u * u * a.ldp;
        if (!STATE) rq[u] = at(rows, ro);
        rk[u] = at(rows + H * d, ro);
        if (MODE == GLA) rz[u] = at(a.z + (long)tc * a.ldz + h * d, zat + 4u * u * a.ldz);
        rv[u] = at(vals, ro);
      }
      return;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = 4 * tg + u;
      rq[u] = rk[u] = rz[u] = rv[u] = 0.f;
      if (t < n) {
        const float* row = a.proj + (long)(tc + t) * a.ldp;
        if (chan) {
          if (!STATE) rq[u] = row[h * d + sc];
          rk[u] = row[H * d + h * d + sc];
          if (MODE == GLA) rz[u] = a.z[(long)(tc + t) * a.ldz + h * d + sc];
        }
        if (scol) rv[u] = row[2 * H * d + h * dv + c0 + sc];
      }
    }
  };
  auto load_gates = [&](int b) {                // MLSTM: the gate wave's
    if (MODE == MLSTM && w == GW && b < nb && fr < tokens(b))
      gin = *reinterpret_cast<const f32x4*>(a.gates + ((long)(t0 + b * TB + fr) * H + h) * 4);
  };
  // per-channel decays of the block in the registers, and their products over 4 tokens
  auto channel_gates = [&](int b, auto FULL) __attribute__((always_inline)) {
    const int n = tokens(b);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const bool real = decltype(FULL)::value || (4 * tg + u < n && chan);
      if (MODE == HGRN2) {
        ra[u] = real ? low + (1.f - low) * sigmoid1(rk[u] + bias) : 1.f;
        rk[u] = real ? 1.f - ra[u] : 0.f;
      } else {
        ra[u] = real ? decay_pow(rz[u] + bias, a.inv_tau) : 1.f;
      }
    }
    if (decltype(FULL)::value || sc < DP) cm.part[3 + 7 * (b & 1) + tg][sc] = (ra[0] * ra[1]) * (ra[2] * ra[3]);
  };
  // scalar tables of a block of n tokens (one wave; lane t of every row of 16 holds token t)
  auto scalar_gates = [&](int n, Gates& gt) {
    float at = 1.f, bt = 0.f, em = 0.f;
    if (MODE == FIXED) {
      // one decay for the whole sequence: its error adds up over the blocks, so the powers are formed
      // in double and the block's decay carries a second float
      const double a1 = (double)a.decays[h];
      double p = 1.0, A = 1.0, B = 1.0, D[4] = {1.0, 1.0, 1.0, 1.0};
      for (int t = 0; t <= n; ++t, p *= a1) {   // p = a^t
        if (t == min(fr, n - 1) + 1) A = p;
        if (t == n - 1 - fr) B = p;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (t == min(fr, n - 1) - (4 * q + r)) D[r] = p;
        if (t == n && lane == 0) {
          gt.G[0] = (float)p;
          gt.G[1] = (float)(p - (double)(float)p);
        }
      }
      f32x4 Df;
#pragma unroll
      for (int r = 0; r < 4; ++r) Df[r] = 4 * q + r <= fr && 4 * q + r < n ? (float)D[r] : 0.f;
      *reinterpret_cast<f32x4*>(gt.D + fr * LT + 4 * q) = Df;
      if (lane < TB) {
        gt.A[lane] = (float)A;
        gt.kb[lane] = lane < n ? (float)B : 0.f;
      }
      return;
    }
    at = fr < n ? gin[0] : 1.f;
    bt = fr < n ? gin[1] : 0.f;
    em = fr < n ? gin[2] : 0.f;
    float A = at, B = at;                       // products up to a token, and from it on
#define PRODUCTS(N) A *= row<0x110 + N>(1.f, A), B *= row<0x100 + N>(1.f, B)
    PRODUCTS(1); PRODUCTS(2); PRODUCTS(4); PRODUCTS(8);
#undef PRODUCTS
    B = row<0x101>(1.f, B);
    const float G = from_lane(A, TB - 1);
    f32x4 D = {1.f, 1.f, 1.f, 1.f};
    if (G >= MIN_DECAY) {                       // A_i / A_j
#pragma unroll
      for (int r = 0; r < 4; ++r) D[r] = A * rcp1(__shfl(A, 4 * q + r, 64));
    } else {                                    // the decays in between, one by one
#pragma unroll 1
      for (int t = 0; t < TB; ++t) {
        const float x = from_lane(at, t);
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (t <= fr && t > 4 * q + r) D[r] *= x;
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) D[r] = 4 * q + r <= fr ? D[r] * __shfl(bt, 4 * q + r, 64) : 0.f;
    *reinterpret_cast<f32x4*>(gt.D + fr * LT + 4 * q) = D;
    if (lane < TB) {
      gt.A[lane] = A;
      gt.kb[lane] = bt * B;
      gt.em[lane] = em;
    }
    if (lane == 0) gt.G[0] = G;
    G_seg *= G;
  };
  // fixed decays: table 0 for full blocks, 1 for a shorter last one
  auto table = [&](int b, auto FULL) __attribute__((always_inline)) -> Gates& {
    return gm.g[MODE == FIXED ? !decltype(FULL)::value && tokens(b) < TB : (b & 3)];
  };
  // a block's LDS image from the registers
  auto stage = [&](int b, auto FULL) __attribute__((always_inline)) {
    const int buf = b & 1;
    f32x4 kb, vv;
    if (decltype(FULL)::value || sc < DP) {
      if constexpr (CHANNEL) {
        float A[4], B[4];
        const float* const around = &cm.part[7 * buf + tg][sc];
        const float pre = around[0] * around[DP] * around[2 * DP], post = around[4 * DP] * around[5 * DP] * around[6 * DP];
        A[0] = pre * ra[0]; A[1] = A[0] * ra[1]; A[2] = A[1] * ra[2]; A[3] = A[2] * ra[3];
        B[3] = post; B[2] = B[3] * ra[3]; B[1] = B[2] * ra[2]; B[0] = B[1] * ra[1];
        const float G = A[3] * post;
        const bool bad = !(G >= MIN_DECAY);
        if (tg == 0) {
          cm.G[buf][sc] = G;
          if (STATE) G_seg *= G;
          const unsigned long long m = __ballot(bad);
          if (lane == 0) cm.bad[buf][w] = m;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int t = 4 * tg + u;
          kb[u] = rk[u] * B[u];
          if (STATE) continue;
          const float qq = MODE == HGRN2 ? silu1(rq[u]) : rq[u] * a.qscale;
          sm.Q[buf][t * LQ + sc] = qq * A[u];
          sm.K[buf][t * LQ + sc] = bad ? 0.f : rk[u] * rcp1(A[u]);
          if (bad) {
            cm.raw[buf][sc][t] = qq;
            cm.raw[buf][sc][TB + t] = rk[u];
            cm.raw[buf][sc][2 * TB + t] = ra[u];
          }
        }
      } else {
        const f32x4 kw = *reinterpret_cast<const f32x4*>(table(b, FULL).kb + 4 * tg);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int t = 4 * tg + u;
          const float kk = MODE == FIXED ? silu1(rk[u]) : rk[u];
          kb[u] = kk * kw[u];
          if (STATE) continue;
          const float qq = MODE == FIXED ? silu1(rq[u]) : rq[u] * a.qscale;
          sm.Q[buf][t * LQ + sc] = qq;
          sm.K[buf][t * LQ + sc] = kk;
        }
      }
      *reinterpret_cast<f32x4*>(sm.Kb[buf] + sc * LT + 4 * tg) = kb;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) vv[u] = MODE == FIXED ? silu1(rv[u]) : rv[u];
    *reinterpret_cast<f32x4*>(sm.V[buf] + sc * LT + 4 * tg) = vv;
  };

  unsigned long long bad0 = 0, bad1 = 0, bad0n = 0, bad1n = 0;
  f32x4 vf = {0.f, 0.f, 0.f, 0.f}, acc = vf, vfn = vf, accn = vf;
  // block b: P's partial sums to LDS, the read-out of the state before it to accn, the state after it
  auto products = [&](int b, auto FULL) __attribute__((always_inline)) {
    const int buf = b & 1;
    const float* Q = sm.Q[buf];
    if (w < ND && (!STATE || MODE == MLSTM)) {  // this wave's 16 channels of P^T
      f32x4 qf;
      if (!STATE) {
        qf = *reinterpret_cast<const f32x4*>(Q + fr * LQ + 16 * w + 4 * q);
        const f32x4 kf = *reinterpret_cast<const f32x4*>(sm.K[buf] + fr * LQ + 16 * w + 4 * q);
        const f32x4 p = mfma4(kf, qf, f32x4{0.f, 0.f, 0.f, 0.f});
        *reinterpret_cast<f32x4*>(&sm.P[buf][w][4 * lane]) = p;
      }
      if (MODE == MLSTM) {                      // n . q_i over them, then n after the block
        if (!STATE) {
          const f32x4 nf = *reinterpret_cast<const f32x4*>(gm.n + 16 * w + 4 * q);
          float x = (nf[0] * qf[0] + nf[1] * qf[1]) + (nf[2] * qf[2] + nf[3] * qf[3]);
          x += __shfl_xor(x, 16, 64);
          x += __shfl_xor(x, 32, 64);
          if (q == 0) gm.nq[buf][w][fr] = x;
        }
        const f32x4 kb = *reinterpret_cast<const f32x4*>(sm.Kb[buf] + (16 * w + fr) * LT + 4 * q);
        float y = (kb[0] + kb[1]) + (kb[2] + kb[3]);
        y += __shfl_xor(y, 16, 64);
        y += __shfl_xor(y, 32, 64);
        if (q == 0) gm.n[16 * w + fr] = table(b, FULL).G[0] * gm.n[16 * w + fr] + y;
      }
    }
    if constexpr (CHANNEL && !STATE) {
      bad0n = cm.bad[buf][0];
      bad1n = DP > 64 ? cm.bad[buf][1] : 0;
      if ((bad0n | bad1n) != 0 && tid < 256) {
        const int i = tid & 15, j = tid >> 4;
        float x = 0.f;
        if (j <= i) {
          for (int half = 0; half < 2; ++half)
            for (unsigned long long m = half ? bad1n : bad0n; m; m &= m - 1) {
              const float* rw = cm.raw[buf][64 * half + __builtin_ctzll(m)];
              float p = rw[i] * rw[TB + j];
              for (int t = j + 1; t <= i; ++t) p *= rw[2 * TB + t];
              x += p;
            }
        }
        cm.xP[buf][tid] = x;
      }
    }
    if (decltype(FULL)::value || wave_on) {
      vfn = *reinterpret_cast<const f32x4*>(sm.V[buf] + (16 * w + fr) * LT + 4 * q);
      f32x4 part[4];                            // short sums round less than one of d terms
#pragma unroll
      for (int t = 0; t < 4; ++t) part[t] = f32x4{0.f, 0.f, 0.f, 0.f};
      float Gs = 0.f, Gl = 0.f;
      if constexpr (!CHANNEL) Gs = table(b, FULL).G[0];
      if (MODE == FIXED) Gl = table(b, FULL).G[1];
      f32x4 qf, kb, Gt, qn, kn, Gn;
      if constexpr (CHANNEL) __builtin_amdgcn_s_setprio(1);
      const auto read = [&](int t) __attribute__((always_inline)) {
        if (!STATE) qn = *reinterpret_cast<const f32x4*>(Q + fr * LQ + 16 * t + 4 * q);
        kn = *reinterpret_cast<const f32x4*>(sm.Kb[buf] + (16 * t + fr) * LT + 4 * q);
        if constexpr (CHANNEL) Gn = *reinterpret_cast<const f32x4*>(cm.G[buf] + 16 * t + 4 * q);
      };
      read(0);
#pragma unroll
      for (int t = 0; t < ND; ++t) {            // tile t's read-out and update side by side
        qf = qn; kb = kn; Gt = Gn;
        // the next tile's operands on their way ahead of this one's products; hipcc reads them where they are used
        if (t + 1 < ND) read(t + 1);
        __builtin_amdgcn_sched_barrier(0x6);    // (vector and scalar arithmetic may pass)
        f32x4 sn;
        if constexpr (CHANNEL) sn = st[t] * Gt;
        else sn = st[t] * Gs;
        if (MODE == FIXED) sn += st[t] * Gl;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (!STATE)
            part[t & 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[r], st[t][r], part[t & 3], 0, 0, 0);
          sn = __builtin_amdgcn_mfma_f32_16x16x4f32(kb[r], vfn[r], sn, 0, 0, 0);
        }
        st[t] = sn;
      }
      if constexpr (CHANNEL) __builtin_amdgcn_s_setprio(0);
      accn = (part[0] + part[1]) + (part[2] + part[3]);
    }
  };
  f32x4 o = {0.f, 0.f, 0.f, 0.f}, gate = o;
  float nw = 0.f;
  if (!STATE && MODE != FIXED && on) nw = ldf((const S*)a.norm_w + (MODE == MLSTM ? h * dv + col : col));
  // o = the read-outs of block b (rows 4 q + r, this lane's column) from vf, acc and P
  auto finish = [&](int b, auto FULL) __attribute__((always_inline)) {
    const int buf = b & 1;
    if ((MODE == GLA || MODE == MLSTM) && decltype(FULL)::value) {
      const float* rows = a.proj + (long)(t0 + b * TB) * a.ldp + 2 * H * d + H * dv + h * dv + c0;
#pragma unroll
      for (int r = 0; r < 4; ++r) gate[r] = at(rows, gat + 4u * r * a.ldp);
    } else if (MODE == GLA || MODE == MLSTM) {
      // (rows and columns past the last again, unused: with a condition a load hipcc waits for the one before, and so for all
      // in flight, ahead of each. MLSTM, 32 x 256 tokens, 32 heads of 64 317 / 243 us, 16 of 100 191 / 182; GLA, 8 of 64 67 / 63)
      const int n = tokens(b);
#pragma unroll
      for (int r = 0; r < 4; ++r) gate[r] = a.proj[(long)(t0 + b * TB + min(4 * q + r, n - 1)) * a.ldp + goff];
    }
    f32x4 p = {0.f, 0.f, 0.f, 0.f}, ps[ND];     // P_ij, i = fr, j = 4 q + r
#pragma unroll
    for (int x = 0; x < ND; ++x) ps[x] = *reinterpret_cast<const f32x4*>(&sm.P[buf][x][4 * lane]);
    __builtin_amdgcn_sched_barrier(0x6);
#pragma unroll
    for (int x = 0; x < ND; ++x) p += ps[x];
    float inv = 0.f;
    if constexpr (CHANNEL) {
      const bool extra = (bad0 | bad1) != 0;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (extra) p[r] += cm.xP[buf][(4 * q + r) * 16 + fr];
        p[r] = 4 * q + r <= fr ? p[r] : 0.f;
      }
    } else {
      const Gates& gt = table(b, FULL);
      const f32x4 D = *reinterpret_cast<const f32x4*>(gt.D + fr * LT + 4 * q);
#pragma unroll
      for (int r = 0; r < 4; ++r) p[r] = 4 * q + r <= fr ? p[r] * D[r] : 0.f;
      acc *= *reinterpret_cast<const f32x4*>(gt.A + 4 * q);
      if (MODE == MLSTM) {
        float x = (p[0] + p[1]) + (p[2] + p[3]);
        x += __shfl_xor(x, 16, 64);
        x += __shfl_xor(x, 32, 64);
        float y = 0.f;
#pragma unroll
        for (int u = 0; u < ND; ++u) y += gm.nq[buf][u][fr];
        inv = 1.f / (fmaxf(fabsf(x + gt.A[fr] * y), gt.em[fr]) + 1e-6f);
      }
    }
    // a masked P_ij is zero, but zero times a value that is not finite is not: such a block's terms are
    // added one by one, so that no token feels a later one
    if (__ballot(((vf[0] - vf[0]) + (vf[1] - vf[1])) + ((vf[2] - vf[2]) + (vf[3] - vf[3])) != 0.f) == 0) {
      o = mfma4(p, vf, acc);
    } else {
      o = acc;
#pragma unroll 1
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float v = __shfl(vf[u], 16 * g + fr, 64);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float pij = __shfl(p[u], 16 * g + 4 * q + r, 64);
            if (4 * g + u <= 4 * q + r) o[r] = fmaf(pij, v, o[r]);
          }
        }
    }
    if (MODE != FIXED) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (MODE == MLSTM) o[r] *= __shfl(inv, 4 * q + r, 64);
        float x = o[r] * o[r];
        x = row_sum(x);
        if (fr == 0) sm.ss[buf][4 * q + r][w] = x;
      }
    }
  };
  auto write_out = [&](int b, auto FULL) __attribute__((always_inline)) {
    const int n = tokens(b);
    float rs = 0.f;
    if (MODE != FIXED) {                        // row fr's
      const float* sq = sm.ss[b & 1][fr];
      const f32x4 x = *reinterpret_cast<const f32x4*>(sq), y = *reinterpret_cast<const f32x4*>(sq + 4);
      const float n_cols = decltype(FULL)::value ? (float)COLS : (float)dv;
      rs = 1.f / sqrtf((((x[0] + x[1]) + (x[2] + x[3])) + ((y[0] + y[1]) + (y[2] + y[3]))) / n_cols + a.eps);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 4 * q + r;
      const float rr = MODE != FIXED ? __shfl(rs, i, 64) : 0.f;
      if (!decltype(FULL)::value && (i >= n || !on)) continue;
      const long t = (long)t0 + b * TB + i;
      char* const rows = (char*)((S*)a.out + (long)(t0 + b * TB) * a.ldo + h * dv + c0);      // FULL: row 0's
      if (MODE == FIXED) {
        if (decltype(FULL)::value) *(float*)(rows + oat + sizeof(S) * r * a.ldo) = o[r];
        else outf[t * a.ldo + h * dv + col] = o[r];
        continue;
      }
      float v = o[r] * rr * nw;
      if (MODE == GLA) v *= silu1(gate[r]);
      if (MODE == MLSTM) v *= sigmoid1(gate[r]) * a.out_scale;
      stf(decltype(FULL)::value ? (S*)(rows + oat + sizeof(S) * r * a.ldo) : out + t * a.ldo + h * dv + col, v);
    }
  };

  using Any = std::integral_constant<bool, false>;
  load(0, Any{});
  load_gates(0);
  if constexpr (CHANNEL) {
    if (tid < DP)
#pragma unroll
      for (int x = 0; x < 9; ++x) cm.part[x + x / 3 * 4][tid] = 1.f;
    channel_gates(0, Any{});
  } else if (w == GW) {
    scalar_gates(tokens(0), table(0, Any{}));
    if (MODE == FIXED) {
      if (nb > 1) scalar_gates(tokens(nb - 1), table(nb - 1, Any{}));
    } else if (nb > 1) {
      load_gates(1);
      scalar_gates(tokens(1), table(1, Any{}));
    }
    load_gates(2);
  }
  __syncthreads();
  stage(0, Any{});
  if (nb > 1) {
    load(1, Any{});
    if constexpr (CHANNEL) channel_gates(1, Any{});
  }
  __syncthreads();
  // FULL: blocks b - 2 to b + 2 are there, and full
  auto step = [&](int b, auto FULL) __attribute__((always_inline)) {
    constexpr bool full = decltype(FULL)::value;
    // (per-channel decays of wide heads that are no whole tile: GLA, 32 x 256 tokens, 16 heads of 112 198 us, behind it 192)
    constexpr bool FIRST = CHANNEL && (LONG || ND < 8);
    if (!STATE && FIRST && w < 4 && (full || b < nb)) products(b, FULL);
    if (full || b + 1 < nb) stage(b + 1, FULL);
    if (full || b + 2 < nb) {
      load(b + 2, FULL);
      if (MODE == MLSTM && w == GW) {
        scalar_gates(full ? TB : tokens(b + 2), table(b + 2, FULL));
        load_gates(b + 3);
      }
    }
    if constexpr (STATE) {
      products(b, FULL);
    } else {
      if (!FIRST && w < 4 && (full || b < nb)) products(b, FULL);
      if (full || b >= 2) write_out(b - 2, FULL);
      if (full || (b >= 1 && b <= nb)) finish(b - 1, FULL);
      if (w >= 4 && (full || b < nb)) products(b, FULL);
      vf = vfn; acc = accn; bad0 = bad0n; bad1 = bad1n;
    }
    if constexpr (CHANNEL) {
      if (full || b + 2 < nb) channel_gates(b + 2, FULL);
    }
    lds_barrier();
  };
  const int full_to = whole ? (t1 - t0) / TB - 2 : 0;
#pragma unroll 1
  for (int b = 0; b < nb + (STATE ? 0 : 2); ++b) {
    if constexpr (LONG) {
      if (STATE || b >= 2)
#pragma unroll 1
        for (; b < full_to; ++b) step(b, std::integral_constant<bool, true>{});
    }
    step(b, Any{});
  }
  if constexpr (STATE) {
    store_segment(seg);
    if (CHANNEL && tg == 0 && blockIdx.z == 0) a.seg_decay[unit(seg) * UNIT + sc] = sc < DP ? G_seg : 1.f;
    if (MODE == MLSTM) {
      if (w < ND && q == 0 && nc < d) a.seg_n[unit(seg) * UNIT + nc] = gm.n[nc];
      if (w == GW && lane == 0) a.seg_decay[unit(seg) * UNIT] = G_seg;
    }
  } else if (last) {
    store_state(sp);
    if (MODE == MLSTM && w < ND && q == 0 && nc < d) np[nc] = gm.n[nc];
  }
}

// MLSTM's gates: a_t = exp(f_t + m_{t-1} - m_t), b_t = exp(i_t - m_t) and exp(-m_t) of every token of a
// (head, sequence), and the state's m after the portion. Inside the products' launch, where one wave did this for a block
// beside its share of the products, it was what the other waves waited for.
//
// m_t = max(f_t + m_{t-1}, i_t) is a map m -> max(F + m, I), and such maps compose. A lane of one wave composes the
// maps of 33 tokens (an odd stride in LDS), a prefix over the lanes gives the m ahead of each, and every lane walks
// its own: where one walk of all the tokens bound this launch, 64 go side by side. 16 heads, us, that walk / this:
// 5 portions of 900 to 2601 tokens 68 / 17, 1 x 8000 195 / 38, 64 x 33 9.6 / 6.6. The walk within a lane matters: where
// no i_t wins, a_t is one, and a prefix over single tokens, whose a_t round about it, lost up to half a digit against
// 64 bits. So does the prefix in double: read-outs and states are as near as those of the one walk (1.9e-7 and
// 1.2e-7 at forget biases of 3), m nearer where few i_t win (bias 6, 4000 tokens: 1.5e-6 -> 1.2e-7).
__global__ void __launch_bounds__(512) mlstm_gates_kernel(ChunkArgs a, float* gates) {
  constexpr int OWN = 33, N = 64 * OWN, EACH = (N + 511) / 512;
  __shared__ float ig[N], fg[N], m[N + 1];
  const int h = blockIdx.x, s = blockIdx.y, H = a.H, tid = threadIdx.x, lane = tid & 63;
  const int slot = a.slots[s], first = a.cu[s], end = a.cu[s + 1];
  if (slot < 0 || end <= first || end - first < a.min_len) return;
  float* mp = a.nstate + ((long)slot * H + h) * (a.d + 1) + a.d;
  const float* col = a.proj + 2 * H * a.d + 2 * H * a.dv + h;
  const float bi = a.if_b[h], bf = a.if_b[H + h];
  if (tid == 0) m[0] = a.positions[first] == 0 ? 0.f : *mp;
  for (int t0 = first; t0 < end; t0 += N) {
    const int n = min(N, end - t0);
    float ri[EACH], rf[EACH];
#pragma unroll
    for (int x = 0; x < EACH; ++x) {
      const int t = min(tid + 512 * x, n - 1);
      ri[x] = col[(long)(t0 + t) * a.ldp];
      rf[x] = col[(long)(t0 + t) * a.ldp + H];
    }
#pragma unroll
    for (int x = 0; x < EACH; ++x) {
      const int t = tid + 512 * x;
      if (t >= n) break;
      ig[t] = a.cap * tanhf((ri[x] + bi) / a.cap);
      fg[t] = logsigmoid32(a.cap * tanhf((rf[x] + bf) / a.cap));
    }
    __syncthreads();
    if (tid < 64 && lane * OWN < n) {           // (what the last of them makes of rows past the portion, nothing reads)
      const float *il = ig + lane * OWN, *fl = fg + lane * OWN;
      double F = 0.0, I = -INFINITY;
#pragma unroll
      for (int u = 0; u < OWN; ++u) {
        I = fmax(fl[u] + I, (double)il[u]);
        F += fl[u];
      }
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const double Fb = __shfl_up(F, o, 64), Ib = __shfl_up(I, o, 64);
        if (lane >= o) {
          I = fmax(F + Ib, I);
          F += Fb;
        }
      }
      const double Fb = __shfl_up(F, 1, 64), Ib = __shfl_up(I, 1, 64);
      float run = lane == 0 ? m[0] : (float)fmax(Fb + m[0], Ib);
#pragma unroll
      for (int u = 0; u < OWN; ++u) {
        run = fmaxf(fl[u] + run, il[u]);
        m[lane * OWN + u + 1] = run;
      }
    }
    __syncthreads();
    for (int t = tid; t < n; t += 512) {
      const float mt = m[t + 1];
      *reinterpret_cast<f32x4*>(gates + ((long)(t0 + t) * H + h) * 4) =
          f32x4{expf(fg[t] + m[t] - mt), expf(ig[t] - mt), expf(-mt), 0.f};
    }
    __syncthreads();
    if (tid == 0) m[0] = m[n];
    __syncthreads();
  }
  if (tid == 0) *mp = m[0];
}

template <typename S, int ND, int MODE, bool STATE, bool LONG>
int launch_one(const ChunkArgs& a, int num_seqs, hipStream_t st) {
  constexpr size_t sh = sizeof(Smem<ND, STATE>) +
                        (MODE <= GLA ? sizeof(ChannelSmem<ND, STATE>) : sizeof(ScalarSmem<ND>));
  static_assert(sh <= 160 * 1024 && sizeof(Smem<ND, STATE>) % 16 == 0, "LDS image");
  if (sh > 48 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)recurrence_chunk_kernel<S, ND, MODE, STATE, LONG>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)sh);
    if (e != hipSuccess) return (int)e;
  }
  dim3 grid(a.H, num_seqs * (STATE ? a.nseg - 1 : a.nseg), (a.dv + COLS - 1) / COLS);
  recurrence_chunk_kernel<S, ND, MODE, STATE, LONG><<<grid, NTH, sh, st>>>(a);
  DLI_RETURN_LAUNCH();
}
// Whether portions of at most max_seqlen tokens take the kernels with a loop for full blocks. Blocks b - 2 to b + 2 are full
// for the first time in a portion of 5 blocks. 64 portions of 80 / 96 / 128 tokens, us, without and with that loop: HGRN2 235 /
// 273 / 345 and 242 / 275 / 338, GLA 273 / 319 / 412 and 276 / 309 / 379, FIXED 211 / 242 / 302 and 209 / 237 / 293, MLSTM
// 144 / 174 / 220 and 150 / 180 / 219. Segments have 128 tokens and more. Only where the heads can run that loop: the general one
// beside it costs more than by itself (4 x 2048 tokens, HGRN2, 32 heads of 96 534 / 432 us, GLA, 16 of 112 328 / 262)
bool takes_long(int mode, int max_seqlen, int d, int dv, int ldp, int ldz, int ldo) {
  return d == 128 && dv >= COLS && ldp < 1 << 24 && ldz < 1 << 24 && ldo < 1 << 24 && max_seqlen >= (mode == MLSTM ? 128 : 96);
}
template <typename S, int ND, int MODE>
int launch_chunks(const ChunkArgs& a, int num_seqs, int max_seqlen, hipStream_t st) {
  constexpr bool WIDE = ND == 8;
  const bool lng = WIDE && takes_long(MODE, max_seqlen, a.d, a.dv, a.ldp, a.ldz, a.ldo);
  if (a.nseg > 1) {
    const int rc = lng ? launch_one<S, ND, MODE, true, WIDE>(a, num_seqs, st) : launch_one<S, ND, MODE, true, false>(a, num_seqs, st);
    if (rc) return rc;
  }
  return lng ? launch_one<S, ND, MODE, false, WIDE>(a, num_seqs, st) : launch_one<S, ND, MODE, false, false>(a, num_seqs, st);
}

template <typename S, int MODE>
int launch_by_width(const ChunkArgs& a, int num_seqs, int max_seqlen, hipStream_t st) {
  if (a.d <= 32) return launch_chunks<S, 2, MODE>(a, num_seqs, max_seqlen, st);
  if (a.d <= 64) return launch_chunks<S, 4, MODE>(a, num_seqs, max_seqlen, st);
  return launch_chunks<S, 8, MODE>(a, num_seqs, max_seqlen, st);
}

// Segments of a portion of at most max_seqlen tokens (T in all): a CU takes one workgroup, so few heads
// and sequences, or ragged ones, leave most of the chip idle for as long as the longest portion takes.
// Cut, every segment but the last runs twice, the first time (states only, several workgroups a CU) at
// some 0.3 of a block's time. In block times, with 3 to fill and drain a workgroup. The segments' states take at most 256
// MB of scratch.
// A portion may end in a segment of any length, and the lengths are on the device: rounds of workgroups count a whole one for
// each. But where they differ the shorter ones fill the CUs that others leave, so that no more than the work of a CU, half
// a last segment a portion, and part of a workgroup counts. Over 1400 mixes of 1 to 24 portions, 4 to 32 heads of 32 to 128 and all
// four recurrences, every number of segments timed, this is 1.039 of the best one's time (geometric mean), rounds of whole last
// segments alone 1.052; it is more than 3 % behind those on 5 mixes and ahead on 97. Rounds of half last segments are 1.051, and
// behind on 136: 4 of 1994 to 3988 tokens, HGRN2, 16 heads of 32, in 5 segments 225 us, in 9 143.
static size_t unit_floats(int d, int dv) {      // the state, in whole tiles, decays and normaliser
  return (size_t)(d <= 32 ? 32 : d <= 64 ? 64 : 128) * ((dv + COLS - 1) / COLS) * COLS + 2 * UNIT;
}
static int pick_segments(int H, int d, int dv, int num_seqs, int max_seqlen, int T, int min_len) {
  // the sequences that min_len leaves count for nothing: beside the longest at most this many others
  const int others = (T - max_seqlen) / (min_len > 1 ? min_len : 1);
  const int seqs = others < 0 ? 1 : others < num_seqs ? 1 + others : num_seqs;
  const long wg = (long)H * ((dv + COLS - 1) / COLS);
  const bool ragged = T < (long)seqs * max_seqlen;
  // what `units` workgroups a head of at most len tokens take that hold as much as `filled` whole ones' overhead and T tokens
  const auto time = [&](long units, long filled, int len, float behind) {
    const float one = len / 16.f + 3.f, even = (units * wg + 255) / 256 * one;
    if (!ragged || units * wg <= 256) return even;
    const float each = (T / 16.f + 3.f * filled) * wg / 256;
    return fminf(even, fmaxf(one, each) + behind * one);
  };
  float best = time(seqs, seqs, max_seqlen, 0.4f);
  int pick = 1;
  for (int n = 2; n <= 16 && (long)num_seqs * n <= 65535; ++n) {
    const int len = ((max_seqlen + n - 1) / n + TB - 1) / TB * TB;
    if (len < 128) break;
    const int k = (max_seqlen + len - 1) / len;
    if ((size_t)num_seqs * k * H * unit_floats(d, dv) > (64u << 20)) break;
    const long all = (long)seqs * k, whole = T / len + seqs, half = T / len + (seqs + 1) / 2;
    const float cost = time(all < whole ? all : whole, all < half ? all : half, len, 0.7f) * 1.3f + 0.1f * k;
    if (cost < best) { best = cost; pick = k; }
  }
  return pick;
}
static int segment_tokens(int max_seqlen, int nseg) {
  return ((max_seqlen + nseg - 1) / nseg + TB - 1) / TB * TB;
}

}  // namespace

// scratch that dli_recurrence_chunks takes for a step of T tokens (nullptr there: portions stay whole,
// which MLSTM does not take)
extern "C" long dli_recurrence_workspace_bytes(int mode, int num_seqs, int max_seqlen, int T,
                                               int min_len, int H, int d, int dv) {
  const int n = pick_segments(H, d, dv, num_seqs, max_seqlen, T, min_len);
  const size_t gates = mode == MLSTM ? (size_t)T * H * 4 : 0;
  return (long)((gates + (n > 1 ? (size_t)num_seqs * n * H * unit_floats(d, dv) : 0)) * 4);
}

// Portions of a step's sequences that bring at least min_len tokens (mode as above; the others' rows and
// states are left alone). hipErrorNotSupported: a size that the walk takes
// (d > 128, or a normed head wider than 128).
extern "C" int dli_recurrence_chunks(int mode, const float* proj, int ldp, const float* z, int ldz,
                                     const void* bias, const void* lower, float inv_tau, float qscale,
                                     const float* decays, const float* if_b, float cap,
                                     const void* norm_w, float eps, float* state, float* nstate,
                                     const int* slots, const int* cu, const int* positions, void* out,
                                     int ldo, float out_scale, int num_seqs, int max_seqlen, int T,
                                     int min_len, int H, int d, int dv, int dt, void* ws, hipStream_t st) {
  if (num_seqs <= 0 || max_seqlen <= 0) return 0;
  if (H < 1 || d < 1 || dv < 1 || num_seqs > 65535 || state == nullptr || slots == nullptr ||
      out == nullptr || (dt != 0 && dt != 1))
    return (int)hipErrorInvalidValue;
  if (d > 128 || (mode != FIXED && dv > COLS)) return (int)hipErrorNotSupported;
  ChunkArgs a{proj, ldp, z, ldz, bias, lower, inv_tau, qscale, decays, if_b, cap, norm_w, eps, state,
              nstate, slots, cu, positions, out, ldo, out_scale, H, d, dv, min_len, nullptr, 1 << 30, 1,
              nullptr, nullptr, nullptr};
  const int nseg = ws != nullptr ? pick_segments(H, d, dv, num_seqs, max_seqlen, T, min_len) : 1;
  float* scratch = (float*)ws;
  float* gates = scratch;
  if (mode == MLSTM) {
    a.gates = gates;
    scratch += (size_t)T * H * 4;
  }
  if (nseg > 1) {
    a.nseg = nseg;
    a.seg_tokens = segment_tokens(max_seqlen, nseg);
    const size_t units = (size_t)num_seqs * nseg * H;
    a.seg_decay = scratch;
    a.seg_n = a.seg_decay + units * UNIT;
    a.seg_state = a.seg_n + units * UNIT;
  }
  switch (mode) {
    case HGRN2:
      if (bias == nullptr || lower == nullptr || norm_w == nullptr) break;
      return dt == 0 ? launch_by_width<u16, HGRN2>(a, num_seqs, max_seqlen, st)
                     : launch_by_width<float, HGRN2>(a, num_seqs, max_seqlen, st);
    case GLA:
      if (z == nullptr || bias == nullptr || norm_w == nullptr) break;
      return dt == 0 ? launch_by_width<u16, GLA>(a, num_seqs, max_seqlen, st)
                     : launch_by_width<float, GLA>(a, num_seqs, max_seqlen, st);
    case FIXED:
      if (decays == nullptr) break;
      return launch_by_width<float, FIXED>(a, num_seqs, max_seqlen, st);
    case MLSTM:
      if (if_b == nullptr || norm_w == nullptr || nstate == nullptr || !(cap > 0.f) || ws == nullptr) break;
      mlstm_gates_kernel<<<dim3(H, num_seqs), 512, 0, st>>>(a, gates);
      return dt == 0 ? launch_by_width<u16, MLSTM>(a, num_seqs, max_seqlen, st)
                     : launch_by_width<float, MLSTM>(a, num_seqs, max_seqlen, st);
  }
  return (int)hipErrorInvalidValue;
}

// 1 where portions of whole sequences take the loop for full blocks
extern "C" int dli_recurrence_long(int mode, int max_seqlen, int d, int dv, int ldp, int ldz, int ldo) {
  return takes_long(mode, max_seqlen, d, dv, ldp, ldz, ldo) ? 1 : 0;
}
