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
// floor (1.9 us with two waves a SIMD); it takes 4 to 7 us, the rest being the gates and the LDS image.
// The walk's floor is one token after another: 0.5 to 1.2 us each. 4 prompts of 2048 tokens, d = dv =
// 128: HGRN2 1667 -> 621 us, GLA 2342 -> 704, FIXED 976 -> 517 (32 heads), MLSTM 1938 -> 895 (16 heads);
// 32 prompts of 256: 680 -> 354, 824 -> 397, 508 -> 295, 423 -> 240.
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
// matrix pipe and the vector unit busy at the same time.
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
  x = x > 88.f ? 88.f : x;
  x = x < -104.f ? -104.f : x;
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
};

// scalar decays of a block: A_i, b_j B_j, exp(-m_i), G, and D_ij = b_j prod_{j < t <= i} a_t
struct Gates { float A[TB], kb[TB], em[TB], G[4], D[TB * LT]; };   // G as a sum of two floats

template <int ND> struct Smem {
  static constexpr int DP = ND * 16, LQ = DP + 8;
  float Q[2][TB * LQ];              // q (per-channel decays: A_i q_i), token-major
  float K[2][TB * LQ];              // k (per-channel decays: k_j / A_j), token-major
  float Kb[2][DP * LT];             // B_j k_j, channel-major
  float V[2][COLS * LT];            // v, column-major
  float P[2][ND][256];              // partial sums of P^T, an accumulator a lane
  float ss[2][TB][8];               // partial sums of squares of a row
};
template <int ND> struct ChannelSmem {          // per-channel decays
  float G[2][ND * 16];              // over the block
  float part[2][4][ND * 16];        // over 4 tokens
  float raw[2][ND * 16][3 * TB + 4];  // q, k and decays of a channel below MIN_DECAY
  float xP[2][256];                 // such channels' share of P, [j][i]
  unsigned long long bad[2][2];     // which channels
};
template <int ND> struct ScalarSmem {           // one decay a token
  Gates g[4];
  float nq[2][ND][TB], n[ND * 16];  // MLSTM: n . q_i by 16 channels, n
};

// ND * 16 >= d
template <typename S, int ND, int MODE>
__global__ void __launch_bounds__(NTH) recurrence_chunk_kernel(ChunkArgs a) {
  constexpr bool CHANNEL = MODE == HGRN2 || MODE == GLA;
  constexpr int DP = ND * 16, LQ = DP + 8;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  Smem<ND>& sm = *reinterpret_cast<Smem<ND>*>(smem_raw);
  ChannelSmem<ND>& cm = *reinterpret_cast<ChannelSmem<ND>*>(smem_raw + sizeof(Smem<ND>));
  ScalarSmem<ND>& gm = *reinterpret_cast<ScalarSmem<ND>*>(smem_raw + sizeof(Smem<ND>));
  const int H = a.H, d = a.d, dv = a.dv;
  const int h = blockIdx.x, s = blockIdx.y, c0 = blockIdx.z * COLS;
  const int slot = a.slots[s], t0 = a.cu[s], t1 = a.cu[s + 1];
  if (t1 <= t0) return;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
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
  const bool fresh = a.positions[t0] == 0;
  float* sp = a.state + ((long)slot * H + h) * d * dv + col;
  float* np = MODE == MLSTM ? a.nstate + ((long)slot * H + h) * (d + 1) : nullptr;
  f32x4 st[ND];
#pragma unroll
  for (int t = 0; t < ND; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int c = 16 * t + 4 * q + r;
      st[t][r] = (!fresh && on && c < d) ? sp[(long)c * dv] : 0.f;
    }
  float m_run = 0.f;                            // the gate wave's running maximum
  if (MODE == MLSTM) {
    if (!fresh) m_run = np[d];
    if (w < ND && q == 0) gm.n[16 * w + fr] = (!fresh && 16 * w + fr < d) ? np[16 * w + fr] : 0.f;
  }
  // staging: thread = (channel sc and column sc of the block's 128, tokens 4 tg .. 4 tg + 3)
  const int sc = tid & 127, tg = tid >> 7;
  const bool chan = sc < d, scol = c0 + sc < dv;
  float bias = 0.f, low = 0.f;
  if (CHANNEL && chan) {
    bias = ldf((const S*)a.bias + h * d + sc);
    if (MODE == HGRN2) low = ldf((const S*)a.lower + h * d + sc);
  }
  const int goff = 2 * H * d + H * dv + h * dv + col;           // output gate
  const int ioff = 2 * H * d + 2 * H * dv + h;                  // MLSTM gates
  constexpr int GW = 7;                                         // the gate wave
  const int nb = (t1 - t0 + TB - 1) / TB;
  auto tokens = [&](int b) { return min(TB, t1 - t0 - b * TB); };
  float rq[4], rk[4], rz[4], rv[4], ra[4], gin = 0.f;
  auto load = [&](int b) {
    const int tc = t0 + b * TB, n = tokens(b);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = 4 * tg + u;
      rq[u] = rk[u] = rz[u] = rv[u] = 0.f;
      if (t < n) {
        const float* row = a.proj + (long)(tc + t) * a.ldp;
        if (chan) {
          rq[u] = row[h * d + sc];
          rk[u] = row[H * d + h * d + sc];
          if (MODE == GLA) rz[u] = a.z[(long)(tc + t) * a.ldz + h * d + sc];
        }
        if (scol) rv[u] = row[2 * H * d + h * dv + c0 + sc];
      }
    }
  };
  auto load_gates = [&](int b) {                // MLSTM: the gate wave's rows of 16 lanes, i | f | i | f
    if (MODE == MLSTM && w == GW && b < nb && fr < tokens(b))
      gin = a.proj[(long)(t0 + b * TB + fr) * a.ldp + ioff + (q & 1) * H];
  };
  // per-channel decays of the block in the registers, and their products over 4 tokens
  auto channel_gates = [&](int b) {
    const int n = tokens(b);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const bool real = 4 * tg + u < n && chan;
      if (MODE == HGRN2) {
        ra[u] = real ? low + (1.f - low) * sigmoid1(rk[u] + bias) : 1.f;
        rk[u] = real ? 1.f - ra[u] : 0.f;
      } else {
        ra[u] = real ? decay_pow(rz[u] + bias, a.inv_tau) : 1.f;
      }
    }
    if (sc < DP) cm.part[b & 1][tg][sc] = (ra[0] * ra[1]) * (ra[2] * ra[3]);
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
    const float y = a.cap * tanhf((gin + a.if_b[(q & 1) * H + h]) / a.cap);      // odd rows: forget gates
    const float ls = logsigmoid32(y);
    const float ig = fr < n ? __shfl(y, fr, 64) : -INFINITY;
    const float fg = fr < n ? __shfl(ls, 16 + fr, 64) : 0.f;
    float ft = 0.f, mt = 0.f;
#pragma unroll
    for (int t = 0; t < TB; ++t) {
      const float f = from_lane(fg, t) + m_run;
      m_run = fmaxf(f, from_lane(ig, t));
      ft = fr == t ? f : ft;
      mt = fr == t ? m_run : mt;
    }
    at = expf(ft - mt);
    bt = expf(ig - mt);
    em = expf(-mt);
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
  };
  // fixed decays: table 0 for full blocks, 1 for a shorter last one
  auto table = [&](int b) -> Gates& { return gm.g[MODE == FIXED ? int(tokens(b) < TB) : (b & 3)]; };
  // a block's LDS image from the registers
  auto stage = [&](int b) {
    const int buf = b & 1;
    f32x4 kb, vv;
    if (sc < DP) {
      if constexpr (CHANNEL) {
        float A[4], B[4], pre = 1.f, post = 1.f;
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const float px = cm.part[buf][x][sc];
          if (x < tg) pre *= px;
          if (x > tg) post *= px;
        }
        A[0] = pre * ra[0]; A[1] = A[0] * ra[1]; A[2] = A[1] * ra[2]; A[3] = A[2] * ra[3];
        B[3] = post; B[2] = B[3] * ra[3]; B[1] = B[2] * ra[2]; B[0] = B[1] * ra[1];
        const float G = A[3] * post;
        const bool bad = !(G >= MIN_DECAY);
        if (tg == 0) {
          cm.G[buf][sc] = G;
          const unsigned long long m = __ballot(bad);
          if (lane == 0) cm.bad[buf][w] = m;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int t = 4 * tg + u;
          const float qq = MODE == HGRN2 ? silu1(rq[u]) : rq[u] * a.qscale;
          sm.Q[buf][t * LQ + sc] = qq * A[u];
          sm.K[buf][t * LQ + sc] = bad ? 0.f : rk[u] * rcp1(A[u]);
          kb[u] = rk[u] * B[u];
          if (bad) {
            cm.raw[buf][sc][t] = qq;
            cm.raw[buf][sc][TB + t] = rk[u];
            cm.raw[buf][sc][2 * TB + t] = ra[u];
          }
        }
      } else {
        const f32x4 kw = *reinterpret_cast<const f32x4*>(table(b).kb + 4 * tg);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int t = 4 * tg + u;
          const float qq = MODE == FIXED ? silu1(rq[u]) : rq[u] * a.qscale;
          const float kk = MODE == FIXED ? silu1(rk[u]) : rk[u];
          sm.Q[buf][t * LQ + sc] = qq;
          sm.K[buf][t * LQ + sc] = kk;
          kb[u] = kk * kw[u];
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
  auto products = [&](int b) {
    const int buf = b & 1;
    const float* Q = sm.Q[buf];
    if (w < ND) {                               // this wave's 16 channels of P^T
      const f32x4 qf = *reinterpret_cast<const f32x4*>(Q + fr * LQ + 16 * w + 4 * q);
      const f32x4 kf = *reinterpret_cast<const f32x4*>(sm.K[buf] + fr * LQ + 16 * w + 4 * q);
      const f32x4 p = mfma4(kf, qf, f32x4{0.f, 0.f, 0.f, 0.f});
      *reinterpret_cast<f32x4*>(&sm.P[buf][w][4 * lane]) = p;
      if (MODE == MLSTM) {                      // n . q_i over them, then n after the block
        const f32x4 nf = *reinterpret_cast<const f32x4*>(gm.n + 16 * w + 4 * q);
        float x = (nf[0] * qf[0] + nf[1] * qf[1]) + (nf[2] * qf[2] + nf[3] * qf[3]);
        x += __shfl_xor(x, 16, 64);
        x += __shfl_xor(x, 32, 64);
        if (q == 0) gm.nq[buf][w][fr] = x;
        const f32x4 kb = *reinterpret_cast<const f32x4*>(sm.Kb[buf] + (16 * w + fr) * LT + 4 * q);
        float y = (kb[0] + kb[1]) + (kb[2] + kb[3]);
        y += __shfl_xor(y, 16, 64);
        y += __shfl_xor(y, 32, 64);
        if (q == 0) gm.n[16 * w + fr] = table(b).G[0] * gm.n[16 * w + fr] + y;
      }
    }
    if constexpr (CHANNEL) {
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
    if (wave_on) {
      vfn = *reinterpret_cast<const f32x4*>(sm.V[buf] + (16 * w + fr) * LT + 4 * q);
      f32x4 part[4];                            // short sums round less than one of d terms
#pragma unroll
      for (int t = 0; t < 4; ++t) part[t] = f32x4{0.f, 0.f, 0.f, 0.f};
      float Gs = 0.f, Gl = 0.f;
      if constexpr (!CHANNEL) Gs = table(b).G[0];
      if (MODE == FIXED) Gl = table(b).G[1];
#pragma unroll
      for (int t = 0; t < ND; ++t) {            // tile t's read-out and update side by side
        const f32x4 qf = *reinterpret_cast<const f32x4*>(Q + fr * LQ + 16 * t + 4 * q);
        const f32x4 kb = *reinterpret_cast<const f32x4*>(sm.Kb[buf] + (16 * t + fr) * LT + 4 * q);
        f32x4 sn;
        if constexpr (CHANNEL) sn = st[t] * *reinterpret_cast<const f32x4*>(cm.G[buf] + 16 * t + 4 * q);
        else sn = st[t] * Gs;
        if (MODE == FIXED) sn += st[t] * Gl;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          part[t & 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[r], st[t][r], part[t & 3], 0, 0, 0);
          sn = __builtin_amdgcn_mfma_f32_16x16x4f32(kb[r], vfn[r], sn, 0, 0, 0);
        }
        st[t] = sn;
      }
      accn = (part[0] + part[1]) + (part[2] + part[3]);
    }
  };
  f32x4 o = {0.f, 0.f, 0.f, 0.f}, gate = o;
  float nw = 0.f;
  if (MODE != FIXED && on) nw = ldf((const S*)a.norm_w + (MODE == MLSTM ? h * dv + col : col));
  // o = the read-outs of block b (rows 4 q + r, this lane's column) from vf, acc and P
  auto finish = [&](int b) {
    const int buf = b & 1;
    if (MODE == GLA || MODE == MLSTM) {
      const int n = tokens(b);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (on && 4 * q + r < n) gate[r] = a.proj[(long)(t0 + b * TB + 4 * q + r) * a.ldp + goff];
    }
    f32x4 p = {0.f, 0.f, 0.f, 0.f};             // P_ij, i = fr, j = 4 q + r
#pragma unroll
    for (int x = 0; x < ND; ++x) p += *reinterpret_cast<const f32x4*>(&sm.P[buf][x][4 * lane]);
    float inv = 0.f;
    if constexpr (CHANNEL) {
      const bool extra = (bad0 | bad1) != 0;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (extra) p[r] += cm.xP[buf][(4 * q + r) * 16 + fr];
        p[r] = 4 * q + r <= fr ? p[r] : 0.f;
      }
    } else {
      const Gates& gt = table(b);
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
    o = mfma4(p, vf, acc);
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
  auto write_out = [&](int b) {
    const int n = tokens(b);
    float rs = 0.f;
    if (MODE != FIXED) {                        // row fr's
      const float* sq = sm.ss[b & 1][fr];
      const f32x4 x = *reinterpret_cast<const f32x4*>(sq), y = *reinterpret_cast<const f32x4*>(sq + 4);
      rs = 1.f / sqrtf((((x[0] + x[1]) + (x[2] + x[3])) + ((y[0] + y[1]) + (y[2] + y[3]))) / (float)dv + a.eps);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 4 * q + r;
      const float rr = MODE != FIXED ? __shfl(rs, i, 64) : 0.f;
      if (i >= n || !on) continue;
      const long t = (long)t0 + b * TB + i;
      if (MODE == FIXED) {
        outf[t * a.ldo + h * dv + col] = o[r];
        continue;
      }
      float v = o[r] * rr * nw;
      if (MODE == GLA) v *= silu1(gate[r]);
      if (MODE == MLSTM) v *= sigmoid1(gate[r]) * a.out_scale;
      stf(out + t * a.ldo + h * dv + col, v);
    }
  };

  load(0);
  load_gates(0);
  if constexpr (CHANNEL) {
    channel_gates(0);
  } else if (w == GW) {
    scalar_gates(tokens(0), table(0));
    if (MODE == FIXED) {
      if (nb > 1) scalar_gates(tokens(nb - 1), table(nb - 1));
    } else if (nb > 1) {
      load_gates(1);
      scalar_gates(tokens(1), table(1));
    }
    load_gates(2);
  }
  __syncthreads();
  stage(0);
  if (nb > 1) {
    load(1);
    if constexpr (CHANNEL) channel_gates(1);
  }
  __syncthreads();
#pragma unroll 1
  for (int b = 0; b < nb + 2; ++b) {
    if (b + 1 < nb) stage(b + 1);
    if (b + 2 < nb) {
      load(b + 2);
      if (MODE == MLSTM && w == GW) {
        scalar_gates(tokens(b + 2), table(b + 2));
        load_gates(b + 3);
      }
    }
    if (w < 4 && b < nb) products(b);
    if (b >= 2) write_out(b - 2);
    if (b >= 1 && b <= nb) finish(b - 1);
    if (w >= 4 && b < nb) products(b);
    vf = vfn; acc = accn; bad0 = bad0n; bad1 = bad1n;
    if constexpr (CHANNEL) {
      if (b + 2 < nb) channel_gates(b + 2);
    }
    lds_barrier();
  }
  if (on) {
#pragma unroll
    for (int t = 0; t < ND; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int c = 16 * t + 4 * q + r;
        if (c < d) sp[(long)c * dv] = st[t][r];
      }
  }
  if (MODE == MLSTM) {
    if (w < ND && q == 0 && 16 * w + fr < d) np[16 * w + fr] = gm.n[16 * w + fr];
    if (w == GW && lane == 0) np[d] = m_run;
  }
}

template <typename S, int ND, int MODE>
int launch_chunks(const ChunkArgs& a, int num_seqs, hipStream_t st) {
  constexpr size_t sh = sizeof(Smem<ND>) + (MODE <= GLA ? sizeof(ChannelSmem<ND>) : sizeof(ScalarSmem<ND>));
  static_assert(sh <= 160 * 1024 && sizeof(Smem<ND>) % 16 == 0, "LDS image");
  if (sh > 48 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)recurrence_chunk_kernel<S, ND, MODE>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)sh);
    if (e != hipSuccess) return (int)e;
  }
  dim3 grid(a.H, num_seqs, (a.dv + COLS - 1) / COLS);
  recurrence_chunk_kernel<S, ND, MODE><<<grid, NTH, sh, st>>>(a);
  DLI_RETURN_LAUNCH();
}

template <typename S, int MODE>
int launch_by_width(const ChunkArgs& a, int num_seqs, hipStream_t st) {
  if (a.d <= 32) return launch_chunks<S, 2, MODE>(a, num_seqs, st);
  if (a.d <= 64) return launch_chunks<S, 4, MODE>(a, num_seqs, st);
  return launch_chunks<S, 8, MODE>(a, num_seqs, st);
}

}  // namespace

// Portions of a step's sequences (mode as above). hipErrorNotSupported: a size that the walk takes
// (d > 128, or a normed head wider than 128).
extern "C" int dli_recurrence_chunks(int mode, const float* proj, int ldp, const float* z, int ldz,
                                     const void* bias, const void* lower, float inv_tau, float qscale,
                                     const float* decays, const float* if_b, float cap,
                                     const void* norm_w, float eps, float* state, float* nstate,
                                     const int* slots, const int* cu, const int* positions, void* out,
                                     int ldo, float out_scale, int num_seqs, int H, int d, int dv,
                                     int dt, hipStream_t st) {
  if (num_seqs <= 0) return 0;
  if (H < 1 || d < 1 || dv < 1 || num_seqs > 65535 || state == nullptr || slots == nullptr ||
      out == nullptr || (dt != 0 && dt != 1))
    return (int)hipErrorInvalidValue;
  if (d > 128 || (mode != FIXED && dv > COLS)) return (int)hipErrorNotSupported;
  ChunkArgs a{proj, ldp, z, ldz, bias, lower, inv_tau, qscale, decays, if_b, cap, norm_w, eps, state,
              nstate, slots, cu, positions, out, ldo, out_scale, H, d, dv};
  switch (mode) {
    case HGRN2:
      if (bias == nullptr || lower == nullptr || norm_w == nullptr) break;
      return dt == 0 ? launch_by_width<u16, HGRN2>(a, num_seqs, st) : launch_by_width<float, HGRN2>(a, num_seqs, st);
    case GLA:
      if (z == nullptr || bias == nullptr || norm_w == nullptr) break;
      return dt == 0 ? launch_by_width<u16, GLA>(a, num_seqs, st) : launch_by_width<float, GLA>(a, num_seqs, st);
    case FIXED:
      if (decays == nullptr) break;
      return launch_by_width<float, FIXED>(a, num_seqs, st);
    case MLSTM:
      if (if_b == nullptr || norm_w == nullptr || nstate == nullptr || !(cap > 0.f)) break;
      return dt == 0 ? launch_by_width<u16, MLSTM>(a, num_seqs, st) : launch_by_width<float, MLSTM>(a, num_seqs, st);
  }
  return (int)hipErrorInvalidValue;
}
