// Row kernels of the hyper-connected designs (models/hybrid.py, ops/hybrid.py). S = storage
// type (u16 = bf16 bits, or float); the streams, norms and sums are fp32.
//
//  * hyper_mix     hyper-connections over ns copies of the residual stream, xs [T, ns, dim]:
//                  with a finished sublayer's output y and its vector prev = [read | write |
//                  mix] (ns + ns + ns*ns floats, mix indexed [from, to]) every stream becomes
//                      xs[r] = sum_s mix[s][r] xs[s] + write[r] * y          (all r at once)
//                  and with the next sublayer's read weights the row u = sum_s read[s] xs[s]
//                  leaves RMS-normed times (w + w_offset) as S, or as it is in fp32 (w null).
//                  One launch does a sublayer's write-back and the next one's read + norm. Two
//                  finished sublayers may be handed over at once: the first one's write-back is
//                  then formed again on the way instead of having been stored. The streams may
//                  come from another array than they go to, also from one row for all of them.
//  * sink_prepare  q / k RMS-normed over their whole rows (all heads at once) with a weight
//                  per column, the first rot_dims dims of every head rotated (dimension i with
//                  i + rot_dims/2; angle = position * freq[i] formed in double; cos and sin
//                  times mscale), k and v -> cache rows, q -> S
#include "common.h"

namespace {

template <typename S> __device__ __forceinline__ float ldf(const S* p);
template <> __device__ __forceinline__ float ldf<u16>(const u16* p) { return bf2f(*p); }
template <> __device__ __forceinline__ float ldf<float>(const float* p) { return *p; }
template <typename S> __device__ __forceinline__ void stf(S* p, float v);
template <> __device__ __forceinline__ void stf<u16>(u16* p, float v) { *p = f2bf(v); }
template <> __device__ __forceinline__ void stf<float>(float* p, float v) { *p = v; }

constexpr int MAXS = 8;          // streams

// One workgroup per token (256 threads; 1024 for the few wide rows of a decode step, which
// are bound by latency). VEC = 4: 16-byte accesses of the fp32 rows (dim % 4 == 0). NS: the number of
// streams in the 16-byte form (0: any). y may be nsplit partial sums, ysplit elements apart, of a
// split-K product: the launch and the pass of its reduce are spared. The coefficients are the same
// for the whole launch: read as scalars, beside the rows' requests and without a barrier before them.
// With the number known, 512 rows of 4096: 1 stream 14.6 -> 9.5 us, 5 29.9 ->
// 23.9, 8 43.8 -> 32.9.
// Decode step, 64 rows of 3 x 4096: 7.5 us with a reduce launch of 5.4 before it -> 6.2. Prefill is bound
// by memory: 8199 rows 199 us with the streams stored, 126 without, 5.1 and 4.8 TB/s; two mixes of which
// one stores 397 -> 350 us. The outputs of sublayers are read and the streams stored past the caches, which
// neither meets again: a mix in a step 125 -> 114 us.
// y0 / prev0 (nullable): the sublayer before y's, whose write-back was not stored (xs null then).
// src: the streams' rows, src_row floats a token and src_stream a stream (0: one row for all).
template <typename S, int VEC, int NS>
__global__ void __launch_bounds__(1024) hyper_mix_kernel(
    const float* src, long src_row, long src_stream, float* xs,
    const float* __restrict__ y0, const float* __restrict__ prev0, const float* __restrict__ y,
    int ldy, int nsplit, long ysplit, const float* __restrict__ prev,
    const float* __restrict__ read, const S* __restrict__ w,
    void* __restrict__ h, int ns_any, int dim, float eps, float w_offset) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  constexpr int MS = NS ? NS : MAXS;
  const int ns = NS ? NS : ns_any;
  float* urow = sm;                        // [dim]
  float* red = urow + dim;                 // [16]
  const int t = blockIdx.x;
  const float* xi = src + t * src_row;
  float* xo = xs == nullptr ? nullptr : xs + (long)t * ns * dim;
  float ss = 0.f;
  for (int c = threadIdx.x * VEC; c < dim; c += blockDim.x * VEC) {
    float x[MS][VEC];
#pragma unroll
    for (int s = 0; s < MS; ++s) {
      if (s < ns) {
        if (VEC == 4) {
          const f32x4 v = *reinterpret_cast<const f32x4*>(xi + s * src_stream + c);
#pragma unroll
          for (int u = 0; u < VEC; ++u) x[s][u] = v[u];
        } else {
          x[s][0] = xi[s * src_stream + c];
        }
      }
    }
    // x <- the streams mixed by a sublayer's vector, plus its output (the same sums whether they
    // are formed once and stored or formed again)
    const auto write_back = [&](const float* vec, const float (&yv)[VEC]) {
      const float* wr = vec + ns;          // write weights
      const float* mix = vec + 2 * ns;     // [from][to]
      float nx[MS][VEC];
#pragma unroll
      for (int r = 0; r < MS; ++r)
        if (r < ns) {
#pragma unroll
          for (int u = 0; u < VEC; ++u) {
            float acc = 0.f;
#pragma unroll
            for (int s = 0; s < MS; ++s)
              if (s < ns) acc += mix[s * ns + r] * x[s][u];
            nx[r][u] = acc + wr[r] * yv[u];
          }
        }
#pragma unroll
      for (int r = 0; r < MS; ++r)
        if (r < ns) {
#pragma unroll
          for (int u = 0; u < VEC; ++u) x[r][u] = nx[r][u];
        }
    };
    if (y0 != nullptr) {
      float yv[VEC];
      if constexpr (VEC == 4) {
        const f32x4 v = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(y0 + (long)t * dim + c));
#pragma unroll
        for (int u = 0; u < VEC; ++u) yv[u] = v[u];
      } else {
        yv[0] = y0[(long)t * dim + c];
      }
      write_back(prev0, yv);
    }
    if (y != nullptr) {
      float yv[VEC];
      const float* yr = y + (long)t * ldy + c;
      if constexpr (VEC == 4) {
        f32x4 v = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(yr));
        for (int s = 1; s < nsplit; ++s) v += *reinterpret_cast<const f32x4*>(yr + s * ysplit);
#pragma unroll
        for (int u = 0; u < VEC; ++u) yv[u] = v[u];
      } else {
        yv[0] = yr[0];
        for (int s = 1; s < nsplit; ++s) yv[0] += yr[s * ysplit];
      }
      write_back(prev, yv);
    }
    if (xo != nullptr) {
#pragma unroll
      for (int r = 0; r < MS; ++r)
        if (r < ns) {
          if (VEC == 4)
            __builtin_nontemporal_store(
                f32x4{x[r][0], x[r][VEC > 1 ? 1 : 0], x[r][VEC > 2 ? 2 : 0], x[r][VEC > 3 ? 3 : 0]},
                reinterpret_cast<f32x4*>(xo + (long)r * dim + c));
          else
            xo[(long)r * dim + c] = x[r][0];
        }
    }
    if (read != nullptr) {
#pragma unroll
      for (int u = 0; u < VEC; ++u) {
        float acc = 0.f;
#pragma unroll
        for (int s = 0; s < MS; ++s)
          if (s < ns) acc += read[s] * x[s][u];
        if (w == nullptr) ((float*)h)[(long)t * dim + c + u] = acc;
        else urow[c + u] = acc;
        ss += acc * acc;
      }
    }
  }
  if (read == nullptr || w == nullptr) return;
  const float tot = block_sum(ss, red);
  const float rs = 1.f / sqrtf(tot / (float)dim + eps);
  if (VEC == 4 && ((uintptr_t)h | (uintptr_t)w) % 16 == 0) {
    for (int c = threadIdx.x * 4; c < dim; c += blockDim.x * 4) {
      f32x4 v = *reinterpret_cast<const f32x4*>(urow + c);
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = v[u] * rs * (ldf(w + c + u) + w_offset);
      st4((S*)h + (long)t * dim + c, v);
    }
    return;
  }
  for (int c = threadIdx.x; c < dim; c += blockDim.x)
    stf((S*)h + (long)t * dim + c, urow[c] * rs * (ldf(w + c) + w_offset));
}

// One workgroup per token. proj row (fp32): [H*d q | G*d k | G*dv v | ...].
template <typename S>
__global__ void __launch_bounds__(1024) sink_prepare_kernel(
    const float* __restrict__ proj, int ldp, const S* __restrict__ qw, const S* __restrict__ kw,
    float eps, int H, int G, int d, int dv, int rot, const double* __restrict__ freq,
    float mscale, const int* __restrict__ positions, S* __restrict__ q_out,
    S* __restrict__ kcache, S* __restrict__ vcache, const int* __restrict__ slots) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int nq = H * d, nk = G * d, hr = rot >> 1;
  float* row = sm;                         // [nq + nk] normed q | k
  float* cs = row + nq + nk;               // [rot / 2]
  float* sn = cs + hr;                     // [rot / 2]
  float* red = sn + hr;                    // [16]
  const int t = blockIdx.x;
  const float* pr = proj + (long)t * ldp;
  float sq = 0.f, sk = 0.f;
  for (int c = threadIdx.x; c < nq + nk; c += blockDim.x) {
    const float v = pr[c];
    row[c] = v;
    if (c < nq) sq += v * v; else sk += v * v;
  }
  const double pos = (double)positions[t];
  for (int i = threadIdx.x; i < hr; i += blockDim.x) {
    const double a = pos * freq[i];
    cs[i] = (float)(cos(a) * (double)mscale);
    sn[i] = (float)(sin(a) * (double)mscale);
  }
  const float tq = block_sum(sq, red);
  const float tk = block_sum(sk, red);
  const float rq = 1.f / sqrtf(tq / (float)nq + eps), rk = 1.f / sqrtf(tk / (float)nk + eps);
  for (int c = threadIdx.x; c < nq + nk; c += blockDim.x)
    row[c] = c < nq ? row[c] * rq * ldf(qw + c) : row[c] * rk * ldf(kw + c - nq);
  __syncthreads();
  const int slot = slots[t];
  for (int c = threadIdx.x; c < nq + nk; c += blockDim.x) {
    const int j = (c < nq ? c : c - nq) % d;
    float v = row[c];
    if (j < rot) {
      const bool second = j >= hr;
      const int i = second ? j - hr : j;
      const float other = row[second ? c - hr : c + hr];
      v = second ? v * cs[i] + other * sn[i] : v * cs[i] - other * sn[i];
    }
    if (c < nq) stf(q_out + (long)t * nq + c, v);
    else if (slot >= 0) stf(kcache + (long)slot * nk + (c - nq), v);
  }
  if (slot >= 0)
    for (int c = threadIdx.x; c < G * dv; c += blockDim.x)
      stf(vcache + (long)slot * G * dv + c, pr[nq + nk + c]);
}

// the same for widths of whole 16-byte pieces (rot a multiple of 8: a piece's partner is a piece),
// 4 columns a thread. 8199 tokens of 32 + 8 heads of 128 (0.3 GB): 167 -> 88 us.
template <typename S>
__global__ void __launch_bounds__(1024) sink_prepare4_kernel(
    const float* __restrict__ proj, int ldp, const S* __restrict__ qw, const S* __restrict__ kw,
    float eps, int H, int G, int d, int dv, int rot, const double* __restrict__ freq,
    float mscale, const int* __restrict__ positions, S* __restrict__ q_out,
    S* __restrict__ kcache, S* __restrict__ vcache, const int* __restrict__ slots) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int nq = H * d, nk = G * d, hr = rot >> 1;
  float* row = sm;                         // [nq + nk] q | k
  float* cs = row + nq + nk;               // [rot / 2]
  float* sn = cs + hr;                     // [rot / 2]
  float* red = sn + hr;                    // [16]
  const long t = blockIdx.x;
  const float* pr = proj + t * ldp;
  float sq = 0.f, sk = 0.f;
#pragma unroll 5
  for (int c = threadIdx.x * 4; c < nq + nk; c += blockDim.x * 4) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(pr + c);
    *reinterpret_cast<f32x4*>(row + c) = v;
    const float x = (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
    if (c < nq) sq += x; else sk += x;
  }
  const double pos = (double)positions[t];
  for (int i = threadIdx.x; i < hr; i += blockDim.x) {
    const double a = pos * freq[i];
    cs[i] = (float)(cos(a) * (double)mscale);
    sn[i] = (float)(sin(a) * (double)mscale);
  }
  const float tq = block_sum(sq, red);
  const float tk = block_sum(sk, red);
  const float rq = 1.f / sqrtf(tq / (float)nq + eps), rk = 1.f / sqrtf(tk / (float)nk + eps);
  const int slot = slots[t];
  const auto normed = [&](int c) {         // the norm's weight, as it is rounded before the rotation
    f32x4 v = *reinterpret_cast<const f32x4*>(row + c);
    const S* w = c < nq ? qw + c : kw + c - nq;
    const float r = c < nq ? rq : rk;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = v[i] * r * ldf(w + i);
    return v;
  };
  for (int c = threadIdx.x * 4; c < nq + nk; c += blockDim.x * 4) {
    if (c >= nq && slot < 0) break;
    const int j = (c < nq ? c : c - nq) % d;
    f32x4 v = normed(c);
    if (j < rot) {
      const bool second = j >= hr;
      const int i = second ? j - hr : j;
      const f32x4 other = normed(second ? c - hr : c + hr);
      const f32x4 co = *reinterpret_cast<const f32x4*>(cs + i), si = *reinterpret_cast<const f32x4*>(sn + i);
      v = second ? v * co + other * si : v * co - other * si;
    }
    if (c < nq) st4(q_out + t * nq + c, v);
    else st4(kcache + (long)slot * nk + (c - nq), v);
  }
  if (slot >= 0)
    for (int c = threadIdx.x * 4; c < G * dv; c += blockDim.x * 4)
      st4(vcache + (long)slot * G * dv + c, *reinterpret_cast<const f32x4*>(pr + nq + nk + c));
}

}  // namespace

#define DT_SWITCH2(dt, A, B)                      \
  do {                                            \
    if ((dt) == 0) { A; }                         \
    else if ((dt) == 1) { B; }                    \
    else return (int)hipErrorInvalidValue;        \
  } while (0)

// src: the streams' rows ([T, ns, dim], or with one_row [T, dim] read as every stream); xs: where the
// new streams go (src itself, another array, or null: not stored). y0 (contiguous) with prev0: a
// finished sublayer whose write-back is not in src yet; y with prev: the one after it, nsplit slabs,
// ysplit elements apart, whose sum is its output (1: the output itself).
extern "C" int dli_hyper_mix(const float* src, int one_row, float* xs, const float* y0,
                             const float* prev0, const float* y, int ldy, int nsplit, long ysplit,
                             const float* prev, const float* read, const void* w, void* h, int T,
                             int ns, int dim, float eps, float w_offset, int dt, hipStream_t st) {
  if (T <= 0) return 0;
  if (ns < 1 || ns > MAXS || dim < 1 || (y != nullptr) != (prev != nullptr) || nsplit < 1 ||
      (y0 != nullptr) != (prev0 != nullptr) || src == nullptr || (one_row && src == xs) ||
      (read != nullptr && h == nullptr) || (read == nullptr && xs == nullptr))
    return (int)hipErrorInvalidValue;
  const size_t sh = ((size_t)dim + 16) * 4;
  if (sh > 60000) return (int)hipErrorInvalidValue;
  const bool v4 = dim % 4 == 0 &&
                  (((uintptr_t)src | (uintptr_t)xs | (uintptr_t)y0 | (uintptr_t)y) & 15) == 0 &&
                  (y == nullptr || (ldy % 4 == 0 && ysplit % 4 == 0));
  const int nt = (T <= 1024 && dim >= 2048) ? 1024 : 256;
  const long row = one_row ? dim : (long)ns * dim, stream = one_row ? 0 : dim;
#define HM_LAUNCH(S, V, N)                                                                    \
  hyper_mix_kernel<S, V, N><<<T, nt, sh, st>>>(src, row, stream, xs, y0, prev0, y, ldy, nsplit, \
                                               ysplit, prev, read, (const S*)w, h, ns, dim, eps, \
                                               w_offset)
#define HM_STREAMS(S)                                                                         \
  (ns == 1 ? (void)HM_LAUNCH(S, 4, 1) : ns == 2 ? (void)HM_LAUNCH(S, 4, 2)                     \
   : ns == 3 ? (void)HM_LAUNCH(S, 4, 3) : ns == 4 ? (void)HM_LAUNCH(S, 4, 4)                   \
   : ns == 5 ? (void)HM_LAUNCH(S, 4, 5) : ns == 6 ? (void)HM_LAUNCH(S, 4, 6)                   \
   : ns == 7 ? (void)HM_LAUNCH(S, 4, 7) : (void)HM_LAUNCH(S, 4, 8))
  if (v4) DT_SWITCH2(dt, HM_STREAMS(u16), HM_STREAMS(float));
  else DT_SWITCH2(dt, (HM_LAUNCH(u16, 1, 0)), (HM_LAUNCH(float, 1, 0)));
#undef HM_STREAMS
#undef HM_LAUNCH
  DLI_RETURN_LAUNCH();
}

extern "C" int dli_sink_prepare(const float* proj, int ldp, const void* qw, const void* kw,
                                float eps, int T, int H, int G, int d, int dv, int rot_dims,
                                const double* freq, float mscale, const int* positions,
                                void* q_out, void* kcache, void* vcache, const int* slots, int dt,
                                hipStream_t st) {
  if (T <= 0) return 0;
  if (H < 1 || G < 1 || H % G || d < 1 || dv < 1 || rot_dims < 0 || (rot_dims & 1) ||
      rot_dims > d || (rot_dims > 0 && freq == nullptr))
    return (int)hipErrorInvalidValue;
  const size_t sh = ((size_t)(H + G) * d + rot_dims + 16) * 4;
  if (sh > 60000) return (int)hipErrorInvalidValue;
  const int nt = (T <= 1024 && (H + G) * d >= 2048) ? 1024 : 256;
  if (d % 4 == 0 && dv % 4 == 0 && rot_dims % 8 == 0 && ldp % 4 == 0 &&
      (((uintptr_t)proj | (uintptr_t)q_out | (uintptr_t)kcache | (uintptr_t)vcache) & 15) == 0) {
    DT_SWITCH2(dt,
               (sink_prepare4_kernel<u16><<<T, nt, sh, st>>>(
                   proj, ldp, (const u16*)qw, (const u16*)kw, eps, H, G, d, dv, rot_dims, freq,
                   mscale, positions, (u16*)q_out, (u16*)kcache, (u16*)vcache, slots)),
               (sink_prepare4_kernel<float><<<T, nt, sh, st>>>(
                   proj, ldp, (const float*)qw, (const float*)kw, eps, H, G, d, dv, rot_dims, freq,
                   mscale, positions, (float*)q_out, (float*)kcache, (float*)vcache, slots)));
    DLI_RETURN_LAUNCH();
  }
  DT_SWITCH2(dt,
             (sink_prepare_kernel<u16><<<T, nt, sh, st>>>(
                 proj, ldp, (const u16*)qw, (const u16*)kw, eps, H, G, d, dv, rot_dims, freq,
                 mscale, positions, (u16*)q_out, (u16*)kcache, (u16*)vcache, slots)),
             (sink_prepare_kernel<float><<<T, nt, sh, st>>>(
                 proj, ldp, (const float*)qw, (const float*)kw, eps, H, G, d, dv, rot_dims, freq,
                 mscale, positions, (float*)q_out, (float*)kcache, (float*)vcache, slots)));
  DLI_RETURN_LAUNCH();
}
