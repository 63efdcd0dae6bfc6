"""The matrix memory's one-token kernel, run on the CPU thread by thread: whatever the order in which threads
reach a barrier, no word of the state may be stored before every thread has loaded it."""
import ctypes
import re
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

SOURCE = Path(__file__).resolve().parents[1] / "csrc" / "kernels" / "recurrent_scalar.hip"
CLANG = shutil.which("clang++", path="/opt/rocm/llvm/bin:/opt/rocm/bin") or shutil.which("clang++")

# 256 threads as contexts of their own; one runs until it meets a barrier or a sum over its wave
HOST = r"""
#include <cmath>
#include <cstdlib>
#include <ucontext.h>
using u16 = unsigned short;
typedef float f32x4 __attribute__((ext_vector_type(4)));
#define __device__
#define __global__ static
#define __forceinline__ inline
#define __shared__ static
#define __launch_bounds__(n)
struct Index { int x, y, z; };
static Index threadIdx, blockIdx;
static const int N = 256;
enum { READY, BARRIER, WAVE, DONE };
static ucontext_t home, at[N];
static int state[N], turn[N];
static float waves[2][N];
static void leave(int why) {
  const int t = threadIdx.x;
  state[t] = why;
  swapcontext(&at[t], &home);
}
static void __syncthreads() { leave(BARRIER); }
static float wave_sum(float v) {
  const int t = threadIdx.x, k = turn[t]++ & 1;
  waves[k][t] = v;
  leave(WAVE);
  float sum = 0.f;
  for (int l = 0; l < 64; ++l) sum += waves[k][(t & ~63) + l];
  return sum;
}
template <typename S> float ldf(const S* p) { return *p; }
template <typename S> void stf(S* p, float v) { *p = v; }
KERNEL
static ScalarRecArgs args;
static void body() {
  scalar_step_kernel<float, 64, 1>(args);
  leave(DONE);
}
extern "C" int run(const float* proj, const float* if_b, const float* norm_w, float* state_, float* nstate,
                   const int* ints, float* out, int descending) {
  args = ScalarRecArgs{};
  args.proj = proj; args.ldp = 4 * 64 + 2; args.if_b = if_b; args.cap = 15.f; args.norm_w = norm_w;
  args.eps = 1e-5f; args.state = state_; args.nstate = nstate; args.cu = ints; args.slots = ints + 2;
  args.positions = ints + 3; args.out = out; args.ldo = 64; args.out_scale = 1.f; args.H = 1;
  args.d = args.dv = args.cw = 64;
  blockIdx = Index{0, 0, 0};
  for (int t = 0; t < N; ++t) {
    getcontext(&at[t]);
    at[t].uc_stack.ss_size = 1 << 16;
    at[t].uc_stack.ss_sp = malloc(1 << 16);
    makecontext(&at[t], body, 0);
    state[t] = READY;
    turn[t] = 0;
  }
  const auto all = [](int from, int to, int why) {       // every thread that is not through waits here
    bool any = false;
    for (int t = from; t < to; ++t) {
      if (state[t] != why && state[t] != DONE) return false;
      any |= state[t] == why;
    }
    return any;
  };
  for (bool moved = true; moved;) {
    moved = false;
    for (int i = 0; i < N; ++i) {
      const int t = descending ? N - 1 - i : i, w = t & ~63;
      if (state[t] != READY) continue;
      threadIdx.x = t;
      swapcontext(&home, &at[t]);
      moved = true;
      if (all(w, w + 64, WAVE))
        for (int l = w; l < w + 64; ++l) state[l] = state[l] == DONE ? DONE : READY;
    }
    if (all(0, N, BARRIER)) {
      for (int t = 0; t < N; ++t) state[t] = state[t] == DONE ? DONE : READY;
      moved = true;
    }
  }
  int left = 0;
  for (int t = 0; t < N; ++t) {
    left += state[t] != DONE;
    free(at[t].uc_stack.ss_sp);
  }
  return left;
}
"""


def _library(tmp_path):
    text = SOURCE.read_text()
    parts = [re.search(p, text, re.S).group(0) for p in (
        r"__device__ __forceinline__ float silu32.*?\n(?=\n// tokens per chunk)", r"struct ScalarRecArgs \{.*?\n\};\n",
        r"template <typename S, int D, int FORM>\n__global__ .*?scalar_step_kernel.*?\n\}\n")]
    src, lib = tmp_path / "step.cpp", tmp_path / "step.so"
    src.write_text(HOST.replace("KERNEL", "\n".join(parts)))
    subprocess.run([CLANG, "-std=c++17", "-O1", "-w", "-fPIC", "-shared", str(src), "-o", str(lib)], check=True)
    return ctypes.CDLL(str(lib))


@pytest.mark.skipif(CLANG is None, reason="needs clang++ (vector types)")
def test_the_running_maximum_is_stored_when_every_thread_has_read_it(tmp_path):
    lib, d, rng = _library(tmp_path), 64, np.random.default_rng(5)
    f32 = np.float32
    row, if_b = rng.standard_normal(4 * d + 2).astype(f32), np.array([0.3, -0.2], f32)
    norm = rng.standard_normal(d).astype(f32)
    state, n, m = rng.standard_normal((d, d)).astype(f32), rng.standard_normal(d).astype(f32), f32(2.5)
    ints = np.array([0, 1, 0, 7], np.int32)              # one token: rows [0, 1), slot 0, position 7
    # float64
    q, k, v, g = (row[i * d:(i + 1) * d].astype(np.float64) for i in range(4))
    q = q / np.sqrt(d)
    gate = 15.0 * np.tanh((row[4 * d:].astype(np.float64) + if_b) / 15.0)
    i, f = gate[0], -np.log1p(np.exp(-gate[1]))
    m1 = max(f + m, i)
    at, bt = np.exp(f + m - m1), np.exp(i - m1)
    new, n1 = at * state + bt * np.outer(k, v), at * n + bt * k
    o = (new.T @ q) / (max(abs(n1 @ q), np.exp(-m1)) + 1e-6)
    want = o / np.sqrt((o * o).mean() + 1e-5) * norm / (1.0 + np.exp(-g))
    for descending in (0, 1):
        s, ns, out = state.copy(), np.append(n, m).astype(f32), np.zeros(d, f32)
        p = [a.ctypes.data_as(ctypes.c_void_p) for a in (row, if_b, norm, s, ns, ints, out)]
        assert lib.run(*p, descending) == 0              # every thread came to its end
        # sums of 64 fp32 products
        np.testing.assert_allclose(s, new, rtol=1e-5, atol=1e-5)
        np.testing.assert_allclose(ns, np.append(n1, m1), rtol=1e-5, atol=1e-5)
        np.testing.assert_allclose(out, want, rtol=1e-4, atol=1e-5)
