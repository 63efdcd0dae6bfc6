// Persistent form of the 4-wave two-barrier 256x256 GEMM (tile 55; tile 45 = gemm4w_kernel
// <EPI, 8 | 4096> is its one-tile-per-workgroup form). Tile by tile the prefill
// projections pay, per 256x256 tile, a prologue (the first two K-tiles' LDS-DMA latency with
// the matrix pipe idle) and an epilogue (the 128-256 KB store tail) that a workgroup-per-tile
// grid cannot hide. Here one workgroup per CU walks tiles v = blockIdx.x, + gridDim.x, ...
// (the same virtual ids, XCD remap and GM-4 grouped order as tile 45, so the tiles in flight
// at any time are the ones a wave of tile 45's grid would run), and the two DMA windows of a
// tile's LAST two K-tiles — idle in tile 45 — stage K-tiles 0 and 1 of the workgroup's next
// tile. The epilogue's stores then drain while those DMAs fly, and the next tile starts with
// both of its first K-tiles in LDS.
//
// Restrictions (the launcher returns hipErrorInvalidValue and the planner never picks it
// otherwise): no split-K, no grouped (MoE) mode, K a multiple of 128 (an even K-tile count:
// the next tile's K-tiles 0 / 1 land in buffers 0 / 1, which the current tile's last two
// K-tiles have just released).
#include "gemm4w.h"

// NJ: tiles of 256 x 32 NJ (wave tiles of 128 x 16 NJ). The narrower ones are for the counts of tiles
// that 256 columns leave at little more than a round of the chip, or at little over half of one: see
// width_of(). Their schedule is the same with fewer MFMAs, W fragments and W pieces.
template <int EPI, int NJ>
__global__ void __launch_bounds__(256, 1) gemm4wp_kernel(
    const u16* __restrict__ A, int lda, const u16* __restrict__ W, int ldw,
    void* __restrict__ C, int ldc, int M, int N, int K, const u16* __restrict__ bias) {
  constexpr int BM = 256, BN = 32 * NJ, GM = 4;
  constexpr int A_BYTES = BM * BK * 2, BUF = A_BYTES + BN * BK * 2;
  constexpr int NF = 8 + NJ, NP = 8 + NJ;          // fragments of a half K-tile, DMA pieces a wave
  extern __shared__ __attribute__((aligned(16))) char smem[];

  const int tiles_m = (M + BM - 1) / BM;
  const int tiles_n = (N + BN - 1) / BN;
  const int nwg = tiles_m * tiles_n;
  const int nk = K / BK;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wid >> 1, wn = wid & 1;

  // virtual tile id -> (m0, n0): tile 45's XCD remap + GM-4 grouped order
  auto coords = [&](int v, int& m0, int& n0) {
    const int tile = xcd_remap(v, nwg);
    const int per_group = GM * tiles_n;
    const int first_m = (tile / per_group) * GM;
    const int gsz = min(tiles_m - first_m, GM);
    const int in_g = tile % per_group;
    m0 = (first_m + in_g % gsz) * BM;
    n0 = (in_g / gsz) * BN;
  };

  // ---- staging: piece f (0..NP-1) of K-tile kg of the tile whose operand panels start at
  // sa / sw (sab / swb bytes in range: rows past the matrix read as zeros) into buffer buf
  const int prow = 64 * wid + (lane >> 3), wprow = 8 * NJ * wid + (lane >> 3);
  const int ce = (lane & 7) ^ ((lane >> 4) & 7), co = (lane & 7) ^ (((lane >> 4) + 4) & 7);
  const int a_off[2] = {prow * lda * 2 + ce * 16, prow * lda * 2 + co * 16};
  // (a wave's W rows start at an odd multiple of 8 where NJ and the wave are odd)
  const bool flip = (NJ * wid) & 1;
  const int w_off[2] = {wprow * ldw * 2 + (flip ? co : ce) * 16, wprow * ldw * 2 + (flip ? ce : co) * 16};
  const u16* sa = A;
  const u16* sw = W;
  int sab = 0, swb = 0;
  auto set_stage = [&](int m0, int n0) {
    sa = A + (long)m0 * lda;
    sw = W + (long)n0 * ldw;
    sab = min(M - m0, BM) * lda * 2;
    swb = min(N - n0, BN) * ldw * 2;
  };
  auto stage_piece = [&](int kg, int buf, int f) {
    const int i = f & 7;
    if (f < 8)
      buf_lds16(sa, sab, smem + buf * BUF + (64 * wid + 8 * i) * 128, a_off[i & 1],
                i * 16 * lda + kg * (BK * 2));
    else
      buf_lds16(sw, swb, smem + buf * BUF + A_BYTES + (8 * NJ * wid + 8 * i) * 128, w_off[i & 1],
                i * 16 * ldw + kg * (BK * 2));
  };

  const int fr = lane & 15, fq = lane >> 4;
  auto read_frag = [&](const char* part, int row, int kk) -> bf16x8 {
    const int c = kk * 4 + fq;
    return *reinterpret_cast<const bf16x8*>(part + row * 128 + ((c ^ ((row >> 1) & 7)) << 4));
  };
  const int arow = wm * 128 + fr, wrow = wn * 16 * NJ + fr;
  auto abuf = [&](int kt) -> const char* { return smem + (kt & 1) * BUF; };
  auto wbuf = [&](int kt) -> const char* { return smem + (kt & 1) * BUF + A_BYTES; };

  auto barrier = [&]() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
  };

  f32x4 acc[8][NJ];
  bf16x8 a0[8], b0[NJ], a1[8], b1[NJ];
  auto read_f0 = [&](int kt) {       // kk = 0 fragments of K-tile kt (order A0, B0.., A1..)
    a0[0] = read_frag(abuf(kt), arow, 0);
#pragma unroll
    for (int j = 0; j < NJ; ++j) b0[j] = read_frag(wbuf(kt), wrow + 16 * j, 0);
#pragma unroll
    for (int i = 1; i < 8; ++i) a0[i] = read_frag(abuf(kt), arow + 16 * i, 0);
  };
  auto read_fx = [&](int f, bf16x8 (&av)[8], bf16x8 (&bv)[NJ], const char* pa, const char* pw,
                     int kk) __attribute__((always_inline)) {
    if (f >= 1 && f <= NJ) bv[f - 1] = read_frag(pw, wrow + 16 * (f - 1), kk);
    else { const int ia = f == 0 ? 0 : f - NJ; av[ia] = read_frag(pa, arow + 16 * ia, kk); }
  };

  // one K-tile of the two-barrier schedule (gemm4w.h ktile2): MFMAs 0-15 read F1(kt), B1
  // after MFMA 19, the DMA window (16 pieces over MFMAs 20-95) stages K-tile kg of the
  // staging panels into kt's buffer, B2 after MFMA 103 (vmcnt: the pieces just issued may
  // fly), MFMAs 104-119 read F0(kt+1). STG: this K-tile stages; MORE: a K-tile of the same
  // tile follows (B2 and the F0 reads).
  auto ktile = [&](auto STG, bool more, int kt, int kg) __attribute__((always_inline)) {
    constexpr bool stg = decltype(STG)::value;
    const char* ab = abuf(kt);
    const char* wb = wbuf(kt);
    const char* nab = abuf(kt + 1);
    const char* nwb = wbuf(kt + 1);
    constexpr int QB1 = NF + 3, QB2 = 16 * NJ - NF - 9, SP = (QB2 - QB1) / NP;
    static_assert(SP >= 1 && QB2 + NF < 16 * NJ, "the window fits the K-tile");
    auto step = [&](int q) __attribute__((always_inline)) {
      if (q < NF) {
        read_fx(q, a1, b1, ab, wb, 1);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (q == QB1) {
        __builtin_amdgcn_s_waitcnt(0xC07F);        // lgkmcnt(0)
        barrier();
      }
      if (stg && q > QB1 && q <= QB1 + SP * NP && (q - QB1 - 1) % SP == 0) {
        stage_piece(kg, kt & 1, (q - QB1 - 1) / SP);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (q == QB2 && more) {
        wait_vmcnt<stg ? NP : 0>();
        barrier();
      }
      if (more && q > QB2 && q <= QB2 + NF) {
        read_fx(q - QB2 - 1, a0, b0, nab, nwb, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int v = 0; v < NJ; ++v) {
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                     : "+a"(acc[u][v]) : "v"(b0[v]), "v"(a0[u]));
        step(NJ * u + v);
      }
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int v = 0; v < NJ; ++v) {
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                     : "+a"(acc[u][v]) : "v"(b1[v]), "v"(a1[u]));
        step(8 * NJ + NJ * u + v);
      }
  };
  auto vget = [&](const f32x4& a) -> f32x4 {
    f32x4 v;
    asm volatile("" : "=v"(v) : "0"(a));
    return v;
  };

  using T_ = std::integral_constant<bool, true>;
  using F_ = std::integral_constant<bool, false>;
  int v = blockIdx.x;
  if (v >= nwg) return;                              // wave-uniform: every wave exits
  int m0, n0;
  coords(v, m0, n0);
  set_stage(m0, n0);
  // prologue of the first tile: K-tiles 0 and 1 in flight, then F0 of K-tile 0
#pragma unroll
  for (int f = 0; f < NP; ++f) stage_piece(0, 0, f);
#pragma unroll
  for (int f = 0; f < NP; ++f) stage_piece(1, 1, f);
  wait_vmcnt<NP>();
  barrier();

  while (true) {                                     // every wave runs the same tiles
    const int vn = v + (int)gridDim.x;
    const bool has_next = vn < nwg;
    int mn = 0, nn = 0;
    if (has_next) coords(vn, mn, nn);
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // the zeroed accumulators are read by inline-asm MFMAs, which hipcc pads no hazard for:
    // pin every write ahead of a few wait states (gemm4w.h: nothing copies them in the loop)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) asm volatile("" : "+a"(acc[i][j]));
      asm volatile("s_nop 3");
    }
    read_f0(0);
    int kt = 0;
    for (; kt + 2 < nk; ++kt) ktile(T_{}, true, kt, kt + 2);
    // the last two K-tiles stage the next tile's K-tiles 0 and 1 (buffers 0 / 1: nk even).
    // Without a next tile they stage through an empty buffer range (no memory traffic, the
    // range check returns zeros): one code path — a branch here doubled the unrolled tail
    // and hipcc spilled the fragments (1 KB/lane of scratch)
    set_stage(mn, nn);
    sab = has_next ? sab : 0;
    swb = has_next ? swb : 0;
    ktile(T_{}, true, kt, 0);
    ktile(T_{}, false, kt + 1, 1);
    // MFMA results -> the epilogue's copies: XDL write-back wait states (gemm4w.h)
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int j = 0; j < NJ; ++j) asm volatile("" : "+a"(acc[7][j]));
    // ---- epilogue of tile (m0, n0), transposed accumulators:
    // acc[I][J][r] = C[m0 + 128 wm + 16I + fr][n0 + 16 NJ wn + 16J + 4fq + r]
    const int wr0 = m0 + 128 * wm, wc0 = n0 + 16 * NJ * wn;
    const bool vec = out_vec<EPI>(C, ldc, N, bias);
    if (epi_pairs(EPI)) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int row = wr0 + 16 * i + fr;
#pragma unroll
        for (int j = 0; j + 1 < NJ; j += 2) {
          const f32x4 g = vget(acc[i][j]), u = vget(acc[i][j + 1]);
          const int gcol = wc0 + 16 * j;
          if (row < M && gcol < N)
            store_pair_quad<EPI>(C, ldc, row, (gcol >> 5) * 16 + 4 * fq, g, u, vec);
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int row = wr0 + 16 * i + fr;
        BlockMax top;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const f32x4 val = vget(acc[i][j]);
          const int col = wc0 + 16 * j + 4 * fq;
          if (EPI == EPI_F32 && col < N) top.take(val);
          if (row < M && col < N) store_quad<EPI>(C, ldc, row, col, N, val, bias, vec);
        }
        if constexpr (EPI == EPI_F32)
          if (bias != nullptr) {                   // uniform: the block's largest value (BlockMax)
            const uint32_t key = row_key(top);
            if (fq == 0 && row < M && wc0 < N)
              ((uint32_t*)bias)[(long)row * ((N + 16 * NJ - 1) / (16 * NJ)) + wc0 / (16 * NJ)] = key;
          }
      }
    }
    // the next tile's K-tiles 0 and 1 (issued in the last two K-tiles) landed for every wave
    // (also before exiting: no LDS-DMA outlives the workgroup)
    wait_vmcnt<0>();
    if (!has_next) break;
    barrier();
    v = vn;
    m0 = mn;
    n0 = nn;
  }
}

static int cu_count() {
  static int cus = 0;
  if (!cus) {
    int dev = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (cus <= 0) cus = 256;
  }
  return cus;
}

// The tile width (8, 6 or 5 times 32 columns) whose rounds take least: a round's price is its width times
// what the narrower schedule costs more (fewer MFMAs between the same barriers: 9 and 13 %), the last one's
// by how many CUs it keeps, and little less for few of them, which clock higher. 256 columns unless
// another is 3 % better. (7 is hardly ever best, and then by as little.) N = 4096, one weight again and again, us at 8 /
// 7 / 6 / 5 (four weights in turn, as in a step: 4352 rows, K = 14336 551 and 412, K = 4096 163 and 125): 2304 rows, K = 14336 241 / 226 / 218 / 202,
// K = 4096 83 / 79 / 74 / 65; 4352 rows 535 / 476 / 424 / 402 and 164 / 149 / 136 / 127; 5120 rows 168 / 153 /
// 149 / 175; 8192 rows, two whole rounds at 8, 195 / 240 / 224 / 240. N = 6144, K = 4096: 2816 rows 164 / 149 /
// 134 / 121, 4096 rows 172 / 159 / 157 / 182. ops/gemm.py's persistent_width is its copy.
static int width_of(int M, int N, bool pairs) {
  const double cus = cu_count();
  const double price[9] = {0, 0, 0, 0, 0, 1.13 * 5 / 8, 1.09 * 6 / 8, 0, 1.0};
  int best = 8;
  double least = 0.0;
  for (int nj = 8; nj >= 5; --nj) {
    if (nj == 7 || (pairs && nj & 1)) continue;
    const long tiles = (long)((M + 255) / 256) * ((N + 32 * nj - 1) / (32 * nj));
    const double whole = (double)(tiles / (long)cus), x = tiles / cus - whole;
    const double last = x == 0 ? 0.0 : whole == 0 ? 0.8 + 0.2 * x * x * x
                                                  : 0.66 + 0.25 * x + 0.09 * x * x * x;
    const double c = (whole + last) * price[nj];
    if (nj == 8) least = 0.97 * c;
    else if (c < least) { least = c; best = nj; }
  }
  return best;
}

template <int EPI, int NJ>
static int launch_4wp_width(const void* A, int lda, const void* W, int ldw, void* C, int ldc, int M,
                            int N, int K, const void* bias, hipStream_t st) {
  constexpr size_t lds = 2 * (size_t)(256 + 32 * NJ) * BK * 2;
  static bool raised = false;
  if (!raised) {
    hipFuncSetAttribute((const void*)gemm4wp_kernel<EPI, NJ>,
                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    raised = true;
  }
  const int cus = cu_count();
  const int tiles = ((M + 255) / 256) * ((N + 32 * NJ - 1) / (32 * NJ));
  // one workgroup per CU (over 80 KiB of LDS each); a multiple of 8 keeps every workgroup's
  // virtual tile ids on one XCD residue class, as tile 45's grid places them
  int grid = tiles < cus ? tiles : (cus / 8) * 8;
  if (grid < 1) grid = 1;
  gemm4wp_kernel<EPI, NJ><<<grid, 256, lds, st>>>((const u16*)A, lda, (const u16*)W, ldw, C, ldc,
                                                  M, N, K, (const u16*)bias);
  DLI_RETURN_LAUNCH();
}

template <int EPI>
static int launch_4wp(const void* A, int lda, const void* W, int ldw, void* C, int ldc, int M,
                      int N, int K, int splits, const void* bias, const int* group_off,
                      hipStream_t st) {
  if (splits != 1 || group_off != nullptr || K % (2 * BK) || C == nullptr ||
      (epi_pairs(EPI) && N % 32))
    return (int)hipErrorInvalidValue;
  // (the biased epilogues, which the plans give to other tiles, keep one width)
  const int nj = EPI == EPI_BIAS || EPI == EPI_BIAS_GELU ? 8 : width_of(M, N, epi_pairs(EPI));
#define DLI_4WP(NJ) return launch_4wp_width<EPI, NJ>(A, lda, W, ldw, C, ldc, M, N, K, bias, st)
  if constexpr (EPI != EPI_BIAS && EPI != EPI_BIAS_GELU) {
    if (nj == 6) DLI_4WP(6);
    if constexpr (!epi_pairs(EPI)) {
      if (nj == 5) DLI_4WP(5);
    }
  }
  DLI_4WP(8);
#undef DLI_4WP
}

template <int EPI>
static int dispatch_4wp(int tile_cfg, DLI_GEMM_ARGS) {
  (void)ws;
  (void)groups;
  if (tile_cfg != 55) return DLI_NOT_MINE;
  return launch_4wp<EPI>(A, lda, W, ldw, C, ldc, M, N, K, splits, bias, go, st);
}

int gemm_4wp_dispatch(int epi, int tile_cfg, DLI_GEMM_ARGS) {
  if (epi == EPI_GELU_MUL) return dispatch_4wp<EPI_GELU_MUL>(tile_cfg, DLI_GEMM_PASS);
  DLI_EPI_SWITCH_BASE(dispatch_4wp)
}

// the columns of the tiles that the persistent kernel takes for a product
extern "C" int dli_gemm_persistent_width(int M, int N, int pairs) { return 32 * width_of(M, N, pairs != 0); }
