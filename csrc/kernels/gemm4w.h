// GEMM tiles of 32 MI x 32 NJ (256 rows, MI = 8, where a comment says no other) with ONE wave per SIMD: four waves of
// 16 MI x 16 NJ, their MI NJ 16x16 blocks accumulated in the AGPR file, on a grid of at most one workgroup a CU that
// walks its tiles (tiles 22, 28, 34, 41, 45 and 55: gemm4w.hip).
//
// What bounds it. Bare 16x16x32 MFMAs on random data run at 2.0 GHz (2.07 PFLOP/s), which the power
// budget sets; with this tile's 32 fragment reads and 16 LDS-DMA pieces a K-tile at 1.75 GHz and 17.6
// cycles an MFMA (1.68, operands in the L2). So what costs is (a) cycles in which the matrix pipe waits
// and (b) energy beside the MFMAs; a cycle saved gives about 0.6 of itself, the clock gives the rest back.
// 32x32x16 MFMAs, half the instructions, hold 1.73 GHz and 1.81 PFLOP/s alone: not used. The order in which a wave
// takes its blocks (Walk4w) is about (b) alone.
//
// (a) is this schedule's business; measured amid MFMAs of 16 cycles, one wave a SIMD: an LDS-DMA piece
// costs 2 to 4 cycles, every scalar instruction beside it 4, vector ones nothing. So a lane's offsets advance by
// vector adds, four pieces share M0 through their immediate offsets (which move the address in memory and in LDS
// alike: the soffset takes them back), and the pieces are spread as thinly as the ring of two buffers allows (K =
// 14336: 1.43 PFLOP/s with a piece every 4 MFMAs, 1.54 with one every 6 or 7).
// The tile's epilogue was 20 k of 170 k cycles at K = 4096 (bounds by branches, 8-byte stores, a division a
// SiLU, and a wait for all of its stores): now stores of 16 bytes a lane through range-checked descriptors that
// nothing waits for until the tile's second K-tile. Both against a schedule of reads and pieces in bursts and
// the former epilogue, us, one card (others run 3 to 4 % faster): 16384 x 6144 x 4096 570 -> 540 (1.53 PFLOP/s), 8192 x
// 4096 x 4096 191 -> 182 and x 14336 655 -> 629, 8192 x 28672 x 4096 with SiLU pairs 1295 -> 1249 (1.54). fp32 outputs
// of 8192 x 4096 x 4096 gain nothing (189): all CUs store 67 MB at once, at 6.4 TB/s, behind which the next tile's pieces wait.
#pragma once
#include "gemm_common.h"

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
typedef const __attribute__((address_space(3))) bf16x8 lds_frag;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}
// silu(g) u, or gelu(g) u by its tanh form, with a quotient that costs 6 instructions for a division's ten (128 of them
// a lane are 5 k cycles of a tile) and equals it to the bit (by all of 2^26 random gates and as many of each range of
// exponents; gates below 2^-124 to 2^-149). The reciprocal alone, 2 instructions, is an ulp off in a quarter of the cases.
// g / d as (g / 4) / (d / 4), whose reciprocal is no denormal number, which v_rcp_f32 would flush; the quotient's
// remainder corrects it, and v_div_fixup_f32 sees to infinities
template <int EPI> __device__ __forceinline__ float pair_div(float g, float u) {
  const float e = EPI == EPI_GELU_MUL ? 1.5957691216057308f * (g + 0.044715f * g * g * g) : g;
  const float n = 0.25f * g, d = fmaf(0.25f, __expf(-e), 0.25f), r = __builtin_amdgcn_rcpf(d), q = n * r;
  return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, q, n), r, q), d, n) * u;
}
// 1 KiB of LDS-DMA (16 B a lane); IMM moves both the address in memory and the one in LDS
template <int IMM>
__device__ __forceinline__ void dma16(const void* base, int bytes, uint32_t lds, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(make_rsrc(base, bytes), (lds_void*)lds, 16, voff, soff, IMM, 0);
}

// The schedule of a K-tile: 2 MI NJ MFMAs, the first half on the fragments F0 (its first 32 values of K, read
// before it began), the second on F1. After MFMA q:
//   0 .. NF - 1         a fragment of F1 each
//   B1                  every wave has read the buffer: a barrier frees it
//   D, D + DS, ..       a DMA piece of the K-tile after the next into it, NP of them
//   B2                  the next K-tile landed (the pieces just issued may fly) for every wave
//   B2 + 1, + 3, ..     a fragment of the next K-tile's F0 each
// Positions by measurement, times of 8192 x 4096 x 4096 and 16384 x 4096 x 14336 against these: reads one MFMA apart
// instead of two -0.7 % and +0.2 %, pieces 5 instead of 6 apart -1.0 % and +1.3 %.
template <int NJ, int MI> struct Sched4w {
  static constexpr int Q = 2 * MI * NJ, NF = MI + NJ, NP = MI + NJ;
  static constexpr int B1 = NF + 3 + NJ / 3, D = B1 + 1, DS = (Q - 4 - D) / (NP - 1), DL = D + DS * (NP - 1);
  static constexpr int B2 = Q - 1 - 2 * NF;
  static constexpr int ahead = B2 < D ? 0 : (B2 - D) / DS + 1;      // pieces issued when B2 waits
  static_assert(DS >= 1 && DL + 2 < Q && B2 > B1 && ahead <= NP, "the pieces fit the K-tile");
};

// The u-th block of a half K-tile: two rows of blocks down, then up, column after column, and back on the next two,
// so that each MFMA shares one of its two fragments with the one before and each of both is taken anew every other
// time (the first columns need W's first fragments and A's first two, in the order in which they are read). The sums are
// the same. us against row after row, a step as much as 4 % ahead of a new pair each time, one card: 8192 x 28672 x 4096
// with SiLU pairs 1250 -> 1226 (1.57 PFLOP/s), 8192 x 6144 x 4096 272 -> 268, 8192 x 4096 x 14336 642 -> 634, 512 x
// 128256 x 4096 421 -> 409. Rows back and forth give 0.8 %, columns likewise 0.8, three rows at a time 1.4, four
// 1.2, two columns 1.6 and a Hilbert curve 1.7, against this one's 1.6.
template <int NJ> struct Walk4w {
  static constexpr int col_of(int u) {
    const int j = u % (2 * NJ) / 2;
    return u / (2 * NJ) % 2 ? NJ - 1 - j : j;
  }
  static constexpr int row_of(int u) { return u / (2 * NJ) * 2 + ((u ^ u % (2 * NJ) / 2) & 1); }
};

// EPI_F32's bias (unsplit): where the block maxima go (BlockMax). ws: the partial sums' slabs of a product
// split over K (fp32, or fp16 with EPI_SLAB16). group_off: rows of group g are [off[g], off[g + 1]).
template <int EPI, int NJ, int MI>
__global__ void __launch_bounds__(256, 1) gemm4w_kernel(
    const u16* __restrict__ A, int lda, const u16* __restrict__ W, int ldw,
    void* __restrict__ C, int ldc, int M, int N, int K, int splits, const u16* __restrict__ bias,
    float* __restrict__ ws, const int* __restrict__ group_off, int groups) {
  using S = Sched4w<NJ, MI>;
  constexpr int BM = 32 * MI, BN = 32 * NJ, GM = 4;
  constexpr int A_BYTES = BM * BK * 2;
  constexpr int NF = S::NF, NP = S::NP;
  constexpr bool PAIRS = epi_pairs(EPI);
  // two buffers 64 KiB apart: the bit that tells them apart. The kernel has no other LDS, so it starts at 0
  constexpr uint32_t FLIP = 0x10000;
  static_assert(MI % 2 == 0 && (BM + BN) * BK * 2 <= (int)FLIP && MI * NJ <= 64, "a K-tile's buffer, and accumulators");

  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wid >> 1, wn = wid & 1;
  const int tiles_n = (N + BN - 1) / BN;
  const int ksl = K / splits, nk = ksl / BK;

  // ---- tiles. Dense: virtual id -> XCD remap -> (split, grouped order of GM row tiles). Grouped: a group's
  // row tiles follow those of the groups before it, 64 groups a step, a group a lane
  int tiles_m = (M + BM - 1) / BM;
  int ga = 0, gb = 0, gsum = 0;                    // this lane's group: its rows, row tiles up to and with it
  auto load_groups = [&](int g0) {
    const int g = g0 + lane;
    ga = g < groups ? group_off[g] : 0;
    gb = g < groups ? group_off[g + 1] : 0;
    gsum = (gb - ga + BM - 1) / BM;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int up = __shfl_up(gsum, o, 64);
      if (lane >= o) gsum += up;
    }
    return __builtin_amdgcn_readlane(gsum, 63);
  };
  if (group_off != nullptr) {
    tiles_m = 0;
    for (int g0 = (groups - 1) & ~63; g0 >= 0; g0 -= 64) tiles_m += load_groups(g0);
  }
  const int nwg = tiles_m * tiles_n;
  const int total = nwg * splits;
  struct Tile { int m0, n0, ks, row0, rows; const u16* w; };
  auto locate = [&](int v) -> Tile {
    Tile t;
    const int lg = xcd_remap(v, total);
    t.ks = lg / nwg;
    int tile = lg - t.ks * nwg, tm = tiles_m;
    t.row0 = 0;
    t.rows = M;
    t.w = W;
    if (group_off != nullptr) {
      int before = 0;                              // row tiles of the groups before this step's
      for (int g0 = 0; g0 < groups; g0 += 64) {
        // (the first 64 groups' stay in registers: a load here would wait for the stores in flight)
        const int sum = groups > 64 ? load_groups(g0) : __builtin_amdgcn_readlane(gsum, 63);
        const unsigned long long past = __ballot((before + gsum) * tiles_n > tile);
        if (past != 0) {
          const int l = __builtin_ctzll(past);
          t.row0 = __builtin_amdgcn_readlane(ga, l);
          t.rows = __builtin_amdgcn_readlane(gb, l) - t.row0;
          tm = (t.rows + BM - 1) / BM;
          tile -= (before + __builtin_amdgcn_readlane(gsum, l) - tm) * tiles_n;
          t.w = W + (long)(g0 + l) * N * ldw;
          break;
        }
        before += sum;
      }
    }
    const int per_group = GM * tiles_n;
    const int first_m = (tile / per_group) * GM;
    const int gsz = min(tm - first_m, GM);
    const int in_g = tile % per_group;
    t.m0 = (first_m + in_g % gsz) * BM;
    t.n0 = (in_g / gsz) * BN;
    return t;
  };

  // ---- staging. LDS rows of 128 B whose 16-B chunk c of row r lies at c ^ ((r >> 1) & 7). A wave moves 8 MI rows
  // of A and 8 NJ of W a K-tile, piece i the rows 8 i + lane / 8 of them: only i's parity changes the chunk
  // (MI is even) that a lane fetches, the rest is the soffset's. Rows past the matrix read as zeros
  const int prow = 8 * MI * wid + (lane >> 3), wprow = 8 * NJ * wid + (lane >> 3);
  const int ce = (lane & 7) ^ ((lane >> 4) & 7), co = (lane & 7) ^ (((lane >> 4) + 4) & 7);
  // (a wave's W rows start at an odd multiple of 8 where NJ and the wave are odd)
  const bool flip = (NJ * wid) & 1;
  const int va0 = prow * lda * 2 + ce * 16, va1 = prow * lda * 2 + co * 16;
  const int vw0 = wprow * ldw * 2 + (flip ? co : ce) * 16, vw1 = wprow * ldw * 2 + (flip ? ce : co) * 16;
  int xa0, xa1, xw0, xw1;                          // those of the next K-tile to stage
  int sofa[MI], sofw[NJ];                           // a piece's soffset, less its immediate offset
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    sofa[i] = i * 16 * lda - (i & 3) * 1024;
    asm volatile("" : "+s"(sofa[i]));
  }
#pragma unroll
  for (int i = 0; i < NJ; ++i) {
    sofw[i] = i * 16 * ldw - (i & 3) * 1024;
    asm volatile("" : "+s"(sofw[i]));
  }
  const u16 *sa, *sw;                              // the staged tile's panels, and their bytes in range
  int sab, swb;
  auto begin_stage = [&](const Tile& t, bool any) {
    sa = A + (long)(t.row0 + t.m0) * lda + t.ks * ksl;
    sw = t.w + (long)t.n0 * ldw + t.ks * ksl;
    sab = any && nk > 0 ? (min(t.rows - t.m0, BM) * lda - t.ks * ksl) * 2 : 0;
    swb = any && nk > 0 ? (min(N - t.n0, BN) * ldw - t.ks * ksl) * 2 : 0;
    xa0 = va0; xa1 = va1; xw0 = vw0; xw1 = vw1;
  };
  uint32_t da = 8 * MI * wid * 128, dw = A_BYTES + 8 * NJ * wid * 128;
  auto piece = [&](auto F) __attribute__((always_inline)) {
    constexpr int f = decltype(F)::value;
    if constexpr (f < MI)
      dma16<(f & 3) * 1024>(sa, sab, da + (f >> 2) * 4096, f & 1 ? xa1 : xa0, sofa[f]);
    else
      dma16<((f - MI) & 3) * 1024>(sw, swb, dw + ((f - MI) >> 2) * 4096, f & 1 ? xw1 : xw0, sofw[f - MI]);
  };
  auto next_buffer = [&]() { da ^= FLIP; dw ^= FLIP; };
  auto next_k = [&]() { xa0 += 2 * BK; xa1 += 2 * BK; xw0 += 2 * BK; xw1 += 2 * BK; };

  // ---- fragments: rows 16 apart swizzle alike, so one address a half K-tile and operand
  const int fr = lane & 15, fq = lane >> 4;
  const int arow = wm * 16 * MI + fr, wrow = wn * 16 * NJ + fr;
  uint32_t ra0 = arow * 128 + ((fq ^ ((arow >> 1) & 7)) << 4);
  uint32_t ra1 = arow * 128 + (((4 + fq) ^ ((arow >> 1) & 7)) << 4);
  uint32_t rw0 = A_BYTES + wrow * 128 + ((fq ^ ((wrow >> 1) & 7)) << 4);
  uint32_t rw1 = A_BYTES + wrow * 128 + (((4 + fq) ^ ((wrow >> 1) & 7)) << 4);
  f32x4 acc[MI][NJ];
  bf16x8 a0[MI], b0[NJ], a1[MI], b1[NJ];
  // in the order of their use: A's first, all of W's, A's others
  auto read = [&](auto F, bf16x8 (&av)[MI], bf16x8 (&bv)[NJ], uint32_t pa, uint32_t pw)
      __attribute__((always_inline)) {
    constexpr int f = decltype(F)::value;
    if constexpr (f >= 1 && f <= NJ) {
      bv[f - 1] = *(lds_frag*)(pw + (f - 1) * 2048);
    } else {
      constexpr int i = f == 0 ? 0 : f - NJ;
      av[i] = *(lds_frag*)(pa + i * 2048);
    }
  };
  auto fence = [&]() __attribute__((always_inline)) { __builtin_amdgcn_sched_barrier(0); };
  auto barrier = [&]() __attribute__((always_inline)) {
    asm volatile("" ::: "memory");
    fence();
    __builtin_amdgcn_s_barrier();
    fence();
    asm volatile("" ::: "memory");
  };

  // one K-tile. FIRST: its sums begin at zero; MORE: another of the same tile follows, in LDS already where landed
  auto ktile = [&](auto FIRST, auto MORE, bool landed) __attribute__((always_inline)) {
    constexpr bool first = decltype(FIRST)::value, more = decltype(MORE)::value;
    auto after = [&](auto QC) __attribute__((always_inline)) {
      constexpr int q = decltype(QC)::value;
      if constexpr (q < NF) {
        read(int_c<q>{}, a1, b1, ra1, rw1);
        fence();
      }
      if constexpr (q == S::B1) {
        __builtin_amdgcn_s_waitcnt(0xC07F);        // lgkmcnt(0)
        barrier();
      }
      if constexpr (q >= S::D && q <= S::DL && (q - S::D) % S::DS == 0) {
        piece(int_c<(q - S::D) / S::DS>{});
        fence();
      }
      if constexpr (q == S::DL + 1) { next_buffer(); fence(); }
      if constexpr (q == S::DL + 2) { next_k(); fence(); }
      if constexpr (q == S::B2 - 1) { ra0 ^= FLIP; rw0 ^= FLIP; fence(); }
      if constexpr (q == S::B2 && more) {
        if (!landed) {
          wait_vmcnt<S::ahead>();
          barrier();
        }
      }
      if constexpr (more && q > S::B2 && (q - S::B2) % 2 == 1) {
        read(int_c<(q - S::B2) / 2>{}, a0, b0, ra0, rw0);
        fence();
      }
      if constexpr (q == S::Q - 1) { ra1 ^= FLIP; rw1 ^= FLIP; fence(); }
    };
    // inline asm keeps the accumulators in the AGPR file ("+a"; hipcc's own selection moves them through
    // VGPRs); it pads no hazard inside: the fragments' reads it waits for by register, the accumulators are
    // read only as the next MFMA's C until the pad behind the loop
    unroll<MI * NJ>([&](auto U) __attribute__((always_inline)) {
      constexpr int u = decltype(U)::value, i = Walk4w<NJ>::row_of(u), j = Walk4w<NJ>::col_of(u);
      if constexpr (first)
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0"
                     : "=a"(acc[i][j]) : "v"(b0[j]), "v"(a0[i]));
      else
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                     : "+a"(acc[i][j]) : "v"(b0[j]), "v"(a0[i]));
      after(U);
    });
    unroll<MI * NJ>([&](auto U) __attribute__((always_inline)) {
      constexpr int u = decltype(U)::value, i = Walk4w<NJ>::row_of(u), j = Walk4w<NJ>::col_of(u);
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                   : "+a"(acc[i][j]) : "v"(b1[j]), "v"(a1[i]));
      after(int_c<MI * NJ + u>{});
    });
  };
  // an accumulator leaves the AGPR file by one pinned copy, ahead of any condition
  auto vget = [&](const f32x4& a) __attribute__((always_inline)) -> f32x4 {
    f32x4 v;
    asm volatile("" : "=v"(v) : "0"(a));
    return v;
  };

  // ---- epilogue of a tile: acc[i][j][r] = C[m0 + 16 MI wm + 16 i + fr][n0 + 16 NJ wn + 16 j + 4 fq + r].
  // ranged: whole quads (fp32, partial sums) or octets (16 bits) at aligned addresses, so that rows past the
  // matrix fall out of the descriptor's range and columns past it get an offset out of it
  const bool slab = splits > 1;
  constexpr bool OUT32 = EPI == EPI_F32;
  const int ld = slab ? N : ldc;
  const bool ranged = [&]() {
    const uintptr_t at = (uintptr_t)(slab ? (const void*)ws : C);
    const bool wide = OUT32 || (slab && EPI != EPI_SLAB16);
    const bool bias_ok = !(EPI == EPI_BIAS || EPI == EPI_BIAS_GELU) || ((uintptr_t)bias & 7) == 0;
    return bias_ok && ld < (int)((1u << 31) / (4 * BM)) - 1024 &&
           (wide ? ((N | ld) & 3) == 0 && (at & 15) == 0 : ((N | ld) & 7) == 0 && (at & 15) == 0);
  }();
  auto quad_f = [&](const f32x4& v, uint2 bq) __attribute__((always_inline)) -> f32x4 {
    f32x4 o = v;
    if (EPI == EPI_BIAS || EPI == EPI_BIAS_GELU) {
      o[0] += __uint_as_float(bq.x << 16); o[1] += __uint_as_float(bq.x & 0xffff0000u);
      o[2] += __uint_as_float(bq.y << 16); o[3] += __uint_as_float(bq.y & 0xffff0000u);
    }
    if (EPI == EPI_BIAS_GELU) {
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = gelu_f(o[r]);
    }
    return o;
  };
  constexpr int OUT_OF_RANGE = (int)0x80000000;
  // fp32 quads: logits, fp32 outputs, partial sums; returns with them in flight
  auto store32 = [&](const Tile& t, char* base, uint32_t* keys) __attribute__((always_inline)) {
    const int left = min(t.rows - t.m0, BM), cols = N - t.n0;
    const auto rc = make_rsrc(base, left * ld * 4);
    const int c0 = 16 * NJ * wn + 4 * fq, vo = ((16 * MI * wm + fr) * ld + c0) * 4;
    unroll<MI>([&](auto I) __attribute__((always_inline)) {
      constexpr int i = decltype(I)::value;
      BlockMax top;
      unroll<NJ>([&](auto J) __attribute__((always_inline)) {
        constexpr int j = decltype(J)::value;
        const f32x4 v = vget(acc[i][j]);
        const bool in = c0 + 16 * j < cols;
        if (EPI == EPI_F32 && in) top.take(v);
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rc,
                                               in ? vo + 64 * j : OUT_OF_RANGE, i * 16 * ld * 4, 0);
      });
      if constexpr (EPI == EPI_F32) {
        if (keys != nullptr) {                     // uniform
          const uint32_t key = row_key(top);
          const int row = t.m0 + 16 * MI * wm + 16 * i + fr, wc0 = t.n0 + 16 * NJ * wn;
          if (fq == 0 && row < t.rows && wc0 < N)
            keys[(long)row * ((N + 16 * NJ - 1) / (16 * NJ)) + wc0 / (16 * NJ)] = key;
        }
      }
    });
  };
  // 16-bit outputs: neighbouring blocks' quads change places between lanes 16 apart, so that a lane holds 8
  // columns and a store covers 64 B of each row
  auto store16 = [&](const Tile& t, char* base) __attribute__((always_inline)) {
    constexpr int NO = PAIRS ? NJ / 2 : NJ;        // blocks of 16 output columns
    const int left = min(t.rows - t.m0, BM), cols = (PAIRS ? N / 2 : N) - (PAIRS ? t.n0 / 2 : t.n0);
    const auto rc = make_rsrc(base, left * ld * 2);
    const int c0 = 16 * NO * wn + 16 * (fq & 1) + 8 * (fq >> 1), c1 = 16 * NO * wn + 16 * (NO - 1) + 4 * fq;
    const int ro = (16 * MI * wm + fr) * ld * 2;
    // What the tile is added to is requested all at once, into the fragments' registers: 128 KB a CU at the
    // memory's rate, 3 to 7 us a round of tiles (three row blocks' requests ahead of the last K-tile changed nothing). The
    // add behind it read and wrote twice that: ops._add_product has the times
    if constexpr (EPI == EPI_RES) {
      u32x4 old[MI][NO / 2];
      u32x2 odd[MI];
      auto fetch = [&](auto I) __attribute__((always_inline)) {
        constexpr int i = decltype(I)::value;
        unroll<NO / 2>([&](auto J) __attribute__((always_inline)) {
          constexpr int j = 2 * decltype(J)::value;
          old[i][j / 2] = __builtin_amdgcn_raw_buffer_load_b128(
              rc, c0 + 16 * j < cols ? ro + 2 * c0 + 32 * j : OUT_OF_RANGE, i * 16 * ld * 2, 0);
        });
        if constexpr (NO & 1)
          odd[i] = __builtin_amdgcn_raw_buffer_load_b64(rc, c1 < cols ? ro + 2 * c1 : OUT_OF_RANGE,
                                                            i * 16 * ld * 2, 0);
      };
      auto sum = [](uint32_t c, float lo, float hi) __attribute__((always_inline)) -> uint32_t {
        return pack2bf(__uint_as_float(c << 16) + lo, __uint_as_float(c & 0xffff0000u) + hi);
      };
      unroll<MI>(fetch);
      asm volatile("" ::: "memory");
      unroll<MI>([&](auto I) __attribute__((always_inline)) {
        constexpr int i = decltype(I)::value;
        unroll<NO / 2>([&](auto J) __attribute__((always_inline)) {
          constexpr int j = 2 * decltype(J)::value;
          const f32x4 x = vget(acc[i][j]), y = vget(acc[i][j + 1]);
          float f[8];
          unroll<4>([&](auto R) __attribute__((always_inline)) {
            constexpr int k = decltype(R)::value;
            const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(x[k]), __float_as_uint(y[k]), false, false);
            f[k] = __uint_as_float(p[0]);
            f[4 + k] = __uint_as_float(p[1]);
          });
          const u32x4 c = old[i][j / 2];
          __builtin_amdgcn_raw_buffer_store_b128(
              u32x4{sum(c[0], f[0], f[1]), sum(c[1], f[2], f[3]), sum(c[2], f[4], f[5]), sum(c[3], f[6], f[7])}, rc,
              c0 + 16 * j < cols ? ro + 2 * c0 + 32 * j : OUT_OF_RANGE, i * 16 * ld * 2, 0);
        });
        if constexpr (NO & 1) {
          const f32x4 x = vget(acc[i][NO - 1]);
          const u32x2 c = odd[i];
          __builtin_amdgcn_raw_buffer_store_b64(u32x2{sum(c[0], x[0], x[1]), sum(c[1], x[2], x[3])}, rc,
                                                c1 < cols ? ro + 2 * c1 : OUT_OF_RANGE, i * 16 * ld * 2, 0);
        }
      });
      return;
    }
    uint2 bq[NJ];
    if constexpr (EPI == EPI_BIAS || EPI == EPI_BIAS_GELU) {
      const auto rb = make_rsrc(bias, N * 2);
      unroll<NJ>([&](auto J) __attribute__((always_inline)) {
        constexpr int j = decltype(J)::value;
        const auto b = __builtin_amdgcn_raw_buffer_load_b64(rb, (t.n0 + 16 * NJ * wn + 16 * j + 4 * fq) * 2, 0, 0);
        bq[j] = uint2{b[0], b[1]};
      });
    }
    unroll<MI>([&](auto I) __attribute__((always_inline)) {
      constexpr int i = decltype(I)::value;
      auto quad = [&](auto J) __attribute__((always_inline)) -> uint2 {
        constexpr int j = decltype(J)::value;
        if constexpr (PAIRS) {
          const f32x4 g = vget(acc[i][2 * j]), u = vget(acc[i][2 * j + 1]);
          float o[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = pair_div<EPI>(g[r], u[r]);
          return uint2{pack2bf(o[0], o[1]), pack2bf(o[2], o[3])};
        } else if constexpr (EPI == EPI_SLAB16) {
          const f32x4 v = vget(acc[i][j]);
          return uint2{pack2h(v[0] * SLAB16_SCALE, v[1] * SLAB16_SCALE),
                       pack2h(v[2] * SLAB16_SCALE, v[3] * SLAB16_SCALE)};
        } else {
          const f32x4 o = quad_f(vget(acc[i][j]), bq[j]);
          return uint2{pack2bf(o[0], o[1]), pack2bf(o[2], o[3])};
        }
      };
      unroll<NO / 2>([&](auto J) __attribute__((always_inline)) {
        constexpr int j = 2 * decltype(J)::value;
        const uint2 x = quad(int_c<j>{}), y = quad(int_c<j + 1>{});
        const auto p = __builtin_amdgcn_permlane16_swap(x.x, y.x, false, false);
        const auto q = __builtin_amdgcn_permlane16_swap(x.y, y.y, false, false);
        __builtin_amdgcn_raw_buffer_store_b128(u32x4{p[0], q[0], p[1], q[1]}, rc,
                                               c0 + 16 * j < cols ? ro + 2 * c0 + 32 * j : OUT_OF_RANGE,
                                               i * 16 * ld * 2, 0);
      });
      if constexpr (NO & 1) {
        const uint2 x = quad(int_c<NO - 1>{});
        __builtin_amdgcn_raw_buffer_store_b64(u32x2{x.x, x.y}, rc, c1 < cols ? ro + 2 * c1 : OUT_OF_RANGE,
                                              i * 16 * ld * 2, 0);
      }
    });
  };
  // any width and alignment, quad by quad
  auto store_any = [&](const Tile& t) __attribute__((always_inline)) {
    const int wr0 = t.m0 + 16 * MI * wm, wc0 = t.n0 + 16 * NJ * wn;
    const bool vec = slab ? (N & 3) == 0 : out_vec<EPI>(C, ldc, N, bias);
    float* sl = ws + (long)t.ks * M * N;
    unroll<MI>([&](auto I) __attribute__((always_inline)) {
      constexpr int i = decltype(I)::value;
      const int row = wr0 + 16 * i + fr;
      BlockMax top;
      unroll<NJ>([&](auto J) __attribute__((always_inline)) {
        constexpr int j = decltype(J)::value;
        const int col = wc0 + 16 * j + 4 * fq;
        if constexpr (PAIRS) {
          if constexpr (j % 2 == 0) {
            const f32x4 g = vget(acc[i][j]), u = vget(acc[i][j + 1]);
            if (slab) {
              float* p = sl + (long)(t.row0 + row) * N + col;
              if (row < t.rows && col < N) slab_quad_fp32(p, g, 0, vec, N - col);
              if (row < t.rows && col + 16 < N) slab_quad_fp32(p + 16, u, 0, vec, N - col - 16);
            } else if (row < t.rows && col < N) {
              store_pair_quad<EPI>(C, ldc, t.row0 + row, ((wc0 + 16 * j) >> 5) * 16 + 4 * fq, g, u, vec);
            }
          }
        } else {
          const f32x4 v = vget(acc[i][j]);
          if (EPI == EPI_F32 && col < N) top.take(v);
          if (row < t.rows && col < N) {
            if (EPI == EPI_SLAB16)
              slab_quad16(sl + (long)(t.row0 + row) * N + col, v, vec, N - col, ws);
            else if (slab)
              slab_quad_fp32(sl + (long)(t.row0 + row) * N + col, v, 0, vec, N - col);
            else
              store_quad<EPI>(C, ldc, t.row0 + row, col, N, v, bias, vec);
          }
        }
      });
      if constexpr (EPI == EPI_F32) {
        if (!slab && bias != nullptr) {            // uniform: the block's largest value (BlockMax)
          const uint32_t key = row_key(top);
          if (fq == 0 && row < t.rows && wc0 < N)
            ((uint32_t*)bias)[(long)row * ((N + 16 * NJ - 1) / (16 * NJ)) + wc0 / (16 * NJ)] = key;
        }
      }
    });
  };
  // stores issued behind the next tile's pieces, which may fly while those are waited for (6 bits count)
  constexpr int N32 = MI * NJ, N16 = MI * (((PAIRS ? NJ / 2 : NJ) + 1) / 2);
  auto epilogue = [&](const Tile& t) __attribute__((always_inline)) {
    if (EPI != EPI_RES && !ranged) {
      store_any(t);
      asm volatile("" ::: "memory");
      wait_vmcnt<0>();
    } else if (EPI == EPI_F32 || (EPI != EPI_SLAB16 && EPI != EPI_RES && slab)) {
      char* base = slab ? (char*)(ws + ((long)t.ks * M + t.row0 + t.m0) * N + t.n0)
                        : (char*)((float*)C + (long)(t.row0 + t.m0) * ldc + t.n0);
      store32(t, base, EPI == EPI_F32 && !slab ? (uint32_t*)const_cast<u16*>(bias) : nullptr);
      asm volatile("" ::: "memory");
      wait_vmcnt<(N32 < 63 ? N32 : 63)>();
    } else {
      char* base = EPI == EPI_SLAB16 ? (char*)((u16*)ws + ((long)t.ks * M + t.row0 + t.m0) * N + t.n0)
                                     : (char*)((u16*)C + (long)(t.row0 + t.m0) * ldc + (PAIRS ? t.n0 / 2 : t.n0));
      store16(t, base);
      asm volatile("" ::: "memory");
      wait_vmcnt<(N16 < 63 ? N16 : 63)>();
    }
  };

  using T_ = std::integral_constant<bool, true>;
  using F_ = std::integral_constant<bool, false>;
  int v = blockIdx.x;
  if (v >= total) return;                          // wave-uniform: every wave exits
  Tile t = locate(v);
  // K-tiles 0 and 1 of the first tile (a K of one K-tile: the second is zeros)
  begin_stage(t, true);
  unroll<NP>(piece);
  next_buffer();
  next_k();
  if (nk < 2) sab = swb = 0;
  unroll<NP>(piece);
  next_buffer();
  next_k();
  wait_vmcnt<0>();
  barrier();

  while (true) {                                   // every wave runs the same tiles
    const int vn = v + (int)gridDim.x;
    const bool has_next = vn < total;
    Tile tn = t;
    if (has_next) tn = locate(vn);
    unroll<NF>([&](auto F) __attribute__((always_inline)) { read(F, a0, b0, ra0, rw0); });
    if (nk > 2) {
      // (K-tile 1 is there, and the last tile's stores need not have left: nothing to wait for in K-tile 0)
      ktile(T_{}, T_{}, true);
    } else {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      // these are read by inline-asm MFMAs, which hipcc pads no hazard for: every write ahead of wait states
#pragma unroll
      for (int i = 0; i < MI; ++i) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) asm volatile("" : "+a"(acc[i][j]));
        asm volatile("s_nop 3");
      }
    }
    for (int kt = 1; kt + 2 < nk; ++kt) ktile(F_{}, T_{}, false);
    // the last two K-tiles stage the next tile's first two. Without a next tile they stage through an
    // empty range (no memory traffic, zeros): one code path, since a branch doubles the unrolled tail and hipcc
    // spills the fragments or moves the descriptors into VGPRs
    begin_stage(tn, has_next);
    ktile(F_{}, T_{}, nk <= 2);
    if (nk < 2) sab = swb = 0;
    ktile(F_{}, F_{}, false);
    // MFMA results -> the epilogue's copies: the XDL write-back's wait states, tied to the last rows of
    // accumulators written so that no copy of them moves above the pad
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int j = 0; j < NJ; ++j) asm volatile("" : "+a"(acc[MI - 2][j]), "+a"(acc[MI - 1][j]));
    epilogue(t);       // (and its wait: the next tile's K-tiles 0 and 1 landed, also before an exit)
    if (!has_next) break;
    barrier();
    v = vn;
    t = tn;
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

// the mode that dli_gemm_set_slab_store asked for
int gemm_4w_store_mode();

// the stride of a tile's 32 L rows from which its offsets no longer fit 31 bits, to a power of two
template <int L> constexpr int MAX_LD = L > 8 ? 1 << 21 : 1 << 22;

// M: rows, or the most rows of a group (group_off: their offsets, groups of them)
template <int EPI, int NJ, int MI = 8>
static int launch_4w(const void* A, int lda, const void* W, int ldw, void* C, int ldc, int M, int N,
                     int K, int splits, const void* bias, void* ws, const int* group_off, int groups,
                     hipStream_t st) {
  if (epi_pairs(EPI) && N % 32) return (int)hipErrorInvalidValue;
  if (K % (splits * BK)) return (int)hipErrorInvalidValue;
  // (a panel's range is its rows times their stride in 32 bits, which overlapping rows would reach past: ops/gemm.py's
  // spaced copies those)
  if (lda < K || ldw < K || lda >= MAX_LD<MI> || ldw >= MAX_LD<NJ>) return (int)hipErrorInvalidValue;
  // The kernel has one way to store fp32 partial sums (the others' probe modes would more than double its code): while
  // another is set, split products are refused and not timed as what they are not
  if (splits > 1 && EPI != EPI_SLAB16 && gemm_4w_store_mode() != 0) return (int)hipErrorInvalidValue;
  if (EPI == EPI_RES && (splits != 1 || group_off != nullptr || ((N | ldc) & 7) || ((uintptr_t)C & 15) || C == nullptr ||
                         ldc >= (1 << 21) - 1024))
    return (int)hipErrorInvalidValue;
  constexpr size_t lds = 0x10000 + (size_t)(32 * MI + 32 * NJ) * BK * 2;
  static bool raised = false;
  if (!raised) {
    hipFuncSetAttribute((const void*)gemm4w_kernel<EPI, NJ, MI>, hipFuncAttributeMaxDynamicSharedMemorySize,
                        (int)lds);
    raised = true;
  }
  const int cus = cu_count();
  const long tiles = (long)((M + 32 * MI - 1) / (32 * MI)) * ((N + 32 * NJ - 1) / (32 * NJ)) * splits *
                     (group_off != nullptr ? groups : 1);
  // one workgroup per CU (over 80 KiB of LDS each); a multiple of 8 keeps every workgroup's virtual tile ids
  // on one XCD residue class
  int grid = tiles < cus ? (int)tiles : (cus / 8) * 8;
  if (grid < 1) grid = 1;
  gemm4w_kernel<EPI, NJ, MI><<<grid, 256, lds, st>>>((const u16*)A, lda, (const u16*)W, ldw, C, ldc, M, N, K, splits,
                                                 (const u16*)bias, (float*)ws, group_off, groups);
  if constexpr (EPI != EPI_RES) {                  // (never split)
    if (splits > 1 && C != nullptr) {
      const int outN = epi_pairs(EPI) ? N / 2 : N;
      const long total = (long)M * outN;
      splitk_reduce_kernel<EPI><<<(int)((total + 255) / 256), 256, 0, st>>>(
          C, ldc, (const float*)ws, M, N, splits, (const u16*)bias);
    }
  }
  DLI_RETURN_LAUNCH();
}

// the epilogues of the tiles that gemm4w.hip chooses by rounds
template <int NJ, int MI = 8> static int launch_nj(int epi, DLI_GEMM_ARGS) {
  switch (epi) {
    case EPI_BF16: return launch_4w<EPI_BF16, NJ, MI>(DLI_GEMM_PASS);
    case EPI_F32: return launch_4w<EPI_F32, NJ, MI>(DLI_GEMM_PASS);
    case EPI_SLAB16: return launch_4w<EPI_SLAB16, NJ, MI>(DLI_GEMM_PASS);
    case EPI_RES: return launch_4w<EPI_RES, NJ, MI>(DLI_GEMM_PASS);
    default: break;
  }
  if constexpr (NJ % 2 == 0) {                     // a gate block and its up block in one wave tile
    if (epi == EPI_SILU) return launch_4w<EPI_SILU, NJ, MI>(DLI_GEMM_PASS);
    if (epi == EPI_GELU_MUL) return launch_4w<EPI_GELU_MUL, NJ, MI>(DLI_GEMM_PASS);
  }
  return DLI_NOT_MINE;
}
