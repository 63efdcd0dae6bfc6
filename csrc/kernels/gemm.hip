// bf16 GEMM on CDNA4 matrix cores: C[M,N] = A[M,K] . W[N,K]^T (+ fused epilogue).
// Dense projections and the experts' grouped products.
//
// Structure (cdna_hip_programming.md §5):
//  * WM x WN waves (2x2 = 256 threads, or 2x4 / 4x2 = 512 threads for 256-wide tiles); block
//    tile BM x BN x 64; wave tile (BM/WM) x (BN/WN) built from v_mfma_f32_16x16x32_bf16 (the bf16 shape that holds the higher clock on random
//    data, /opt/skills/guides/MI355X_MICROARCH.md 'DVFS give-back' item 7).
//  * global -> LDS by global_load_lds_dwordx4 (16 B per lane, no VGPR round trip), 2 LDS
//    buffers: the next K-tile's DMA is issued before the current tile's ds_reads + MFMAs.
//  * LDS rows are 128 B (64 bf16); the 16-B chunk c of row r is stored at physical chunk
//    c ^ ((r >> 1) & 7). glds writes lane-linearly, so the permutation is applied to the
//    per-lane GLOBAL source address and the same XOR on the ds_read_b128 address (rule 21);
//    verified conflict-free for all four ds_read_b128 lane groups of the 16x16x32 A/B maps.
//  * XCD-aware bijective block remap (T1) with n-major tile order so consecutive tiles share
//    one W panel in an XCD's L2; split-K grids are remapped split-major so an XCD's blocks
//    share one K slice of A and W (split_tile).
//  * split-K over grid.y writes fp32 slabs; a second pass reduces and applies the epilogue.
//  * grouped mode (MoE): grid.z = expert; rows of group g are [off[g], off[g+1]) of A/C,
//    weights W + g*N*ldw. Rows past the group end are skipped. Split-K composes with it
//    (slab rows are the permuted rows), for long-K expert GEMMs with few row tiles.
// Epilogues: 0 bf16 store, 1 fp32 store (logits), 2 SiLU(gate)*up over the 16-row-interleaved
// gate/up weight (output width N/2), 3 bias + tanh-GELU, 4 bias, 16 C += (4-wave tiles).
//
// Files: gemm_common.h (shared epilogue / split-K pieces), gemm_tiles.hip (ids 0-21, 23-25),
// gemm_stream.hip (60-72: few rows, weights streamed), gemm4w.h +
// gemm4w.hip, gemm4w_narrow.hip (22, 28, 34, 41, 45, 55), gemm8p.hip (26; 22 and 28 with the rarer epilogues), gemv.hip (29-33 and the fused batch-1 combine).
#include "gemm_common.h"

extern "C" int dli_gemm_set_slab_store(int mode) {
  const int old = gemm_tiles_set_slab_store(mode);
  gemm_stream_set_slab_store(mode);
  gemm_8p_set_slab_store(mode);
  gemm_4w_set_slab_store(mode);
  return old;
}

// one family's split-K slab store (0 plain, 1 nt, 2 sc1, 3 sc0 sc1): family 0 = the generic
// tiles (decode O / QKV), 1 = the 8-phase kernels, 2 = the 4-wave tiles (22 and 28 too), which refuse split products
// in any but mode 0
extern "C" int dli_gemm_set_slab_store_family(int family, int mode) {
  switch (family) {
    case 0: gemm_stream_set_slab_store(mode); return gemm_tiles_set_slab_store(mode);
    case 1: return gemm_8p_set_slab_store(mode);
    case 2: return gemm_4w_set_slab_store(mode);
    default: return -1;
  }
}

// tile_cfg: 0=64x64 1=64x128 2=128x128 3=128x256 4=256x128 (2 LDS stages); 5..9 = the same
// tiles with 3 LDS stages (one tile in flight across the barrier); 10/11 = 192x128 with 2/3
// stages, 12 = 160x128 (MoE experts of ~130-190 rows in one pass); 13-17 = 8-wave tiles
// 256x256, 256x128, 128x256 (2 stages) and 256x128, 128x256 (3 stages); 18/19 = 128x96 and
// 20/21 = 128x64 with 2/3 stages; 22 = 256x256; 23/24 = 128x192 (3/2
// stages), 25 = 256x192, 8 waves; 26 = 256x224 ping-pong; 29-33 = the M <= 4 weight
// stream (16 / 32 rows per workgroup, dispatch_gemv); 28 = 256x128; 34, 41, 45 = 256x256;
// 55 = 256x256, 192 or 160 (no split-K / grouped mode); 60-72 = weight-streaming tiles
// (gemm_stream.h). ws: fp32 [splits, M, N] when splits>1.
// group_off (nullable): int[groups+1] row offsets; M is then the max rows of any group.
// Grouped SiLU*up GEMM whose permuted row p reads activation row arow[p] (the MoE gate/up
// projection without the gathered copy of its input rows): the generic and streaming tiles
// only, unsplit. M: the row bound per group, as dli_gemm's grouped mode.
extern "C" int dli_gemm_grouped_gather(const void* A, int lda, const void* W, int ldw, void* C,
                                       int ldc, int M, int N, int K, int tile_cfg,
                                       const int* arow, const int* group_off, int groups,
                                       hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  const bool stream = tile_cfg >= 60 && tile_cfg <= 72;
  const bool generic = (tile_cfg >= 0 && tile_cfg <= 21) || (tile_cfg >= 23 && tile_cfg <= 25);
  if (!(generic || stream) || arow == nullptr || group_off == nullptr || groups < 1 || K % BK ||
      lda % 8 || ldw % 8 || N % 32)
    return (int)hipErrorInvalidValue;
  const void* bias = arow;
  void* ws = nullptr;
  const int* go = group_off;
  const int splits = 1;
  if (stream) return gemm_stream_dispatch(EPI_SILU, tile_cfg, DLI_GEMM_PASS);
  return gemm_tiles_dispatch(EPI_SILU, tile_cfg, DLI_GEMM_PASS);
}

extern "C" int dli_gemm(const void* A, int lda, const void* W, int ldw, void* C, int ldc, int M,
                        int N, int K, int epi, int tile_cfg, int splits, const void* bias,
                        void* ws, const int* group_off, int groups, hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  if (((tile_cfg < 29 || tile_cfg > 33) && K % BK) || lda % 8 || ldw % 8 || splits < 1)
    return (int)hipErrorInvalidValue;
  if (epi_pairs(epi) && N % 32) return (int)hipErrorInvalidValue;
  if (epi == EPI_CLAMP && (bias == nullptr || group_off != nullptr)) return (int)hipErrorInvalidValue;
  if ((epi == EPI_BIAS || epi == EPI_BIAS_GELU) && bias == nullptr) return (int)hipErrorInvalidValue;
  if (splits > 1 && ws == nullptr) return (int)hipErrorInvalidValue;
  if (groups < 1) groups = 1;
  if (epi == EPI_F32) bias = nullptr;              // (where the block maxima go: dli_gemm_head)
  const int* go = group_off;
  int r = gemm_tiles_dispatch(epi, tile_cfg, DLI_GEMM_PASS);
  if (r == DLI_NOT_MINE) r = gemm_stream_dispatch(epi, tile_cfg, DLI_GEMM_PASS);
  if (r == DLI_NOT_MINE) r = gemm_4w_dispatch(epi, tile_cfg, DLI_GEMM_PASS);
  if (r == DLI_NOT_MINE) r = gemm_8p_dispatch(epi, tile_cfg, DLI_GEMM_PASS);
  if (r == DLI_NOT_MINE) r = gemm_gemv_dispatch(epi, tile_cfg, DLI_GEMM_PASS);
  return r == DLI_NOT_MINE ? (int)hipErrorInvalidValue : r;
}

extern "C" int dli_gemm_4w_width(int tile_cfg, int epi, int M, int N, int splits);

// columns of the blocks whose maxima dli_gemm_head can write for a tile; 0: not for this one
static int head_block(int tile_cfg, int M, int N) {
  if (N % 4) return 0;
  if (tile_cfg == 55) return dli_gemm_4w_width(55, EPI_F32, M, N, 1) / 2;
  if (tile_cfg == 30 || tile_cfg == 32) return M <= 4 ? 16 : 0;
  if (tile_cfg == 31 || tile_cfg == 33) return M <= 4 ? 32 : 0;
  switch (tile_cfg) {                              // columns of a wave tile
    case 60: case 66: return 32;
    case 61: case 63: case 67: case 68: return 64;
    case 62: case 64: case 69: case 70: case 71: case 72: return 32;
    case 65: return 128;
    default: return 0;
  }
}
extern "C" int dli_gemm_head_block(int tile_cfg, int M, int N) { return head_block(tile_cfg, M, N); }

// C = A W^T in fp32 and, in keys [M, ceil(N / block)], each row's largest value by blocks of
// dli_gemm_head_block columns (BlockMax). Unsplit; the tiles with a block only.
extern "C" int dli_gemm_head(const void* A, int lda, const void* W, int ldw, void* C, int ldc, int M,
                             int N, int K, int tile_cfg, void* keys, hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  if (((tile_cfg < 29 || tile_cfg > 33) && K % BK) || lda % 8 || ldw % 8 || C == nullptr ||
      keys == nullptr || head_block(tile_cfg, M, N) == 0)
    return (int)hipErrorInvalidValue;
  const void* bias = keys;
  void* ws = nullptr;
  const int* go = nullptr;
  const int splits = 1, groups = 1;
  if (tile_cfg == 55) return gemm_4w_dispatch(EPI_F32, tile_cfg, DLI_GEMM_PASS);
  if (tile_cfg >= 60) return gemm_stream_dispatch(EPI_F32, tile_cfg, DLI_GEMM_PASS);
  return gemm_gemv_dispatch(EPI_F32, tile_cfg, DLI_GEMM_PASS);
}
