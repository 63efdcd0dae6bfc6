// Weight-streaming MFMA tiles for 2 to 128 rows (tile ids 60-72): the generic kernel
// (gemm_tiles.h) with one row of tiles, so every weight is read once, and three changes for a
// product that is bound by that read:
//  * weights requested nontemporal: they do not push the activations, which every workgroup
//    reads again, out of L2;
//  * column tile t starts its K loop at K-tile t mod nk and wraps around. Workgroups start
//    together, and a weight row is a power of two of bytes in most models: from one K offset all
//    of them ask the same few memory channels at a time;
//  * 48 to 96 KB in flight a CU: 3 to 6 LDS stages, widths from 32 to 256 columns so that one
//    launch is about one round of the chip without a split of K and its pass over partial sums.
// N = 28672, K = 4096 (235 MB), before -> after: 24 rows 51.2 -> 36.6 us (6.4 TB/s), 64 rows 52.7 ->
// 39.6, 96 rows 56.1 -> 44.1, 128 rows 56 -> 48. Of that, at 24 rows: depth alone 51 -> 46, nontemporal
// as well 41, the turned K loop as well 36.6. N = 128256, K = 4096: 24 rows 197 -> 167, 64 rows 209 ->
// 177, 128 rows 218 -> 192. fp32 outputs of 64 rows, K = 4096, with the reduce where K is split: N = 8192
// 20.0 -> 16.5, 16384 35.2 -> 26.5. At 192 rows and more the tiles of gemm_tiles.hip and gemm8p.hip are
// as fast or faster: the second row of tiles reads the weights again, from L2 if they stay there.
#pragma once
#include "gemm_tiles.h"

template <int EPI>
static int dispatch_stream(int tile_cfg, DLI_GEMM_ARGS) {
  switch (tile_cfg) {
#define DLI_STREAM(id, bm, bn, ns, wm, wn, bk) \
    case id: return launch_cfg<bm, bn, EPI, ns, wm, wn, bk, true>(DLI_GEMM_PASS);
    DLI_STREAM(60, 32, 32, 3, 2, 1, 256) DLI_STREAM(61, 32, 128, 4, 2, 2, 64)
    DLI_STREAM(62, 32, 64, 3, 2, 2, 256) DLI_STREAM(63, 64, 128, 3, 2, 2, 64)
    DLI_STREAM(64, 64, 64, 5, 2, 2, 64) DLI_STREAM(65, 64, 256, 4, 2, 2, 64)
    DLI_STREAM(66, 96, 128, 4, 1, 4, 64) DLI_STREAM(67, 128, 128, 3, 2, 2, 64)
    DLI_STREAM(68, 128, 256, 3, 2, 4, 64) DLI_STREAM(69, 64, 32, 3, 4, 1, 256)
    DLI_STREAM(70, 96, 64, 4, 2, 2, 64) DLI_STREAM(71, 128, 64, 6, 2, 2, 64)
    DLI_STREAM(72, 128, 32, 4, 4, 1, 128)
#undef DLI_STREAM
    default: return DLI_NOT_MINE;
  }
}

int gemm_stream_pairs_dispatch(int epi, int tile_cfg, DLI_GEMM_ARGS);
int gemm_stream_act_dispatch(int epi, int tile_cfg, DLI_GEMM_ARGS);
int gemm_stream_pairs_set_slab_store(int mode);
int gemm_stream_act_set_slab_store(int mode);
