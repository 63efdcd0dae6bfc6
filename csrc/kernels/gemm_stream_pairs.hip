// Weight-streaming tiles: epilogues that pair a gate block with the up block beside it.
#include "gemm_stream.h"

int gemm_stream_pairs_dispatch(int epi, int tile_cfg, DLI_GEMM_ARGS) {
  switch (epi) {
    case EPI_SILU: return dispatch_stream<EPI_SILU>(tile_cfg, DLI_GEMM_PASS);
    case EPI_CLAMP: return dispatch_stream<EPI_CLAMP>(tile_cfg, DLI_GEMM_PASS);
    case EPI_RELU: return dispatch_stream<EPI_RELU>(tile_cfg, DLI_GEMM_PASS);
    case EPI_GELU_MUL: return dispatch_stream<EPI_GELU_MUL>(tile_cfg, DLI_GEMM_PASS);
    default: return DLI_NOT_MINE;
  }
}

int gemm_stream_pairs_set_slab_store(int mode) { return set_slab_store_tu(mode); }
