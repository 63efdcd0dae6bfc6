// Weight-streaming tiles: plain, fp32 and fp16-slab epilogues, and the family's dispatch.
#include "gemm_stream.h"

int gemm_stream_dispatch(int epi, int tile_cfg, DLI_GEMM_ARGS) {
  switch (epi) {
    case EPI_BF16: return dispatch_stream<EPI_BF16>(tile_cfg, DLI_GEMM_PASS);
    case EPI_F32: return dispatch_stream<EPI_F32>(tile_cfg, DLI_GEMM_PASS);
    case EPI_SLAB16:
      if (C != nullptr || splits < 2) return (int)hipErrorInvalidValue;
      return dispatch_stream<EPI_SLAB16>(tile_cfg, DLI_GEMM_PASS);
    default: break;
  }
  if (epi_pairs(epi)) return gemm_stream_pairs_dispatch(epi, tile_cfg, DLI_GEMM_PASS);
  return gemm_stream_act_dispatch(epi, tile_cfg, DLI_GEMM_PASS);
}

int gemm_stream_set_slab_store(int mode) {
  gemm_stream_pairs_set_slab_store(mode);
  gemm_stream_act_set_slab_store(mode);
  return set_slab_store_tu(mode);
}
