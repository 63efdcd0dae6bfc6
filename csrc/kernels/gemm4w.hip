// Tiles 34, 41 and 45: 256x256, split-K and grouped products (gemm4w.h). One kernel: the three ids remain from
// kernels that differed in their schedules.
#include "gemm4w.h"

template <int EPI>
static int dispatch_4w(int tile_cfg, DLI_GEMM_ARGS) {
  if (tile_cfg != 34 && tile_cfg != 41 && tile_cfg != 45) return DLI_NOT_MINE;
  return launch_4w<EPI, 8>(DLI_GEMM_PASS);
}

int gemm_4w_dispatch(int epi, int tile_cfg, DLI_GEMM_ARGS) { DLI_EPI_SWITCH_BASE(dispatch_4w) }
