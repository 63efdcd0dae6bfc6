// The 4-wave kernel (gemm4w.h) on tiles of 224, 192, 160 and 128 columns; gemm4w.hip chooses.
#include "gemm4w.h"

template <int NJ> static int launch_nj(int epi, DLI_GEMM_ARGS) {
  switch (epi) {
    case EPI_BF16: return launch_4w<EPI_BF16, NJ>(DLI_GEMM_PASS);
    case EPI_F32: return launch_4w<EPI_F32, NJ>(DLI_GEMM_PASS);
    case EPI_SLAB16: return launch_4w<EPI_SLAB16, NJ>(DLI_GEMM_PASS);
    case EPI_RES: return launch_4w<EPI_RES, NJ>(DLI_GEMM_PASS);
    default: break;
  }
  if constexpr (NJ % 2 == 0) {                     // a gate block and its up block in one wave tile
    if (epi == EPI_SILU) return launch_4w<EPI_SILU, NJ>(DLI_GEMM_PASS);
    if (epi == EPI_GELU_MUL) return launch_4w<EPI_GELU_MUL, NJ>(DLI_GEMM_PASS);
  }
  return DLI_NOT_MINE;
}

int gemm_4w_narrow(int epi, int nj, DLI_GEMM_ARGS) {
  switch (nj) {
    case 7: return launch_nj<7>(epi, DLI_GEMM_PASS);
    case 6: return launch_nj<6>(epi, DLI_GEMM_PASS);
    case 5: return launch_nj<5>(epi, DLI_GEMM_PASS);
    case 4: return launch_nj<4>(epi, DLI_GEMM_PASS);
    default: return DLI_NOT_MINE;
  }
}
