// The 4-wave kernel (gemm4w.h) on tiles of 320 rows; gemm4w.hip chooses.
#include "gemm4w.h"

int gemm_4w_rows320(int epi, int nj, DLI_GEMM_ARGS) {
  switch (nj) {
    case 6: return launch_nj<6, 10>(epi, DLI_GEMM_PASS);
    case 4: return launch_nj<4, 10>(epi, DLI_GEMM_PASS);
    default: return DLI_NOT_MINE;
  }
}
