// The 4-wave kernel (gemm4w.h) on tiles of 192 rows; gemm4w.hip chooses.
#include "gemm4w.h"

int gemm_4w_rows192(int epi, int nj, DLI_GEMM_ARGS) {
  switch (nj) {
    case 10: return launch_nj<10, 6>(epi, DLI_GEMM_PASS);
    case 8: return launch_nj<8, 6>(epi, DLI_GEMM_PASS);
    case 6: return launch_nj<6, 6>(epi, DLI_GEMM_PASS);
    case 4: return launch_nj<4, 6>(epi, DLI_GEMM_PASS);
    default: return DLI_NOT_MINE;
  }
}
