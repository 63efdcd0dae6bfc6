// The 4-wave kernel (gemm4w.h) on tiles of 224, 192, 160 and 128 columns; gemm4w.hip chooses.
#include "gemm4w.h"

int gemm_4w_narrow(int epi, int nj, DLI_GEMM_ARGS) {
  switch (nj) {
    case 7: return launch_nj<7>(epi, DLI_GEMM_PASS);
    case 6: return launch_nj<6>(epi, DLI_GEMM_PASS);
    case 5: return launch_nj<5>(epi, DLI_GEMM_PASS);
    case 4: return launch_nj<4>(epi, DLI_GEMM_PASS);
    default: return DLI_NOT_MINE;
  }
}
