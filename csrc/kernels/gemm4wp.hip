// Tile 55: the 4-wave kernel (gemm4w.h) on the tile width that leaves the last round of the chip fullest.
// Unsplit dense products with K a multiple of 128.
#include "gemm4w.h"

// The tile width (8, 6 or 5 times 32 columns) whose rounds take least: a round's price is its width times
// what the narrower schedule costs more (fewer MFMAs between the same barriers: 9 and 13 %), the last one's
// by how many CUs it keeps, and little less for few of them, which clock higher. 256 columns unless
// another is 3 % better. (7 is hardly ever best, and then by as little.) N = 4096, one weight again and again, us at 8 /
// 7 / 6 / 5 (four weights in turn, as in a step: 4352 rows, K = 14336 551 and 412, K = 4096 163 and 125): 2304 rows, K = 14336 241 / 226 / 218 / 202,
// K = 4096 83 / 79 / 74 / 65; 4352 rows 535 / 476 / 424 / 402 and 164 / 149 / 136 / 127; 5120 rows 168 / 153 /
// 149 / 175; 8192 rows, two whole rounds at 8, 195 / 240 / 224 / 240. N = 6144, K = 4096: 2816 rows 164 / 149 /
// 134 / 121, 4096 rows 172 / 159 / 157 / 182. ops/gemm.py's persistent_width is its copy.
static int width_of(int M, int N, bool pairs) {
  const double cus = cu_count();
  const double price[9] = {0, 0, 0, 0, 0, 1.13 * 5 / 8, 1.09 * 6 / 8, 0, 1.0};
  int best = 8;
  double least = 0.0;
  for (int nj = 8; nj >= 5; --nj) {
    if (nj == 7 || (pairs && nj & 1)) continue;
    const long tiles = (long)((M + 255) / 256) * ((N + 32 * nj - 1) / (32 * nj));
    const double whole = (double)(tiles / (long)cus), x = tiles / cus - whole;
    const double last = x == 0 ? 0.0 : whole == 0 ? 0.8 + 0.2 * x * x * x
                                                  : 0.66 + 0.25 * x + 0.09 * x * x * x;
    const double c = (whole + last) * price[nj];
    if (nj == 8) least = 0.97 * c;
    else if (c < least) { least = c; best = nj; }
  }
  return best;
}

template <int EPI>
static int dispatch_4wp(int tile_cfg, DLI_GEMM_ARGS) {
  if (tile_cfg != 55) return DLI_NOT_MINE;
  if (splits != 1 || go != nullptr || K % (2 * BK) || C == nullptr) return (int)hipErrorInvalidValue;
  // (the biased epilogues, which the plans give to other tiles, keep one width)
  const int nj = EPI == EPI_BIAS || EPI == EPI_BIAS_GELU ? 8 : width_of(M, N, epi_pairs(EPI));
  if constexpr (EPI != EPI_BIAS && EPI != EPI_BIAS_GELU) {
    if (nj == 6) return launch_4w<EPI, 6>(DLI_GEMM_PASS);
    if constexpr (!epi_pairs(EPI)) {
      if (nj == 5) return launch_4w<EPI, 5>(DLI_GEMM_PASS);
    }
  }
  return launch_4w<EPI, 8>(DLI_GEMM_PASS);
}

int gemm_4wp_dispatch(int epi, int tile_cfg, DLI_GEMM_ARGS) {
  if (epi == EPI_GELU_MUL) return dispatch_4wp<EPI_GELU_MUL>(tile_cfg, DLI_GEMM_PASS);
  DLI_EPI_SWITCH_BASE(dispatch_4wp)
}

// the columns of the tiles that the persistent kernel takes for a product
extern "C" int dli_gemm_persistent_width(int M, int N, int pairs) { return 32 * width_of(M, N, pairs != 0); }
