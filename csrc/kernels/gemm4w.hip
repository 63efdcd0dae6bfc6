// Tiles 22, 28, 34, 41, 45 and 55 on the 4-wave kernel (gemm4w.h): 256 columns here, narrower ones in
// gemm4w_narrow.hip, tiles of 192 and 320 rows in gemm4w_rows192.hip and gemm4w_rows320.hip, and the rules that choose
// between them.
//   34, 41, 45  256 columns (three ids from kernels that differed in their schedules)
//   22          256 columns, or by rounds as below where the product is dense and not biased
//   28          128 columns
//   55          256, 192 or 160 by rounds; dense, unsplit, K a multiple of 128
// 22 and 55 take 192 or 320 rows instead of 256 where those fill the rounds better (shape_of).
// Against the 8-phase kernels that 22 and 28 were (gemm8p.hip keeps what is not built here), us, on gemm4w.h's card:
// 16384 x 6144 x 4096 591 -> 540, 8192 x 4096 x 14336 663 -> 632, 8192 x 28672 with SiLU pairs 1348 -> 1248, 4096 x
// 2304 x 768 with a bias 33 -> 24.5; partial sums in 16 bits of 512 rows: 6144 x 4096 in four 32.4 -> 26.0, 4096 x
// 4096 in four 23.0 (tile 28) -> 19.5, 4096 x 14336 in eight 52 -> 47.
#include "gemm4w.h"

int gemm_4w_narrow(int epi, int nj, DLI_GEMM_ARGS);
int gemm_4w_rows192(int epi, int nj, DLI_GEMM_ARGS);
int gemm_4w_rows320(int epi, int nj, DLI_GEMM_ARGS);

// The tile width, in 32 columns, whose rounds take least. A round's price is its width times what the narrower
// schedule costs more (fewer MFMAs between the same barriers: 1.6, 5, 9 and 15 %), the last one's by how many CUs
// it keeps, and little less for few of them, which clock higher. 256 columns unless another is 3 % better.
// K = 4096, bf16 outputs, 16 columns of tiles, us at 256 / 224 / 192 / 160 / 128: a quarter of a round 69 / 62 / 54
// / 48 / 40, three 80 / 74 / 64 / 57 / 47, one round 95 / 84 / 75 / 65 / 54, 1.25 155 / 139 / 122 / 106 / 88, 1.75
// 173 / 154 / 133 / 117 / 98, two 186 / 166 / 147 / 127 / 105; K = 1024 and 14336 and fp32 outputs within 5 % of the
// same ratios. Tile 55 chooses among 8, 6 and 5, its widths where the LM head's block maxima are laid out by them
// (ops/gemm.py's persistent_width is its copy).
static double cost_of(int M, int N, int splits, int mi, int nj, double price) {
  const double cus = cu_count();
  const long tiles = (long)((M + 32 * mi - 1) / (32 * mi)) * ((N + 32 * nj - 1) / (32 * nj)) * splits;
  const double whole = (double)(tiles / (long)cus), x = tiles / cus - whole;
  const double last = x == 0 ? 0.0 : whole == 0 ? 0.72 + 0.28 * x * x * x
                                                : 0.60 + 0.25 * x + 0.15 * x * x * x;
  return (whole + last) * price;
}
static const double PRICE[9] = {0, 0, 0, 0, 0.573, 0.684, 0.794, 0.889, 1.0};

static int width_of(int M, int N, int splits, bool pairs, bool all) {
  int best = 8;
  double least = 0.0;
  for (int nj = 8; nj >= 4; --nj) {
    if ((!all && (nj == 7 || nj == 4)) || (pairs && nj & 1)) continue;
    const double c = cost_of(M, N, splits, 8, nj, PRICE[nj]);
    if (nj == 8) least = 0.97 * c;
    else if (c < least) { least = c; best = nj; }
  }
  return best;
}

static int launch8(int epi, DLI_GEMM_ARGS) {
  switch (epi) {
    case EPI_BF16: return launch_4w<EPI_BF16, 8>(DLI_GEMM_PASS);
    case EPI_F32: return launch_4w<EPI_F32, 8>(DLI_GEMM_PASS);
    case EPI_SILU: return launch_4w<EPI_SILU, 8>(DLI_GEMM_PASS);
    case EPI_GELU_MUL: return launch_4w<EPI_GELU_MUL, 8>(DLI_GEMM_PASS);
    case EPI_BIAS: return launch_4w<EPI_BIAS, 8>(DLI_GEMM_PASS);
    case EPI_BIAS_GELU: return launch_4w<EPI_BIAS_GELU, 8>(DLI_GEMM_PASS);
    case EPI_SLAB16: return launch_4w<EPI_SLAB16, 8>(DLI_GEMM_PASS);
    case EPI_RES: return launch_4w<EPI_RES, 8>(DLI_GEMM_PASS);
    default: return DLI_NOT_MINE;
  }
}

static int g_store_mode = 0;
int gemm_4w_set_slab_store(int mode) { return std::exchange(g_store_mode, mode); }
int gemm_4w_store_mode() { return g_store_mode; }

// a tile's columns, in 32, for a product
static int columns(int tile_cfg, int epi, int M, int N, int splits, bool grouped) {
  if (tile_cfg == 28) return 4;
  // (the biased epilogues, which few products take, are built in one width)
  const bool bias_epi = epi == EPI_BIAS || epi == EPI_BIAS_GELU;
  if ((tile_cfg != 22 && tile_cfg != 55) || grouped || bias_epi) return 8;
  return width_of(M, N, splits, epi_pairs(epi), tile_cfg == 22);
}

// The rows and columns of a tile, in 32. A product of some hundred to some thousand rows is a round or a few of them, and whole
// tiles of 256 rows leave up to a quarter of the last row of tiles or of the last round empty; tiles of 192 or 320 rows,
// at their own price of a full round (measured as above, 16 x 16 tiles; 192 x 320 columns 0.947, x 256 0.779, x 192 0.610, x
// 128 0.456, 320 x 192 0.935, x 128 0.675), are taken where by the same reckoning they cost 3 % less; 6 % with 8192 and
// more of K. In launches of up to a round, or of two rows of tiles, the smaller ones 7 %: there few tiles share what each reads, and two shapes that
// move as many bytes take as long however many products they have (so 128 columns are 8 % dearer with such K, 320 x 128
// another 5). us, the best of 256 rows and the one taken: 2112 rows, 6144 x 4096 81 -> 77, 4096 x 4096 60 -> 55, 4096 x 14336 187 ->
// 173, 28672 x 4096 344 -> 331; 1100 rows 4096 x 4096 44 -> 39, 4096 x 14336 137 -> 123; 600 rows 41 -> 37, 41 -> 37, 126 ->
// 113, 118 -> 106; 5000 rows, 4096 x 14336 453 -> 406; fp32 outputs, 7623 x 12288 x 4096 562 -> 554, 8199 x 16384 x
// 4096 844 -> 822, 9000 x 4096 x 14336 829 -> 769. Of 629 products of 260 to 16384 rows that 3 % alone would have moved, 33
// were slower by over 1 %, by up to 14 (820 x 8192 x 5120 with SiLU pairs 60 -> 65, 640 x 14336 x 14336 229 -> 248); of the
// 480 that this takes 3 are, by up to 3. 1247 others, drawn and on a grid, take 0.90 of the former time in the mean, 26 of
// them over 1 % more, the worst 6 (520 x 11008 x 11008). Every
// shape adds a product's terms in one order, so that the choice does not change a bit. Not for short K, whose tiles are mostly
// epilogue, nor where block maxima are laid out by the width or rows lie too far apart for 320 of them (such a
// product is not a plain one).
struct Shape { int mi, nj; };
static Shape shape_of(int tile_cfg, int epi, int M, int N, int K, int splits) {
  Shape best{8, columns(tile_cfg, epi, M, N, splits, false)};
  const bool bias_epi = epi == EPI_BIAS || epi == EPI_BIAS_GELU;
  if ((tile_cfg != 22 && tile_cfg != 55) || bias_epi || K < 1536 || K / splits < 512) return best;
  double least = cost_of(M, N, splits, 8, best.nj, PRICE[best.nj]);
  const bool deep = K / splits >= 8192;
  static const struct { int mi, nj; double price; } other[] = {{6, 10, 0.947}, {6, 8, 0.779}, {6, 6, 0.610}, {6, 4, 0.456},
                                                              {10, 6, 0.935}, {10, 4, 0.675}};
  for (const auto& o : other) {
    const long rows = (M + 32 * o.mi - 1) / (32 * o.mi), cols = (N + 32 * o.nj - 1) / (32 * o.nj);
    const bool few = rows * cols * splits <= cu_count() || rows <= 2;
    double c = cost_of(M, N, splits, o.mi, o.nj, o.price) / (few && o.mi * o.nj < 60 ? 0.93 : !few && deep ? 0.94 : 0.97);
    if (few && o.nj == 4) c *= (o.mi == 10 ? 1.05 : 1.0) * (deep ? 1.08 : 1.0);
    if (c < least) { least = c; best = {o.mi, o.nj}; }
  }
  return best;
}

int gemm_4w_dispatch(int epi, int tile_cfg, DLI_GEMM_ARGS) {
  switch (tile_cfg) {
    case 34: case 41: case 45:
      if (epi == EPI_GELU_MUL || epi == EPI_SLAB16) return DLI_NOT_MINE;
      break;
    case 22:
      if (epi_pairs(epi) && N % 64) return (int)hipErrorInvalidValue;
      break;
    case 28:
      break;
    case 55:
      if (epi == EPI_SLAB16) return DLI_NOT_MINE;
      if (splits != 1 || go != nullptr || K % (2 * BK) || C == nullptr) return (int)hipErrorInvalidValue;
      break;
    default: return DLI_NOT_MINE;
  }
  if (epi == EPI_SLAB16 && (C != nullptr || splits < 2)) return (int)hipErrorInvalidValue;
  const int nj = columns(tile_cfg, epi, M, N, splits, go != nullptr);
  const bool plain = go == nullptr && !(epi == EPI_F32 && bias != nullptr) && lda < MAX_LD<10> && ldw < MAX_LD<10>;
  const Shape s = plain ? shape_of(tile_cfg, epi, M, N, K, splits) : Shape{8, nj};
  switch (s.mi) {
    case 6: return gemm_4w_rows192(epi, s.nj, DLI_GEMM_PASS);
    case 10: return gemm_4w_rows320(epi, s.nj, DLI_GEMM_PASS);
    default: return s.nj == 8 ? launch8(epi, DLI_GEMM_PASS) : gemm_4w_narrow(epi, s.nj, DLI_GEMM_PASS);
  }
}

// the rows of the tiles of a plain product
extern "C" int dli_gemm_4w_rows(int tile_cfg, int epi, int M, int N, int K, int splits) {
  return 32 * shape_of(tile_cfg, epi, M, N, K, splits).mi;
}
// the columns that a tile (22, 28, 34, 41, 45 or 55) of 256 rows has for a dense product
extern "C" int dli_gemm_4w_width(int tile_cfg, int epi, int M, int N, int splits) {
  return 32 * columns(tile_cfg, epi, M, N, splits, false);
}
