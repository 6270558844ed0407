// Which tiles a product of more than 64 rows takes, and into how many chains its sums are cut (gemm.hip); which kernel one of fewer takes.  Plain arithmetic, apart from
// the kernels, so that it can be checked on the host.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstddef>

namespace lcu {

constexpr int PLAN_STAGE = 64;  // of K

inline long tiles_of(int M, int N, int rows, int columns) { return (long)((M + rows - 1) / rows) * ((N + columns - 1) / columns); }

// Many rows, few 256x128 tiles and a long K (W2 at 512 rows: 64 tiles, K = 11008): with one tile per
// workgroup most compute units idle, with smaller tiles every workgroup reads more operand bytes per
// multiply-add than its load path delivers.  So the large tiles stay and the K stages of each are
// dealt to cus / tiles workgroups, partial sums through the workspace -- when that leaves at least
// 40 stages per workgroup: the partial sums cost a second launch and M * N * 4 bytes per split each
// way (K = 11008, N = 4096: 73 -> 59 us with four splits; K = 4096, N = 4096: 25 -> 36 us with two).
// Returns the number of splits, 0 when the shape does not suit it.
inline int large_tile_splits(int M, int K, int N, int n_mats, long cus, size_t workspace_bytes) {
  const long tiles = tiles_of(M, N, 256, 128) * n_mats;
  long splits = std::min<long>(cus / tiles, 8);
  splits = std::min<long>(splits, K / PLAN_STAGE / 40);
  if (M <= 64 || splits < 2 || (size_t)splits * M * N * n_mats * sizeof(float) > workspace_bytes) {
    return 0;
  }
  return (int)splits;
}

// The tiles of a product whose K is whole stages of 128, and with them the order of its sums: one ascending chain, but `splits` chains of
// neighbouring stages in split_large, and the even and the odd stages in halves.
enum class row_tiles {
  large,        // 256 rows by 128, 192 or 256 columns
  split_large,  // 256x128, K dealt to `splits` workgroups
  medium,       // 128x128
  narrow,       // 128x64, two to a compute unit
  halves        // 128x64, one to a compute unit
};
struct row_plan_t {
  row_tiles tiles;
  int splits;
};
inline row_plan_t plan_rows(int M, int K, int N, int n_mats, long cus, size_t workspace_bytes) {
  if (tiles_of(M, N, 256, 128) * n_mats >= 160) return {row_tiles::large, 1};
  const int splits = large_tile_splits(M, K, N, n_mats, cus, workspace_bytes);
  if (splits > 0) return {row_tiles::split_large, splits};
  if (tiles_of(M, N, 128, 128) * n_mats >= 160) return {row_tiles::medium, 1};
  return {tiles_of(M, N, 128, 64) * n_mats > 256 ? row_tiles::narrow : row_tiles::halves, 1};
}

// Rows and columns of the tiles of a product that a round of 128x64 ones (row_tiles::halves) or a few large ones with K dealt to `splits`
// workgroups each leave compute units idle with: the smallest that still come out as one round.  What bounds these is the bytes
// that a compute unit brings into LDS for a stage, lhs and columns, 24 KB with 128x64, 16 KB with 64x64, 12 KB with 64x32 (`narrowest`; codes would be
// converted once more: 200 rows of width 2048, eight uint8 layers 0.87 ms with 64x64, 0.90 so); with two to a compute unit they meet there again
// (us with weights from memory, 128x64 / 64x64 / 64x32, workgroups in brackets: fp16 90x4096x4096 25.8 (64) / 20.0 (128) / 18.8 (256), 200 rows 27.7 (128) / 20.5 (256) /
// 26.0 (512), 300 rows 28.3 (192) / 31.5 (320); uint8 200 rows 32.5 / 22.5, 300 rows 33.7 / 37.1).  The sums are those of larger tiles.
// each: matrices times splits.
struct tile_size_t {
  int rows, columns;
};
inline tile_size_t plan_tile_size(int M, int N, int each, tile_size_t largest, bool narrowest, long cus) {
  constexpr tile_size_t sizes[] = {{64, 32}, {64, 64}, {128, 64}, {128, 128}, {256, 128}};
  for (tile_size_t t : sizes) {
    if (t.columns == 32 && !narrowest) continue;
    if ((t.rows == largest.rows && t.columns == largest.columns) || tiles_of(M, N, t.rows, t.columns) * each <= cus) return t;
  }
  return largest;
}

// Whether a gated product of less than 160 tiles of 128x128 takes 128x64 tiles of gemm_tile_kernel or smaller ones of gemm_dl_kernel.  The former's ring of four
// stages hides the way from memory over a long K, but leaves a compute unit one workgroup: weights that may lie in a cache, and more tiles than one
// round, are sooner with the latter.  us, gemm_dl_kernel / gemm_tile_kernel, from memory: 100 rows of 11264 columns, K 1536, 1792, 2048 17.6 / 17.7, 19.4 / 18.6,
// 20.9 / 19.3, 258x4096x768 30.7 / 28.0, 133x8192x6656 60.7 / 51.1, 71x17920x5504 124 / 104; 327x3072x5632 (264 tiles) 30.5 / 43.8, 637x1792x3456 (270) 20.0 /
// 30.1.  The same weights again and again 258x4096x768 24.7 / 27.9, 134x5632x3200 32.6 / 36.6, 378x8192x4096 49.6 / 53.3, 309x2048x5632 (264) 21.6 / 33.9.
inline bool gated_on_tiles(int M, int K, int N, long cus, bool memory) { return memory && K >= 1792 && tiles_of(M, N, 128, 64) <= cus; }

// Which columns of a product a launch of gemm_tile_kernel takes: the first `tiles` tiles along N, counted through the matrices
// (0: all of them), or those from column `from` of the last matrix on.
struct columns_t {
  int tiles = 0, from = 0;
};

// Tiles of a product that fills most of the chip with those of 256x128: `columns` wide, of 256 rows (128 up to 128 rows); from column `from` of
// the last matrix on, where that is not 0, tiles of rest_rows x rest_columns in a launch of their own.
struct large_tiles_t {
  int columns;
  columns_t first, rest;
  int rest_rows, rest_columns;
};

enum class product_type { f16, bf16, bf16_gated, u8 };

// What a round of workgroups takes, in us: a part that goes with K, per 4096 of it, and what a tile pays before its first and behind its last
// stage, which is outputs above all; more of that where rows of outputs begin off 16 bytes.  Fitted to the times of every width, and of whole rounds
// with each kind of rest, for 23 000 drawn products of 129 to 2600 rows with weights from memory; the plan with the least sum of rounds is within
// 0.5 % of the best one of a product on average.  With one figure per width for all types and K, lcu_linear was up to 1.3 times as long as
// with 128 columns (bfloat16 1099x640x6639 46.8 us / 25.9, 1224x1152x17920 70.0 / 61.3) and uint8 of K 512 had 128 columns only (264x512x17920 27.6 us, 192 columns 20.3).
struct round_cost_t {
  double per_4096, tile, ragged;
};
inline round_cost_t round_cost(product_type type, int columns, bool half_rows = false) {
  if (half_rows) return type == product_type::u8 ? round_cost_t{38.5, 4, 0} : type == product_type::f16 ? round_cost_t{34, 4, 0} : round_cost_t{35, 5.5, 0};
  const int w = columns == 128 ? 0 : columns == 192 ? 1 : 2;
  const round_cost_t f16[3] = {{48, 5, 1.5}, {65, 10, 4}, {81, 13.5, 5}}, bf16[3] = {{44, 5.5, 1.5}, {60, 18, 4}, {75, 18, 5}};
  const round_cost_t gated[3] = {{44, 6.5, 1.5}, {60, 13, 4}, {75, 16, 5}}, u8[3] = {{53, 7.5, 1.5}, {71.5, 10.5, 4}, {96, 14, 5}};
  return type == product_type::f16 ? f16[w] : type == product_type::bf16 ? bf16[w] : type == product_type::bf16_gated ? gated[w] : u8[w];
}

// The tiles whose rounds of workgroups cost least.  A last round that is nearly empty goes to smaller tiles: whole rounds of one width, then the
// columns that are left in those tiles that cost least (us, the best single width / so: uint8 512 rows, K 6656, twice 17920 columns 254 / 234; fp16
// K 4096, twice 11008 columns, 700 rows 143 / 136, 1000 rows 164 / 158, 1987 rows 300 / 290), by a launch that costs 4 us more; below 1024 of K
// that is what it gains.
// Gated outputs come in pairs of 32 columns and 32 columns behind them, so there 192 columns go to each of four wavefronts of 64 rows
// (bfloat16, us with 128 and 256 columns only / so: 512x4096x22016 104 / 84, 1500 rows 260 / 236, 1987x2048x5632 57 / 46).
// Up to 128 rows: tiles of 128 rows, a round of 128 / 256 columns taking 52 / 66 us in fp16 and 42 / 62 in uint8 (100
// rows, twice 11008 columns 61 -> 52 us and 55 -> 42 against tiles of 256 rows; twice 17920 of K 6656 140 -> 118 and 170 -> 109).
inline large_tiles_t plan_large(product_type type, int M, int K, int N, int n_mats, long cus, bool ragged) {
  const auto rounds = [&](long n) { return (n + cus - 1) / cus; };
  if (M <= 128) {
    const bool u8 = type == product_type::u8;
    const long c128 = rounds(tiles_of(M, N, 128, 128) * n_mats) * (u8 ? 42 : 52), c256 = rounds(tiles_of(M, N, 128, 256) * n_mats) * (u8 ? 62 : 66);
    return {c256 < c128 ? 256 : 128, {}, {}, 0, 0};
  }
  const auto cost = [&](long n, int columns, bool half_rows = false) {
    const round_cost_t c = round_cost(type, columns, half_rows);
    return (double)rounds(n) * (c.per_4096 * K / 4096 + c.tile + (ragged ? c.ragged : 0));
  };
  large_tiles_t best{128, {}, {}, 0, 0};
  double least = cost(tiles_of(M, N, 256, 128) * n_mats, 128);
  for (int columns : {192, 256}) {
    const double c = cost(tiles_of(M, N, 256, columns) * n_mats, columns);
    if (c < least) {
      least = c;
      best.columns = columns;
    }
  }
  if (K < 1024) return best;
  const long tiles_m = (M + 255) / 256;
  for (int columns : {256, 192, 128}) {
    const long per = (N + columns - 1) / columns, whole = per * n_mats * tiles_m / cus, first = whole * cus / tiles_m;
    const long from = (first - per * (n_mats - 1)) * columns;
    if (whole == 0 || from <= 0 || from >= N) continue;  // what is left lies in the last matrix
    const int left = N - (int)from;
    for (int rest : {0, 128, 192}) {  // 0: tiles of 128x128
      const double last = rest == 0 ? cost(tiles_of(M, left, 128, 128), 128, true) : cost(tiles_of(M, left, 256, rest), rest);
      const double c = cost(whole * cus, columns) + last + 4;
      if (c < least) {
        least = c;
        best = {columns, {(int)first, 0}, {0, (int)from}, rest == 0 ? 128 : 256, rest == 0 ? 128 : rest};
      }
    }
  }
  return best;
}

// More than 64 rows of one matrix whose chains plan_rows keeps apart, with the chains' sums left in the workspace for the launch that goes on with
// them: how many, 0 where they are not.  Splits lie there in any case; the even and the odd stages are dealt to workgroups of 128x128 tiles
// (step 2) where that gains more than the sums cost on their way through memory, and where the workspace is the stream's own: the separate
// kernels use none, so that such calls may overlap on streams that share the device's.  Over a short K one launch fewer counts, over a long
// one the tiles do, in between both less (product, residual and norm, separate / here, us: fp16 80x4096x4096 30 / 24, 256 rows 33 / 29, 512 rows
// 35.5 / 34.7, 1301x1408x512 15.7 / 17.3, 1096x1152x512 14.6 / 15.7; uint8 512x4096x4096 45 / 39, 700x2048x2048 25.1 / 23.1, 693x1408x2048
// 20.2 / 22.0, 1290x768x512 14.9 / 16.3; of 7270 drawn products that these lines take 6 are more than 3 % slower so, on average they take 0.8 of
// the time).  That was against separate products on gemm_dl_kernel.  On the 128x64 tiles of gemm_tile_kernel, which they take now, they are ahead of some
// that these lines take (fp16 80x4096x4096 27.6 / 24.9, 256 rows 31.1 / 29.5, 400 rows 26.9 / 27.7, 512 rows 32.0 / 32.7, 200x2048x2048 16.2 / 16.6;
// uint8 300x1152x1030 19.3 / 16.4, 512x4096x4096 34.3 / 35.4, 700x2048x2048 19.7 / 22.2).  Where the tiles of either are smaller now (plan_tile_size) both
// are sooner than these figures.
struct left_sums_t {
  int splits, step;
};
inline left_sums_t plan_left_sums(bool u8, int M, int K, int N, long cus, size_t workspace_bytes, bool owned) {
  const row_plan_t plan = plan_rows(M, K, N, 1, cus, workspace_bytes);
  if (plan.tiles == row_tiles::split_large) return {plan.splits, 1};
  if (plan.tiles != row_tiles::halves || !owned || (size_t)2 * M * N * sizeof(float) > workspace_bytes) return {0, 1};
  const int limit = u8 ? (K > 512 && K < 2048 ? 832 : 1024) : K > 1024 && K < 2800 && N <= 1024 ? 384 : 512;
  if ((size_t)M * N > (size_t)K * limit) return {0, 1};
  return {2, 2};
}

// Rows of a tile for the products of `rows` rows sorted by expert with matrices [2 ff][K] (gated) and [K][ff]: those whose tiles cost least.  An expert
// that a tile does not hold asks for its weights once more, but larger tiles are fewer, and where the product has few of them compute units idle
// (4 experts of 256 hidden columns, 4096 wide, 260 rows: 64-row tiles 37 us, 128 46; top 2 of 16 of 2816, 512 tokens 284, 238, of 256 rows 272, 1000
// tokens 346, 307, 289).  Cost of a round of workgroups (64-row tiles go two to a compute unit) and of what is in it, fitted to 12 600 drawn
// sets with weights from memory; the choice takes 1 % more than the best one on average.  By rows to an expert alone (128 from 52, 256 from 104) a third of
// the sets with 52 rows and more took 3 to 25 % longer than with the lines at 96 and 384.
inline int plan_expert_rows(long rows, int experts, int K, int ff, long cus) {
  const auto cost = [&](int tile, double round, double each, double work, int per_cu) {
    const double mean = (double)rows / experts, tiles = experts * std::ceil((mean + 1.5 * std::sqrt(mean)) / tile);  // few groups are larger
    const auto product = [&](int k, int n) {
      const double full = tiles * ((n + 127) / 128) / (double)(per_cu * cus), rounds = std::ceil(full);
      return rounds * (round * k / 4096 + each) + full * work * k / 4096;
    };
    return product(K, 2 * ff) + product(ff, K);  // us
  };
  const double c64 = cost(64, 17.4, 3, 53, 2), c128 = cost(128, 24.8, 3.8, 19, 1), c256 = cost(256, 34.3, 5.1, 19, 1);
  return c64 <= c128 && c64 <= c256 ? 64 : c128 <= c256 ? 128 : 256;
}

// ---- 2 to 64 rows (gemm_stream.hpp) ----
constexpr int stream_max_waves(bool u8) { return u8 ? 10 : 12; }  // LDS: 160 KB

// Whether weights come from memory: a program goes through `known` bytes of them before it is back at the same ones (lcu_stream_weights), or one launch
// through `bytes`, and the 256 MB cache in front of memory holds neither.  Other weights may lie there, and what is right for them is another
// matter (streams, stream_once).  One product again and again, us as from a cache / as from memory: fp16 of 273 MB 8 rows 43.7 / 44.0, 40 rows 46.6 / 50.3,
// 328 MB 8 rows 62.8 / 56.9, 426 MB 24 rows 79.4 / 73.7, uint8 of 321 MB 40 rows 187 / 161.
constexpr size_t FROM_MEMORY = (size_t)320 << 20;
inline bool from_memory(size_t known, size_t bytes) { return std::max(known, bytes) > FROM_MEMORY; }

// Whether a launch of `bytes` of weights marks them as read once, which keeps their lines out of that cache.  us, unmarked / marked, weights from memory:
// fp16 8x6656x6656 21.9 / 20.3, 24x4096x11008 22.9 / 21.6, 8x6656x17920 48.4 / 43.5; the same ones again and again 19.6 / 18.7, 19.8 / 20.4,
// 40.5 / 42.5, 60 rows 42.5 / 48.1, 60x6656x6656 22.7 / 24.7.  Smaller launches' weights may stay there beside marked ones: eight fp16 layers of width 4096, 20 sequences, 1007 us a step with
// Wo unmarked, 1024 with it marked (at width 2048, where nearly all are smaller, three layers 255 / 242).
inline bool stream_once(bool memory, size_t bytes) { return memory && bytes >= (size_t)64 << 20; }

// Wavefronts (of 16 columns) per workgroup of gemm_stream_kernel: one workgroup runs per compute unit, so the longest
// compute unit has rounds * wavefronts of them to stream; below four a compute unit has too little in flight (8 rows, three
// times 2048x2048: nine rounds of single wavefronts 19.6 us, one of ten 10.7).  *rounds: how many they are.
inline int stream_waves(int N, int n_mats, int splits, long cus, int most, long* rounds) {
  const long groups = (N + 15) / 16;
  int best = 1;
  long least = 0;
  for (int w = 1; w <= most; ++w) {
    const long wgs = (groups + w - 1) / w * n_mats * splits;
    const long cost = (wgs + cus - 1) / cus * std::max(w, 4);
    if (w == 1 || cost <= least) {
      least = cost;
      best = w;
      *rounds = (wgs + cus - 1) / cus;
    }
  }
  return best;
}

// How many workgroups the K stages of BM x 128 tiles are dealt to, and the workgroups in all; splits 0: too few of them, or no room for the sums.
struct skinny_plan_t {
  int splits;
  long tiles;
};
inline skinny_plan_t plan_skinny(int BM, int M, int K, int N, int n_mats, int cus, size_t workspace_bytes) {
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + 127) / 128 * n_mats, nt_all = K / PLAN_STAGE;
  // one workgroup per compute unit and at least four stages each: more, shorter splits only add
  // partial sums (512 workgroups: 16 against 13 us at N = K = 4096)
  int splits = (cus + tiles_m * tiles_n - 1) / (tiles_m * tiles_n);
  splits = std::max(1, std::min(splits, nt_all / 4));
  const size_t each = (size_t)M * N * n_mats * sizeof(float);
  while (splits > 1 && splits * each > workspace_bytes) --splits;
  if (splits * each > workspace_bytes || (long)tiles_m * tiles_n * splits < cus / 2) return {0, 0};
  return {splits, (long)tiles_m * tiles_n * splits};
}

// Whether a product of few rows is one of gemm_stream_kernel, or of BM x 128 tiles of four wavefronts.  Of those several share a
// compute unit; a workgroup here has it alone, so that a second round fills lhs and ring again with nothing beside it, which a long enough run
// of stages pays for.  us with weights from memory, tiles / here: two rounds, fp16 8 rows of 32000 columns, K 2048, 2560, 4096, 6656 29.4 / 32.7, 33.6 / 31.0,
// 62.2 / 54.7, 79.1 / 71.0, 24 rows 30.8 / 35.4, 43.2 / 41.0 (K 3072), 66.9 / 60.9, 64 rows of K 4096 71.9 / 68.0; uint8 32 rows, K 4096, 6656
// 46.3 / 44.0, 70.1 / 61.9, 48 rows 76.3 / 76.2, 16 rows of 4096x11008 twice 36.6 / 32.7; three rounds, 5888x9664 three times 62 / 67.
// One round: uint8 gains, but over short runs (15x512x10304 twice 10.3 / 11.4); fp16 where the tiles (`tiles` in all, with their splits) do not come out
// even (27x17920x6656 62 / 45), or over runs of some stages (10x1024x7304 8.6 / 9.2; 24x4096x4096 13.3 / 13.3, 24x6144x4096 16.4 / 15.7, 20x11008x4096
// 23.6 / 22.2, 20x8192x8192 36.5 / 33.0; 50 rows 18.3 / 18.3, 8192x4096 20.9 / 21.2, 8192x8192 64 rows 39.5 / 35.1).  bfloat16 gains at every count (4x512x3264
// 9.2 / 7.9, 46x17920x6656 68 / 50).  Neither does for more than 16 rows over the shortest runs (28x512x16840 10.5 / 11.1, bfloat16
// 56x512x16576 13.8 / 14.8).  Weights that may lie in a cache keep the lines that are right for them there (tiles / here from a cache: 64x8192x8192 26.6 / 34.0,
// 20x8192x8192 23.7 / 30.8, 8x4096x32000 44.0 / 48.8; up to 16 rows of one round 10x1024x7304 7.4 / 8.3, 13x2048x2048 three times
// 9.1 / 10.0).
inline bool streams(int M, int N, int n_mats, int splits, int stages, long tiles, long cus, bool u8, bool bf16, bool memory) {
  long rounds = 1;
  stream_waves(N, n_mats, splits, cus, stream_max_waves(u8), &rounds);
  const int run = stages / splits;
  if (u8) return rounds == 1 || (rounds == 2 && (M <= 16 ? run >= 12 : memory && M <= 32 && run >= 20));
  const bool short_runs = M > 16 && run <= 4;
  if (bf16) return rounds == 1 && (!short_runs || 4 * tiles <= 3 * cus);
  if (rounds == 1) return (tiles > cus && !short_runs) || (M <= 16 ? run >= 8 : memory && run >= (M <= 32 ? 12 : 24));
  return memory && rounds == 2 && run >= 20;
}

}  // namespace lcu
