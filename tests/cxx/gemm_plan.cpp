// The plans of csrc/gemm_plan.hpp and attention_plan.hpp for the tests (gemm_plan.py).
#include "attention_plan.hpp"
#include "gemm_plan.hpp"

using namespace lcu;

extern "C" {

// tiles (order of row_tiles), splits
void rows(int M, int K, int N, int n_mats, long cus, long workspace, int* out) {
  const row_plan_t p = plan_rows(M, K, N, n_mats, cus, (size_t)workspace);
  out[0] = (int)p.tiles;
  out[1] = p.splits;
}

// columns, tiles of the first launch (0: all), first column of the second (0: none), its rows and columns
void large(int type, int M, int K, int N, int n_mats, long cus, int ragged, int* out) {
  const large_tiles_t p = plan_large((product_type)type, M, K, N, n_mats, cus, ragged != 0);
  out[0] = p.columns;
  out[1] = p.first.tiles;
  out[2] = p.rest.from;
  out[3] = p.rest_rows;
  out[4] = p.rest_columns;
}

// splits, step
void left_sums(int u8, int M, int K, int N, long cus, long workspace, int owned, int* out) {
  const left_sums_t p = plan_left_sums(u8 != 0, M, K, N, cus, (size_t)workspace, owned != 0);
  out[0] = p.splits;
  out[1] = p.step;
}

// rows, columns
void tile_size(int M, int N, int each, int largest_rows, int largest_columns, int narrowest, long cus, int* out) {
  const tile_size_t t = plan_tile_size(M, N, each, {largest_rows, largest_columns}, narrowest != 0, cus);
  out[0] = t.rows;
  out[1] = t.columns;
}

// 2 to 64 rows: splits, whether gemm_stream_kernel takes it, whether its weights are marked as read once
void few_rows(int u8, int bf16, int M, int K, int N, int n_mats, long known, long cus, long workspace, int* out) {
  const int tile = M <= 32 || u8 != 0 ? 32 : 64;
  skinny_plan_t p = plan_skinny(tile, M, K, N, n_mats, (int)cus, (size_t)workspace);
  const size_t bytes = (size_t)N * K * n_mats * (u8 != 0 ? 1 : 2);
  const bool memory = from_memory((size_t)known, bytes);
  out[0] = p.splits;
  out[1] = p.splits > 0 && streams(M, N, n_mats, p.splits, K / PLAN_STAGE, p.tiles, cus, u8 != 0, bf16 != 0, memory);
  out[2] = out[1] && stream_once(memory, bytes);
}

// whether weights of which a program goes through `known` bytes are those of a gated product on gemm_tile_kernel
int gated_tiles(int M, int K, int N, long known, long cus) { return gated_on_tiles(M, K, N, cus, from_memory((size_t)known, (size_t)N * K * 2)); }

int expert_rows(long rows, int experts, int K, int ff, long cus) { return plan_expert_rows(rows, experts, K, ff, cus); }

int attention_again(int n_heads, int n_new, int start_pos, long cus) { return scores_again(n_heads, n_new, start_pos, cus); }

}
