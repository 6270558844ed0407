// Linear layers of the layered decoders: operand conventions and epilogues shared by the bfloat16
// matrix-core kernel (gemm.hip) and the 32-bit one (linear.hip).
//
// An activation is bfloat16 or fp32 ("element type", LCU_BF16 / LCU_F32); products accumulate in
// fp32.  Rows of activations and of weights are padded with zeros to a multiple of 64 elements, so
// every K is one.
#pragma once
#include "common.hpp"

namespace lcu {

__device__ __forceinline__ float sigmoid_f32(float z) { return 1.0f / (1.0f + expf(-z)); }

// 0.5 z (1 + tanh(sqrt(2 / pi) (z + 0.044715 z^3)))
__device__ __forceinline__ float gelu_tanh(float z) {
  const float inner = 0.7978845608028654f * (z + 0.044715f * z * z * z);
  return 0.5f * z * (1.0f + tanhf(inner));
}

// min(g, limit), clamp(u, -limit, limit), then g sigmoid(alpha g) (u + up_shift)
struct clamped_gate {
  float limit, alpha, up_shift;
  __device__ __forceinline__ float operator()(float g, float u) const {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    return g * sigmoid_f32(alpha * g) * (u + up_shift);
  }
};

// Rows that are sorted by group (expert): row tile t belongs to group tile_group[t], starts at row
// tile_row[t] and ends at the group's end; group g multiplies matrix W + g * group_stride bytes; row r of lhs
// is row row_index[r] of the array when row_index is given.  Products of ungrouped rows have none of this.
template <bool GROUPED>
struct row_groups {};
template <>
struct row_groups<true> {
  const float* row_scale;  // factor of row r of lhs, or nullptr (gated products only)
  const int* tile_group;
  const int* tile_row;
  const int* group_end;
  const int* n_tiles;
  const int* row_index;
  int lhs_rows;  // of the array
  size_t group_stride;
  int tile_rows;
};

// Which tile workgroup `bx` takes; group -1: none.  The launch has as many row tiles as the list can ever hold; those that are there are dealt to
// the XCDs in equal runs, group by group, a group's row tiles of the same columns side by side: an XCD's L2 then holds the rows of two or
// three experts, not of all sixteen (512 tokens, top 2 of 16 experts of 4096 x 5632 and 2816 x 4096, 64-row tiles: 199 -> 181 us, 101 -> 92; 2000
// tokens 380 -> 347, 203 -> 193).  A run of the list is found among its 64 entries that hold the tile, so longer ones are cut there.
struct group_tile_t {
  int group, row_tile, column_tile;
};
__device__ __forceinline__ group_tile_t group_tile(const row_groups<true>& g, int columns, int bx) {
  constexpr int XCDS = 8;
  const int lane = threadIdx.x & 63, xcd = bx % XCDS, idx = bx / XCDS;
  const int n_tiles = *g.n_tiles, active = n_tiles * columns, q = active / XCDS, r = active % XCDS;
  if (idx >= q + (xcd < r ? 1 : 0)) return {-1, 0, 0};
  const int at = xcd * q + min(xcd, r) + idx, j = at / columns, block = j & ~63;
  const int mine = g.tile_group[min(block + lane, n_tiles - 1)];
  const int group = __builtin_amdgcn_readlane(mine, j - block);
  const uint64_t others = ~__ballot(mine == group && block + lane < n_tiles);  // bits of the list's other groups
  const uint64_t below = others & ((1ull << (j - block)) - 1), above = others >> (j - block);
  const int first = below ? 64 - __builtin_clzll(below) : 0;
  const int count = (above ? j - block + __builtin_ctzll(above) : 64) - first;
  const int rest = at - (block + first) * columns;
  return {group, block + first + rest % count, rest / count};
}

// GATED: the matrix holds, in blocks of 64 rows, 32 gate rows and the 32 up rows of the same hidden columns.
template <bool GROUPED_, bool GATED_>
struct linear_epilogue : row_groups<GROUPED_> {
  static constexpr bool BF16 = true, GROUPED = GROUPED_, GATED = GATED_, ROTARY = false, PAIRED = false, ONCE = false;
  void* out;
  int ldo;
  bool out_f32;
  const float* bias;         // [N] or nullptr
  int gelu_cols;             // columns below this one pass through the GELU
  float* tail;               // fp32 rows [ld_tail] of the columns from tail_from on, or nullptr
  int tail_from, ld_tail;
  clamped_gate gate;

  __device__ __forceinline__ void put(int m, int n, float v) const {
    const size_t at = (size_t)m * ldo + n;
    if (out_f32) {
      reinterpret_cast<float*>(out)[at] = v;
    } else {
      reinterpret_cast<bf16_t*>(out)[at] = (bf16_t)v;
    }
  }
  __device__ __forceinline__ void store(int m, int n, float v) const {
    if (bias) v += bias[n];
    if (n < gelu_cols) v = gelu_tanh(v);
    if (tail && n >= tail_from) {
      tail[(size_t)m * ld_tail + n - tail_from] = v;
      return;
    }
    put(m, n, v);
  }
  // eight neighbouring columns of `columns`, from a multiple of eight on: in 16-byte pieces, wherever the row begins, but at its end and in the tail
  __device__ __forceinline__ void store8(int m, int n, const float (&x)[8], int columns) const {
    if (n + 8 > columns || (tail && n + 8 > tail_from)) {
      for (int e = 0; e < 8 && n + e < columns; ++e) {
        if constexpr (GATED) {
          put(m, n + e, x[e]);
        } else {
          store(m, n + e, x[e]);
        }
      }
      return;
    }
    float y[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      y[e] = x[e];
      if constexpr (!GATED) {
        if (bias) y[e] += bias[n + e];
        if (n + e < gelu_cols) y[e] = gelu_tanh(y[e]);
      }
    }
    const size_t at = (size_t)m * ldo + n;
    if (out_f32) {
      typedef float4_t any_float4_t __attribute__((aligned(4)));
      any_float4_t* to = reinterpret_cast<any_float4_t*>(reinterpret_cast<float*>(out) + at);
      to[0] = float4_t{y[0], y[1], y[2], y[3]};
      to[1] = float4_t{y[4], y[5], y[6], y[7]};
    } else {
      bf16x8_t v;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = (bf16_t)y[e];
      typedef bf16x8_t any_bf16x8_t __attribute__((aligned(2)));
      *reinterpret_cast<any_bf16x8_t*>(reinterpret_cast<bf16_t*>(out) + at) = v;
    }
  }
  __device__ __forceinline__ void store_gated(int m, int n, float g, float u) const {
    if constexpr (GROUPED) {
      const float s = this->row_scale ? this->row_scale[m] : 1.0f;
      g *= s, u *= s;
    }
    put(m, n, gate(g, u));
  }
};

// experts whose weights come from memory: their lines are marked as read once (gemm_bf16_grouped)
template <bool GATED>
struct read_once : linear_epilogue<true, GATED> {
  static constexpr bool ONCE = true;
};

// gemm.hip
template <bool GATED>
int gemm_bf16(linear_epilogue<false, GATED> const& ep, const void* A, const void* W, int M, int K, int N, hipStream_t st);
template <bool GATED>
int gemm_bf16_grouped(linear_epilogue<true, GATED> const& ep, const void* A, const void* W, int max_tiles, int K, int N,
                      hipStream_t st);

// element access by type
template <class T>
__device__ __forceinline__ float to_f32(T v) { return (float)v; }

}  // namespace lcu
