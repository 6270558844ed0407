// Every buffer request that gemm_tile_kernel and gemm_stream_kernel make for a set of shapes, walked on the host with
// the kernels' own arithmetic (csrc/operand_range.hpp) in the order of their loops: whatever a request may reach lies in
// its operand, under either reading of a raw buffer's range check.  Argument "offset": the scalar offset stays when the
// length becomes 0; "columns": two matrices whose columns alternate are clamped at the columns of both.  The walk must then
// find requests past the end (and says so by its exit code).
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstring>

#include "operand_range.hpp"

namespace {

bool plant = false, plant_columns = false;
long requests = 0, outside = 0;

uint32_t along_of(uint32_t length, uint32_t along) { return plant ? along : lcu::stage_offset(length, along); }

// `bytes` at offset + scalar, of an operand of `size` bytes
void request(uint32_t length, uint32_t offset, uint32_t scalar, uint32_t bytes, uint64_t size) {
  ++requests;
  for (uint32_t b = 0; b < bytes; b += 4) {  // dropped dword by dword
    const bool wrapping = offset + b < length - scalar, adding = (uint64_t)offset + b + scalar < length;
    if ((wrapping || adding) && (uint64_t)offset + scalar + b + 4 > size) {
      ++outside;
      return;
    }
  }
}

struct shape {
  int M, K, N, block, splits;  // block 0: fp16
};

// gemm_tile.hpp: tiles of BM x BN, a ring of NS stages, or of NS for lhs and NB for W; step > 1: every so many of the stages
void walk_tile(const shape& s, int BM, int BN, int NS, int NB = 0, int step = 1) {
  if (NB == 0) NB = NS;
  const bool u8 = s.block != 0;
  int shift = 0;
  while (u8 && (64 << shift) < s.block) ++shift;
  const uint32_t K = s.K, blocks = u8 ? K >> (6 + shift) : 0, wbytes = u8 ? 1 : 2;
  const uint64_t a_size = (uint64_t)s.M * K * 2, w_size = (uint64_t)s.N * K * wbytes, s_size = (uint64_t)s.N * blocks * 2;
  const int nt_all = s.K / 64, splits = step > 1 ? step : s.splits;
  // a tile in the middle asks for what one of the first tile asks for, shifted: the first and the last of each direction
  for (int m0 : {0, (s.M - 1) / BM * BM}) {
    for (int n0 : {0, (s.N - 1) / BN * BN}) {
      for (int split : {0, splits / 2, splits - 1}) {
        const int stage0 = step > 1 ? split : (int)((long)split * nt_all / splits);
        const int nt = step > 1 ? nt_all / step : (int)((long)(split + 1) * nt_all / splits) - stage0;
        uint32_t la = (uint32_t)a_size, lw = (uint32_t)w_size, ls = (uint32_t)s_size;
        const auto issue_lhs = [&](int stage) {
          const uint32_t along = along_of(la, (uint32_t)(stage0 + stage * step) * 128u);
          for (int row = 0; row < BM; ++row)
            for (int g = 0; g < 8; ++g) request(la, lcu::row_piece(m0 + row, s.M, K * 2, g), along, 16, a_size);
        };
        const auto issue_w = [&](int stage) {
          const uint32_t along = along_of(lw, (uint32_t)(stage0 + stage * step) * (u8 ? 64u : 128u));
          for (int row = 0; row < BN; ++row) {
            for (int g = 0; g < (u8 ? 4 : 8); ++g) request(lw, lcu::row_piece(n0 + row, s.N, K * wbytes, g), along, 16, w_size);
            if (u8) request(ls, lcu::scale_word((uint32_t)std::min(n0 + row, s.N - 1) * blocks + ((uint32_t)(stage0 + stage * step) >> shift)), 0, 4, s_size);
          }
        };
        const auto issue = [&](int a, int b) {
          if (a == nt) la = 0;
          if (b == nt) lw = ls = 0;
          if (a >= 0) issue_lhs(a);
          issue_w(b);
        };
        for (int st = 0; st < NB; ++st) issue(st - (NB - NS), st);
        for (int t = 0; t < nt - 1; ++t) issue(t + NS, t + NB);
      }
    }
  }
}

// gemm_tile.hpp with the columns of two matrices of N rows in turn: tiles of BM x BN of WAVES wavefronts from column `from` on, each wavefront's requests
// from one matrix
void walk_paired(const shape& s, int BM, int BN, int waves, int NS, int NB, int from) {
  const uint32_t K = s.K;
  const uint64_t a_size = (uint64_t)s.M * K * 2, w_size = (uint64_t)s.N * K * 2;
  const int nt = s.K / 64, columns = 2 * s.N, last = from + (columns - from - 1) / BN * BN, clamp = plant_columns ? columns : s.N;
  for (int m0 : {0, (s.M - 1) / BM * BM}) {
    for (int n0 : {from, last}) {
      uint32_t la = (uint32_t)a_size, lw = (uint32_t)(plant_columns ? 2 * w_size : w_size);
      const auto issue = [&](int a, int b) {
        if (a == nt) la = 0;
        if (b == nt) lw = 0;
        const uint32_t along_a = along_of(la, (uint32_t)a * 128u), along_w = along_of(lw, (uint32_t)b * 128u);
        for (int row = 0; a >= 0 && row < BM; ++row)
          for (int g = 0; g < 8; ++g) request(la, lcu::row_piece(m0 + row, s.M, K * 2, g), along_a, 16, a_size);
        for (int wave = 0; wave < waves; ++wave) {
          for (int j = 0; j < BN / 8 / waves; ++j) {
            for (int i = 0; i < 8; ++i) {
              const int n = n0 + (wave + j * waves) * 8 + i;
              if (lcu::paired_matrix(n) != lcu::paired_matrix(wave * 8)) ++outside;  // not in the wavefront's matrix
              for (int g = 0; g < 8; ++g) request(lw, lcu::row_piece(lcu::paired_row(n), clamp, K * 2, g), along_w, 16, w_size);
            }
          }
        }
      };
      for (int st = 0; st < NB; ++st) issue(st - (NB - NS), st);
      for (int t = 0; t < nt - 1; ++t) issue(t + NS, t + NB);
    }
  }
}

// gemm_tile.hpp over experts: a tile's rows from `first` to the group's end, each the row of lhs that the list names (a wrong one among them,
// which has to come as zeros), one matrix of many
void walk_grouped(const shape& s, int BM, int BN, int NS, int NB) {
  const uint32_t K = s.K;
  const uint64_t a_size = (uint64_t)s.M * K * 2, w_size = (uint64_t)s.N * K * 2;
  const int nt = s.K / 64, listed = 2 * s.M, ends[] = {1, s.M / 2, listed};
  const auto row_of = [&](int r) { return r % 97 == 96 ? s.M + r : (int)((uint64_t)r * 7919 % s.M); };
  for (int end : ends) {
    for (int first : {std::max(0, end - 1), std::max(0, end - BM), std::max(0, end - BM + 3)}) {
      for (int n0 : {0, (s.N - 1) / BN * BN}) {
        uint32_t la = (uint32_t)a_size, lw = (uint32_t)w_size;
        const auto issue = [&](int a, int b) {
          if (a == nt) la = 0;
          if (b == nt) lw = 0;
          const uint32_t along_a = along_of(la, (uint32_t)a * 128u), along_w = along_of(lw, (uint32_t)b * 128u);
          for (int row = 0; a >= 0 && row < BM; ++row) {
            const int from = row_of(std::min(first + row, end - 1));
            for (int g = 0; g < 8; ++g) request(la, lcu::row_piece(from, from + 1, K * 2, g), along_a, 16, a_size);
          }
          for (int row = 0; row < BN; ++row)
            for (int g = 0; g < 8; ++g) request(lw, lcu::row_piece(n0 + row, s.N, K * 2, g), along_w, 16, w_size);
        };
        for (int st = 0; st < NB; ++st) issue(st - (NB - NS), st);
        for (int t = 0; t < nt - 1; ++t) issue(t + NS, t + NB);
      }
    }
  }
}

// gemm_stream.hpp: 16 columns to a wavefront, a ring of 4 units; lhs is read through clamped addresses
void walk_stream(const shape& s) {
  const bool u8 = s.block != 0;
  int shift = 0;
  while (u8 && (64 << shift) < s.block) ++shift;
  const uint32_t K = s.K, blocks = u8 ? K >> (6 + shift) : 0, wbytes = u8 ? 1 : 2;
  const uint64_t w_size = (uint64_t)s.N * K * wbytes, s_size = (uint64_t)s.N * blocks * 2;
  const int nt_all = s.K / 64, per = u8 ? 2 : 1, ring = 4;
  for (int n0 : {0, (s.N - 1) / 16 * 16}) {
    for (int split = 0; split < s.splits; ++split) {
      const int stage0 = (int)((long)split * nt_all / s.splits), stage1 = (int)((long)(split + 1) * nt_all / s.splits);
      const int base = stage0 & ~1, end = stage1 - base, units = (end + per - 1) / per, u0 = (stage0 - base) / per;
      uint32_t lw = (uint32_t)w_size, ls = (uint32_t)s_size;
      for (int u = u0; u < units + ring - 1; ++u) {
        if (u == units) lw = ls = 0;
        const uint32_t along = along_of(lw, (uint32_t)(base * (u8 ? 64 : 128) + u * 128));
        for (int row = 0; row < 16; ++row) {
          for (int piece = 0; piece < 8; ++piece) request(lw, lcu::row_piece(n0 + row, s.N, K * wbytes, piece), along, 16, w_size);
          if (u8) request(ls, lcu::scale_word((uint32_t)std::min(n0 + row, s.N - 1) * blocks + ((uint32_t)(base + 2 * u) >> shift)), 0, 4, s_size);
        }
      }
    }
  }
}

}  // namespace

int main(int argc, char** argv) {
  plant = argc > 1 && !strcmp(argv[1], "offset");
  plant_columns = argc > 1 && !strcmp(argv[1], "columns");
  // K of one to many stages, shorter than the ring too; rows and columns past the last whole tile; one and several scales per
  // row, the number of all of them even; operands just below 4 GiB
  const shape tiles[] = {{300, 64, 1030, 0, 1},   {65, 128, 20500, 0, 1},    {2049, 192, 4100, 0, 1},  {100, 5120, 1030, 0, 3},
                         {512, 11008, 4096, 0, 4}, {257, 128, 6790, 64, 1},   {300, 5120, 1030, 128, 2}, {1100, 384, 3690, 128, 1},
                         {127, 256, 35000, 256, 1}, {70, 32768, 65535, 0, 1}, {70, 32768, 131070, 32768, 1}, {524287, 4096, 130, 128, 1}};
  for (const shape& s : tiles) {
    walk_tile(s, 256, 256, s.block ? 3 : 2);
    walk_tile(s, 256, 192, 2);
    walk_tile(s, 256, 128, 3);
    walk_tile(s, 128, 256, 3);
    walk_tile(s, 128, 128, 4);
    walk_tile(s, 256, 192, s.block ? 3 : 2, s.block ? 3 : 4);
    walk_tile(s, 256, 256, 2, 3);
    if (s.K % 128 == 0) walk_tile(s, 128, 128, 4, 4, 2);
  }
  // hidden columns a multiple of 16 and of no tile's width; all tiles, and those of a second launch over the columns that whole rounds leave
  const shape pairs[] = {{65, 128, 10256, 0, 1}, {300, 384, 5136, 0, 1}, {1033, 2048, 6704, 0, 1}, {100, 64, 16400, 0, 1}, {129, 16384, 65520, 0, 1}};
  for (const shape& s : pairs) {
    for (int share : {0, 2}) {
      const auto from = [&](int columns) { return share == 0 ? 0 : 2 * s.N / columns * (share - 1) / share * columns; };
      walk_paired(s, 128, 256, 8, 3, 3, from(256));
      walk_paired(s, 128, 128, 4, 4, 4, from(192));
      walk_paired(s, 256, 256, 4, 2, 3, from(256));
      walk_paired(s, 256, 192, 4, 2, 4, from(192));
      walk_paired(s, 256, 128, 8, 3, 3, from(128));
    }
  }
  const shape experts[] = {{512, 4096, 5632, 0, 1}, {700, 576, 1000, 0, 1}, {130, 64, 200, 0, 1}, {50, 1024, 128, 0, 1}, {300, 448, 130, 0, 1}};
  for (const shape& s : experts) {
    walk_grouped(s, 128, 128, 4, 4);
    walk_grouped(s, 256, 128, 3, 3);
  }
  const shape rows[] = {{3, 1152, 520, 0, 4},     {16, 1408, 4099, 0, 5},  {48, 5888, 4100, 0, 2},  {7, 64, 40, 0, 1},
                        {2, 1152, 520, 64, 4},    {17, 2560, 1000, 256, 7}, {64, 5888, 4101, 128, 3}, {7, 17920, 6656, 128, 5},
                        {33, 320, 5000, 0, 2},    {5, 128, 18, 64, 1},      {2, 32768, 65535, 0, 8},  {2, 32768, 131070, 32768, 8}};
  for (const shape& s : rows) walk_stream(s);
  printf("%ld requests, %ld reach past their operand\n", requests, outside);
  return outside != 0;
}
