// Which bytes of an operand the buffer requests of the product kernels ask for (gemm_tile.hpp, gemm_stream.hpp): a
// resource of the operand's own length, an offset per lane and a scalar offset along K.  Plain arithmetic, apart from
// the kernels, so that every request of a shape can be checked on the host.
#pragma once
#include <stdint.h>

namespace lcu {

// 16-byte piece `piece` of row `row`; rows past the last one are the last one, whose sums are not stored again
constexpr uint32_t row_piece(int row, int rows, uint32_t row_bytes, int piece) {
  return (uint32_t)(row < rows ? row : rows - 1) * row_bytes + (uint32_t)piece * 16u;
}

// Columns that alternate between two matrices, sixteen of each: which of them column n is of, and its row there
constexpr int paired_matrix(int n) { return n / 16 % 2; }
constexpr int paired_row(int n) { return n / 32 * 16 + n % 16; }

// scalar offset of a request for the stage that begins `along` bytes into a row.  Behind the last stage the resource's
// length is 0, and the offset is 0 with it: such a request counts as any other and lies outside the length whichever
// way a range check sets the scalar offset off against it.
constexpr uint32_t stage_offset(uint32_t length, uint32_t along) { return length == 0 ? 0 : along; }

// the aligned word that holds scale `at` of an array with an even number of fp16 scales
constexpr uint32_t scale_word(uint32_t at) { return (at & ~1u) * 2u; }

}  // namespace lcu
