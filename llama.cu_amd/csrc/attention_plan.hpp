// Which kernel a prompt's attention takes (attention.hip).  Plain arithmetic, apart from the kernels, so that it can be checked on the host.
#pragma once
#include <cstddef>

namespace lcu {

constexpr int HD = 128;        // head width
constexpr int BR = 16;         // query rows per workgroup of the kernel that stores its scores
constexpr int CW = 64;         // cache rows per staged chunk
constexpr int QLD = HD + 8;    // LDS row stride (halves) of K chunks
constexpr int VLD = HD + 16;   // and of V chunks

inline size_t prefill_lds_bytes(int T) {
  const int Tc = (T + CW - 1) / CW * CW;
  return ((size_t)CW * VLD + (size_t)BR * (Tc + 8)) * 2;
}

// Whether computing the scores three times and storing none (prompt_attention_kernel) is done sooner than keeping a strip of them in LDS
// (prefill_attention_kernel).  A wavefront of the former walks all T columns alone, 4.1 us per 64 of them; the latter shares a tile's columns
// among four wavefronts but does 0.23 M scores per us, and 0.15 M where LDS holds one strip only; the lines cross where the call has 17 000 and
// 9000 scores per column
// (heads, n = T, us again / kept: 32 heads 512 rows 35 / 18, 800 rows 55 / 40, 1024 rows 70 / 69, 1200 rows 83 / 97, 1987 rows 167 / 433;
// 52 heads 600 rows 45 / 41, 700 rows 51 / 50, 900 rows 71 / 78; 16 heads 1500 rows 97 / 78, 2000 rows 129 / 223; 4 heads 2000 rows 117 / 62;
// 32 heads 512 rows of 1500 97 / 85, of 2048 129 / 202, 128 rows of 2000 120 / 58).
// Where a compute unit's LDS holds two strips, 11 000 to 17 000 are a matter of the last round of workgroups: in full it takes as long as the
// others for the columns in front of the prompt, which every tile sees, while those of the prompt itself balance (tiles of later rows, which see
// more of them, go first).  Of 1370 drawn calls 50 take more than 3 % longer than the other kernel so, 303 with the line at 17 000 and 442 at
// 13 000 (40 heads 452 rows of 1712 104 / 128; 52 heads 306 rows of 1531 94 / 123; 24 heads 1019 rows of 1094 70 / 55).
// Both take 6 to 18 % less since then (32 heads 1024 rows 63 -> 52, 800 rows 35.5 -> 32); the lines stand where they were.
inline bool scores_again(int n_heads, int n_new, int start_pos, long cus) {
  const int T = start_pos + n_new;
  const double scores = (double)n_heads * n_new * (start_pos + 0.5 * n_new);
  const size_t strips = (size_t)160 * 1024 / (prefill_lds_bytes(T) + BR * QLD * 2);  // the lines were measured with a tile of queries in LDS too
  if (strips != 2 || scores >= 17000.0 * T || scores < 11000.0 * T) return scores >= (strips >= 2 ? 17000.0 : 9000.0) * T;
  const long tiles = (long)((n_new + BR - 1) / BR) * n_heads, rounds = (tiles + 2 * cus - 1) / (2 * cus);
  const double kept = 0.0283 * (0.5 * n_new * tiles / (2 * cus) + (double)start_pos * rounds) + 1.4 * rounds + 2.7, again = 0.056 * T + 7.3;  // us
  return again < kept;
}

}  // namespace lcu
