// Large tiles of a matrix product with many rows: out[M,N] = lhs[M,K] * W[N,K]^T, fp16 or bfloat16 operands, sums
// in fp32 over ascending k.
//
// What bounds it: the chip's power, and behind it the way from L2 into LDS.  On random operands the matrix
// cores alone, fed from registers, reach 1.6 to 1.9 PFLOP/s (4096^3: 71 to 84 us by the loop; 60 to 70 us on zeros); with the operands on
// their way through LDS this kernel takes 106 us there (1.30 PFLOP/s; 81 us on zeros).  So the design saves
// what costs energy or makes a wavefront wait:
//  * v_mfma_f32_16x16x32 instead of 32x32x16: half the accumulator traffic per multiply-add (4096^3 with 256x128
//    tiles 133 -> 119 us).  Both take their products eight at a time in ascending k, so the bits are the same.
//  * neighbouring instructions share an operand, also where the row of tiles changes (boustrophedon order).
//  * a half stage (32 of K) of fragments is read from LDS while the half before it is multiplied, one read
//    between two matrix instructions; requests for the stages ahead go out the same way.
//  * requests are buffer loads straight into LDS whose stage offset is a scalar.  Behind the last stage the
//    resource holds no records and the offset is 0 (operand_range.hpp): the request counts as any other but touches
//    no memory, so that the loop has one form up to the end and its registers are never copied.
//  * outputs go through LDS and leave in 16-byte pieces, wherever a row begins.
// LDS stage: rows of 128 bytes, lhs tile then W tile, 16-byte chunk g of row r at position g ^ (r / 2) % 8, so that
// neither requests (1 KB per instruction, dense) nor fragment reads (16 rows, one chunk) meet in a bank (counted: 512x4096x12288 98 304
// conflict cycles of 6.7 M; they grow with the outputs, not with K).
#pragma once
#include <type_traits>
#include <utility>

#include "linear.hpp"
#include "operand_range.hpp"

namespace lcu {

// Up to three products lhs * W_g^T with weight matrices of one shape in a single launch (Wq, Wk,
// Wv; W1, W3): the tile index along N runs through matrix 0, then 1, then 2, `tiles_n_per` tiles
// each.  Matrix 0 travels in the kernel's ordinary arguments, the others here.
struct more_matrices_t {
  half_t* out[2];
  const void* W[2];
  const half_t* S[2];
  int tiles_n_per;  // tiles along N of one matrix; 0: a single matrix
};

struct f16_epilogue {
  static constexpr bool BF16 = false, GROUPED = false, GATED = false, ROTARY = false, PAIRED = false;
};
// fp16 outputs whose first `matrices` matrices are rotated (llama_cu.cu:368-389): row r is at position first + r, head_dim a multiple of 8.
// The rotation reads outputs as they would be stored, so the bits are those of lcu_rope_pair afterwards.  512 rows, three times 4096x4096: the
// product 63.6 us and the rotation by itself 7.4 -> 65.7; 1987 rows 183 and 20.7 -> 186.
struct rotary_epilogue {
  static constexpr bool BF16 = false, GROUPED = false, GATED = false, ROTARY = true, PAIRED = false;
  const float2* table;  // [positions][head_dim / 2] (cos, sin)
  int head_dim, first, matrices;
};

// fp16(silu(lhs W^T) * (lhs V^T)), llama_cu.cu:1180-1183: the columns alternate, sixteen of W (matrix 0) and the sixteen of V (matrix 1) that
// they meet, so that a lane holds both; N counts both.  A wavefront requests columns of one matrix only.  Half the outputs and no launch that
// reads them again: 512 rows, K 4096, twice 11008 columns 97.9 us in two launches, 90.2 here (95 with the general exponential and division: 96
// outputs to a lane are 4 us of the tile), 1987 rows 329 and 318; K 2048, twice 5632 columns 38.3 and 33.3, 112 and 101.
struct silu_epilogue {
  static constexpr bool BF16 = false, GROUPED = false, GATED = false, ROTARY = false, PAIRED = true;
};

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// the buffer resource of an operand of `bytes` (below 4 GiB)
__device__ __forceinline__ uint4_t operand_resource(const void* p, uint32_t bytes) {
  const uintptr_t a = (uintptr_t)p;
  uint4_t r;
  r[0] = __builtin_amdgcn_readfirstlane((uint32_t)a);
  r[1] = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32) & 0xffffu);
  r[2] = __builtin_amdgcn_readfirstlane(bytes);
  r[3] = 0x00020000u;
  return r;
}

// f of 0 .. N - 1 as constants: loops whose bodies are too long for the compiler to unroll when asked
template <class F, int... I>
__device__ __forceinline__ void static_for_each(F& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_each(f, std::make_integer_sequence<int, N>{});
}

// two codes, spread to the low bytes of two halves, to fp16((q - 127.5) * scale) each (llama_cu.cu:287-289)
__device__ __forceinline__ half2_t dequant2(uint32_t spread, half2_t scale2x) {
  const uint32_t bits = (spread << 2) | 0x58005800u;                                  // 128 + q/2
  const half2_t t = __builtin_bit_cast(half2_t, bits) - (half2_t)((half_t)191.75f);   // (q - 127.5)/2
  return t * scale2x;                                                                 // one rounding
}

// WM x WN wavefronts of (BM / WM) x (BN / WN) outputs each, rings of NA stages of 64 along K of lhs and NB of W.  The lhs comes from L2, W
// from memory: where LDS does not hold three stages of both, W's ring takes what two of lhs leave (fp16, 512 rows of K 4096, a round of 192
// columns 82 -> 67 us with rings of two and two -> two and four, of 256 columns 93 -> 84; 1987 rows, twice 11008 columns 304 -> 293.  From
// three stages on longer rings of W measured equal or slower, in uint8 too.)
// U8: W is codes with one fp16 scale per `block` of a row, block = 64 << block_shift.  Codes lie in LDS as they are, 64
// bytes a row with the 16-byte pieces of every second group of four rows turned by two (a sixth of LDS's cycles still go to conflicts of
// their 8-byte reads, a ninth with 256 columns: counted on 512x6656x35840 and 512x6656x19968); a wavefront turns
// the eight codes of each of its fragments into fp16 itself, four instructions at a time between the matrix instructions of the half
// stage before.  The wavefronts stand side by side (WM = 1), so that every code
// is converted once; with the lhs read from LDS by all four that leaves vector instructions, LDS and matrix cores about
// equally busy.  512 rows, (N, K) = (11008, 4096): 64 us; two rows of two wavefronts (every code twice) 64-66, four of two
// 88; converted once into an fp16 tile in LDS, with its own ring, 87 us.  1987 rows, twice (11008, 4096): 346 / 432 / 492 / 475 us.
template <int BM, int BN, int WM, int WN, int NA, int NB, bool U8, bool SPLIT, class EP>
struct tile_shape {
  static constexpr int NW = WM * WN, WR = BM / WM, WC = BN / WN;
  static constexpr int A_BYTES = BM * 128, B_BYTES = BN * (U8 ? 64 : 128), SW = (WC + 63) / 64 * 64, S_BYTES = U8 ? NW * SW * 4 : 0;
  static constexpr int W_BYTES = B_BYTES + S_BYTES;      // S: one word per column of every wavefront, of its own
  static constexpr int OUT_LD = (EP::GATED || EP::PAIRED ? WC / 2 : WC) + 4;  // floats per row of a wavefront's 64 output rows in LDS
  static constexpr int RING = NA * A_BYTES + NB * W_BYTES, OUT = NW * 64 * OUT_LD * 4;
  static constexpr int LDS = RING > OUT ? RING : OUT;
  static_assert(LDS <= 160 * 1024 && WR % 64 == 0 && WC % 16 == 0, "tile");
};

// CHAINS 2: the even and the odd stages of K are summed apart, and the two sums added (K a multiple of 128).
template <int BM, int BN, int WM, int WN, int NA, int NB, bool U8, bool SPLIT, class EP, int CHAINS = 1>
__global__ __launch_bounds__(64 * WM * WN, (WM * WN + 3) / 4) void gemm_tile_kernel(
    half_t* __restrict__ out0, const half_t* __restrict__ A, const void* __restrict__ W0, const half_t* __restrict__ S0, int block_shift,
    int M, int K, int N, float beta, int tiles_m, int tiles_n, int from, float* __restrict__ part, int splits, int step, more_matrices_t more, EP ep) {
  using shape = tile_shape<BM, BN, WM, WN, NA, NB, U8, SPLIT, EP>;
  static_assert(!EP::GROUPED || (!SPLIT && EP::BF16), "experts");
  constexpr int NW = shape::NW;
  constexpr int TM = shape::WR / 16, TN = shape::WC / 16;        // 16x16 tiles of a wavefront
  constexpr int A_BYTES = shape::A_BYTES, B_BYTES = shape::B_BYTES, W_BYTES = shape::W_BYTES;
  // rings of one length: a stage's lhs and columns side by side, one slot for both (uint8 with two slots 5 to 7 % slower, 736x4096x4096 40 / 43 us)
  constexpr bool JOINT = NA == NB;
  constexpr int A_STEP = JOINT ? A_BYTES + W_BYTES : A_BYTES, W_STEP = JOINT ? A_STEP : W_BYTES, W_RING = JOINT ? A_BYTES : NA * A_BYTES;
  constexpr int PA = A_BYTES / 1024 / NW, PB = B_BYTES / 1024 / NW, PS = U8 ? shape::SW / 64 : 0;
  constexpr int PW = PB + PS, P = PA + PW;  // requests of a wavefront per stage
  constexpr int BEHIND = NB > NA ? PW : 0;  // of a stage's requests, those behind its lhs that lhs's turn need not wait for
  static_assert(A_BYTES % (1024 * NW) == 0 && B_BYTES % (1024 * NW) == 0 && NA >= 2 && NB >= NA && PA * NA + PW * NB < 64, "requests");
  static_assert(!U8 || !EP::BF16, "codes");
  static_assert(!EP::PAIRED || (!U8 && !SPLIT && NW % 4 == 0 && TN % 2 == 0), "pairs of columns");
  extern __shared__ __attribute__((aligned(16))) unsigned char tile_lds[];

  // consecutive workgroups go round the eight XCDs: each gets one run of the M-fastest tile sequence, so that
  // tiles that share a slice of W share an L2
  const int nb = tiles_m * tiles_n;
  const int split = SPLIT ? blockIdx.x / nb : 0;
  const int bx = SPLIT ? blockIdx.x - split * nb : blockIdx.x;
  const int q = nb / 8, r = nb % 8, xcd = bx % 8;
  const int logical = xcd * q + min(xcd, r) + bx / 8;
  int tm = logical % tiles_m;
  int tn = logical / tiles_m;
  half_t* out = out0;
  const void* W = W0;
  const half_t* S = S0;
  int g = 0;
  if (more.tiles_n_per > 0) {
    g = tn / more.tiles_n_per;
    tn -= g * more.tiles_n_per;
    out = g == 0 ? out0 : (g == 1 ? more.out[0] : more.out[1]);
    W = g == 0 ? W0 : (g == 1 ? more.W[0] : more.W[1]);
    if constexpr (U8) S = g == 0 ? S0 : (g == 1 ? more.S[0] : more.S[1]);
    if constexpr (SPLIT) part += (size_t)g * splits * M * N;  // each matrix has its own partial sums
  }
  int m0 = tm * BM;
  if constexpr (EP::GROUPED) {
    const group_tile_t at = group_tile(ep, tiles_n, bx);
    if (at.group < 0) return;
    m0 = ep.tile_row[at.row_tile];
    M = ep.group_end[at.group];
    tn = at.column_tile;
    W = (const char*)W0 + (size_t)at.group * ep.group_stride;
  }
  const int n0 = from + tn * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = (wave % WM) * shape::WR, wn = (wave / WM) * shape::WC;
  // request j of a wavefront is rows (wave + j NW) 8 .. + 7 of the tile: of the same matrix for every j
  if constexpr (EP::PAIRED) W = paired_matrix(wave * 8) == 1 ? more.W[0] : W0;
  const int matrix_n = EP::PAIRED ? N / 2 : N;

  // this workgroup's K stages
  const int nt_all = K / 64;
  int stage0 = 0, nt = nt_all;
  if constexpr (SPLIT) {  // a run of them, or with step = splits every so many
    stage0 = step > 1 ? split : (int)((long)split * nt_all / splits);
    nt = step > 1 ? nt_all / step : (int)((long)(split + 1) * nt_all / splits) - stage0;
  }
  const auto stage_of = [&](int t) { return (uint32_t)(SPLIT ? stage0 + t * step : t); };

  // request j of this wavefront fills LDS bytes [(wave + j * NW) * 1024, + 1024) of an operand's part of a stage.
  // Rows past M or N are clamped to the last one: their sums are never stored.
  uint32_t a_off[PA], b_off[PB];
#pragma unroll
  for (int j = 0; j < PA; ++j) {
    const int c = (wave + j * NW) * 64 + lane, row = c / 8, g = (c % 8) ^ ((row / 2) % 8);
    if constexpr (EP::GROUPED) {
      const int r = min(m0 + row, M - 1), from_row = ep.row_index ? ep.row_index[r] : r;
      a_off[j] = row_piece(from_row, from_row + 1, (uint32_t)K * 2u, g);
    } else {
      a_off[j] = row_piece(m0 + row, M, (uint32_t)K * 2u, g);
    }
  }
#pragma unroll
  for (int j = 0; j < PB; ++j) {
    const int c = (wave + j * NW) * 64 + lane;
    if constexpr (U8) {
      const int row = c / 4, g = (c % 4) ^ (2 * ((row / 4) % 2));
      b_off[j] = row_piece(n0 + row, N, (uint32_t)K, g);
    } else {
      const int row = c / 8, g = (c % 8) ^ ((row / 2) % 8), n = n0 + row;
      b_off[j] = row_piece(EP::PAIRED ? paired_row(n) : n, matrix_n, (uint32_t)K * 2u, g);
    }
  }
  // first scale of the rows whose scales this lane requests, and of those of its fragments
  uint32_t s_first[U8 ? PS : 1], f_first[U8 ? TN : 1];
  if constexpr (U8) {
    const uint32_t blocks = (uint32_t)K >> (6 + block_shift);
#pragma unroll
    for (int j = 0; j < PS; ++j) s_first[j] = (uint32_t)min(n0 + wn + j * 64 + lane, N - 1) * blocks;
#pragma unroll
    for (int j = 0; j < TN; ++j) f_first[j] = (uint32_t)min(n0 + wn + j * 16 + (lane & 15), N - 1) * blocks;
  }
  int lhs_rows = M;
  if constexpr (EP::GROUPED) lhs_rows = ep.lhs_rows;
  uint4_t ra = operand_resource(A, (uint32_t)lhs_rows * (uint32_t)K * 2u), rw = operand_resource(W, (uint32_t)matrix_n * (uint32_t)K * (U8 ? 1u : 2u)), rs = ra;
  if constexpr (U8) rs = operand_resource(S, (uint32_t)N * ((uint32_t)K >> (6 + block_shift)) * 2u);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)tile_lds;
  // Inline assembly, so that the compiler does not know about the LDS writes: knowing, it waits for every LDS read
  // in front of each matrix instruction.  There is no output register; the waits are the explicit ones below.
  const auto request = [&](uint4_t resource, uint32_t stage_bytes, uint32_t offset, uint32_t at) {
    asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(offset), "s"(resource), "s"(stage_bytes),
                 "s"(lds0 + at)
                 : "memory", "m0");
  };
  // marked as read once: the columns of experts that come from memory (read_once).  Other products' columns stay in the caches: 7B prompts gain 0.5 %, a product
  // called again loses a third.
  const auto request_once = [&](uint4_t resource, uint32_t stage_bytes, uint32_t offset, uint32_t at) {
    asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen nt lds" ::"v"(offset), "s"(resource), "s"(stage_bytes),
                 "s"(lds0 + at)
                 : "memory", "m0");
  };
  // request i of a wavefront's P: lhs of stage `a` into its ring's slot, then the columns (and scales) of stage `b` into theirs
  const auto issue = [&](int a, int a_slot, int b, int b_slot, int i) {
    if (i < PA) {
      request(ra, stage_offset(ra[2], stage_of(a) * 128u), a_off[i], a_slot * A_STEP + (wave + i * NW) * 1024);
    } else if (i < PA + PB) {
      const uint32_t along = stage_offset(rw[2], stage_of(b) * (U8 ? 64u : 128u)), at = W_RING + b_slot * W_STEP + (wave + (i - PA) * NW) * 1024;
      constexpr bool ONCE = [] {
        if constexpr (EP::GROUPED) return EP::ONCE;
        return false;
      }();
      if constexpr (ONCE) {
        request_once(rw, along, b_off[i - PA], at);
      } else {
        request(rw, along, b_off[i - PA], at);
      }
    } else if constexpr (U8) {  // the word that holds the row's scale of this stage
      const uint32_t at = s_first[i - PA - PB] + (stage_of(b) >> block_shift);
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dword %0, %1, 0 offen lds" ::"v"(scale_word(at)), "s"(rs),
                   "s"(lds0 + W_RING + b_slot * W_STEP + B_BYTES + wave * shape::SW * 4 + (i - PA - PB) * 256)
                   : "memory", "m0");
    }
  };

  float4_t acc[TM][TN], odd[CHAINS == 2 ? TM : 1][CHAINS == 2 ? TN : 1];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      acc[i][j] = (float4_t)(0.0f);
      if constexpr (CHAINS == 2) odd[i][j] = (float4_t)(0.0f);
    }
  }
  const int frag_row = lane & 15, frag_chunk = lane >> 4, turn = (frag_row / 2) % 8;
  uint32_t pos[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) pos[h] = (uint32_t)(((frag_chunk + 4 * h) ^ turn) * 16);
  const uint32_t a_row = (uint32_t)(wm + frag_row) * 128, b_row = (uint32_t)W_RING + (uint32_t)(wn + frag_row) * 128;
  half8_t fa[2][TM], fb[2][TN];
  // U8: the eight codes behind a fragment, and twice their scale
  uint2_t codes[2][U8 ? TN : 1];
  uint32_t words[U8 ? TN : 1];
  half2_t scales[U8 ? TN : 1];
  // reads of half 0: (scales, codes,) W and lhs fragments of half 0(, codes of half 1); of half 1 the fragments that are left
  constexpr int READS0 = U8 ? 3 * TN + TM : TN + TM, READS1 = U8 ? TM : TN + TM, PRODUCTS = TM * TN;
  const auto read = [&](int a_slot, int b_slot, int h, int i) {
    const unsigned char *pa = tile_lds + a_slot * A_STEP + a_row, *pw = tile_lds + b_slot * W_STEP;
    if constexpr (U8) {
      const unsigned char* c = pw + W_RING + (wn + frag_row) * 64 + frag_chunk * 8;
      const int half_turn = (frag_row / 4) % 2 * 32;  // pieces turned by two: the halves change places
      if (h == 1) {
        fa[1][i] = *reinterpret_cast<const half8_t*>(pa + pos[1] + i * 2048);
      } else if (i < TN) {
        words[i] = *reinterpret_cast<const uint32_t*>(pw + W_RING + B_BYTES + wave * shape::SW * 4 + (i * 16 + frag_row) * 4);
      } else if (i < 2 * TN) {
        codes[0][i - TN] = *reinterpret_cast<const uint2_t*>(c + (i - TN) * 1024 + half_turn);
      } else if (i < 2 * TN + TM) {
        fa[0][i - 2 * TN] = *reinterpret_cast<const half8_t*>(pa + pos[0] + (i - 2 * TN) * 2048);
      } else {
        codes[1][i - 2 * TN - TM] = *reinterpret_cast<const uint2_t*>(c + (i - 2 * TN - TM) * 1024 + (32 - half_turn));
      }
    } else if (i < TN) {
      fb[h][i] = *reinterpret_cast<const half8_t*>(pw + pos[h] + b_row + i * 2048);
    } else {
      fa[h][i - TN] = *reinterpret_cast<const half8_t*>(pa + pos[h] + (i - TN) * 2048);
    }
  };
  // two of the eight values of a fragment of half h from their codes, which belong to stage `st`; four instructions, as
  // many as go out while a matrix instruction runs
  constexpr int CONVERTS = U8 ? 4 * TN : 0;
  const auto convert = [&](int h, int k, int st) {
    if constexpr (U8) {
      const int j = k / 4, w = k / 2 % 2, high = k % 2;
      if (h == 0 && k % 4 == 0) {
        const uint32_t at = f_first[j] + (stage_of(st) >> block_shift);
        const half_t x = __builtin_bit_cast(half_t, (uint16_t)((at & 1) ? words[j] >> 16 : words[j])) * (half_t)2.0f;
        scales[j] = half2_t{x, x};
      }
      const half2_t y = dequant2(__builtin_amdgcn_perm(0u, codes[h][j][w], high ? 0x0c030c02u : 0x0c010c00u), scales[j]);
      fb[h][j][4 * w + 2 * high] = y.x;
      fb[h][j][4 * w + 2 * high + 1] = y.y;
    }
  };
  const auto multiply = [&](int h, int i, auto chain) {
    const int a = i / TN, b = (a & 1) ? TN - 1 - i % TN : i % TN;
    const auto add_to = [&](float4_t& sum) {
      if constexpr (EP::BF16) {
        sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, fa[h][a]), __builtin_bit_cast(bf16x8_t, fb[h][b]), sum, 0, 0, 0);
      } else {
        sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[h][a], fb[h][b], sum, 0, 0, 0);
      }
    };
    if constexpr (decltype(chain)::value == 1) {
      add_to(odd[a][b]);
    } else {
      add_to(acc[a][b]);
    }
  };
  // the products of half h, with the reads spread over the first five eighths, the requests over all of them, and the
  // conversions of the next half (U8) over the last half (of half 1, whose codes are read first) or all (of half 0)
  const auto half_stage = [&](int h, auto n_reads, auto&& do_read, auto n_requests, auto&& do_request, auto n_converts, int convert_stage, auto chain) {
    constexpr int NR = decltype(n_reads)::value, NQ = decltype(n_requests)::value, SPREAD = PRODUCTS * 5 / 8;
    constexpr int NC = decltype(n_converts)::value;
    static_for<PRODUCTS>([&](auto at) {
      constexpr int i = decltype(at)::value;
      multiply(h, i, chain);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (i < SPREAD) {
#pragma unroll
        for (int k = i * NR / SPREAD; k < (i + 1) * NR / SPREAD; ++k) do_read(k);
      }
#pragma unroll
      for (int k = i * NQ / PRODUCTS; k < (i + 1) * NQ / PRODUCTS; ++k) do_request(k);
      const int from = h == 1 ? PRODUCTS / 2 : 0;
      if (NC > 0 && i >= from) {
#pragma unroll
        for (int k = (i - from) * NC / (PRODUCTS - from); k < (i - from + 1) * NC / (PRODUCTS - from); ++k) convert(1 - h, k, convert_stage);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  // One stage: multiply its first half while the second is read; this wavefront has then read the whole stage, and once its own
  // requests of the next stage have landed the barrier says both for everybody.  Then the second half, with the next stage's first half
  // on its way and the stages NA and NB ahead requested into this one's slots.  Of a stage's requests the lhs goes first: when that of
  // stage t + 1 has to be there, the columns asked for behind it and all of the NA - 2 stages since may still be out.
  const auto stage = [&](int t, int a_slot, int b_slot, int a_next, int b_next, auto more_follow, auto chain) {
    constexpr bool MORE = decltype(more_follow)::value;
    half_stage(0, std::integral_constant<int, READS1>{}, [&](int k) { read(a_slot, b_slot, 1, k); }, std::integral_constant<int, 0>{}, [](int) {},
               std::integral_constant<int, CONVERTS>{}, t, chain);
    if constexpr (MORE) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      wait_vmcnt<(NA - 2) * P + BEHIND>();
      asm volatile("s_barrier" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      half_stage(1, std::integral_constant<int, READS0>{}, [&](int k) { read(a_next, b_next, 0, k); }, std::integral_constant<int, P>{},
                 [&](int k) { issue(t + NA, a_slot, t + NB, b_slot, k); }, std::integral_constant<int, CONVERTS>{}, t + 1, chain);
    } else {
      half_stage(1, std::integral_constant<int, 0>{}, [](int) {}, std::integral_constant<int, 0>{}, [](int) {},
                 std::integral_constant<int, 0>{}, 0, chain);
    }
  };

  // no records behind the last stage: a request brings zeros and reads nothing (stage_offset)
  const auto end_at = [&](int a, int b) {
    if (a == nt) ra[2] = 0;
    if (b == nt) rw[2] = rs[2] = 0;
  };
#pragma unroll
  for (int s = 0; s < NB; ++s) {  // what the stages before stage 0 would have asked for
    end_at(s - (NB - NA), s);
#pragma unroll
    for (int i = s < NB - NA ? PA : 0; i < P; ++i) issue(s - (NB - NA), max(s - (NB - NA), 0), s, s, i);
  }
  wait_vmcnt<(NA - 1) * P + BEHIND>();
  __syncthreads();
#pragma unroll
  for (int i = 0; i < READS0; ++i) read(0, 0, 0, i);
#pragma unroll
  for (int k = 0; k < CONVERTS; ++k) convert(0, k, 0);
  __builtin_amdgcn_sched_barrier(0);
  int a_slot = 0, b_slot = 0;
  constexpr std::integral_constant<int, 0> even_chain{};
  constexpr std::integral_constant<int, CHAINS - 1> odd_chain{};
  const auto step_on = [&](int t, auto chain) {
    end_at(t + NA, t + NB);
    const int a_next = a_slot + 1 == NA ? 0 : a_slot + 1, b_next = JOINT ? a_next : b_slot + 1 == NB ? 0 : b_slot + 1;
    stage(t, a_slot, b_slot, a_next, b_next, std::true_type{}, chain);
    a_slot = a_next;
    b_slot = b_next;
  };
  if constexpr (CHAINS == 2) {
    for (int t = 0; t < nt - 2; t += 2) {
      step_on(t, even_chain);
      step_on(t + 1, odd_chain);
    }
    step_on(nt - 2, even_chain);
  } else {
    for (int t = 0; t < nt - 1; ++t) step_on(t, even_chain);
  }
  stage(nt - 1, a_slot, b_slot, 0, 0, std::false_type{}, odd_chain);
  if constexpr (CHAINS == 2) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] += odd[i][j];
    }
  }
  wait_vmcnt<0>();  // the requests behind the last stage have written their zeros
  __syncthreads();  // LDS is free

  // ---- epilogue, 64 rows of the wavefront's tile at a time.  Register v of lane l holds row 4 (l / 16) + v, column
  // l % 16 of a 16x16 tile.
  float* rows = reinterpret_cast<float*>(tile_lds) + wave * 64 * shape::OUT_LD;
  constexpr bool HALVED = EP::GATED || EP::PAIRED;           // two columns to an output
  constexpr int OC = HALVED ? shape::WC / 2 : shape::WC;     // output columns of the wavefront
  constexpr int PIECES = OC / 8;                             // pieces of eight columns per row, and per lane
  const int out_n0 = HALVED ? (n0 + wn) / 2 : n0 + wn, out_n = HALVED ? N / 2 : N;
  // Pieces of eight columns leave as 16 bytes wherever a row begins, its last ones one by one (fp16 1401x384x16515: 39 us so,
  // 75 with single stores for rows off 16 bytes).
  typedef half8_t any_half8_t __attribute__((aligned(2)));
  typedef float4_t any_float4_t __attribute__((aligned(4)));
  const auto pass = [&](auto which) {
    constexpr int p = decltype(which)::value;
    float scale[4][4];  // of the rows of gated experts
    if constexpr (EP::GROUPED && EP::GATED) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int gm = m0 + wm + p * 64 + i / 4 * 16 + (lane >> 4) * 4 + i % 4;
        scale[i / 4][i % 4] = ep.row_scale ? ep.row_scale[min(gm, M - 1)] : 1.0f;
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float* to = rows + (i * 16 + (lane >> 4) * 4 + v) * shape::OUT_LD + (lane & 15);
        if constexpr (EP::GATED) {
          // 64 columns are 32 gate rows of the matrix, then the 32 up rows that they belong to
          static_assert(TN % 4 == 0, "whole gate / up pairs");
#pragma unroll
          for (int j = 0; j < TN; j += 4) {
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              float gate = acc[p * 4 + i][j + e][v], up = acc[p * 4 + i][j + 2 + e][v];
              if constexpr (EP::GROUPED) gate *= scale[i][v], up *= scale[i][v];
              to[(j / 2 + e) * 16] = ep.gate(gate, up);
            }
          }
        } else if constexpr (EP::PAIRED) {  // both rounded as they would be stored
#pragma unroll
          for (int j = 0; j < TN; j += 2) to[j / 2 * 16] = (float)silu_mul(round_f16(acc[p * 4 + i][j][v]), round_f16(acc[p * 4 + i][j + 1][v]));
        } else {
#pragma unroll
          for (int j = 0; j < TN; ++j) to[j * 16] = acc[p * 4 + i][j][v];
        }
      }
    }
    constexpr int AT_ONCE = PIECES % 4 == 0 ? 4 : 2;
    static_assert(PIECES % AT_ONCE == 0, "pieces");
#pragma unroll 1
    for (int k0 = 0; k0 < PIECES; k0 += AT_ONCE) {
      half8_t old[AT_ONCE];
      if constexpr (!EP::BF16 && !SPLIT) {
        if (beta != 0.0f) {
#pragma unroll
          for (int k = 0; k < AT_ONCE; ++k) {
            const int c = lane + 64 * (k0 + k), gm = m0 + wm + p * 64 + c / PIECES, gn = out_n0 + c % PIECES * 8;
            if (gm < M && gn + 8 <= out_n) old[k] = *reinterpret_cast<const any_half8_t*>(out + (size_t)gm * out_n + gn);
          }
        }
      }
      float4_t turn[EP::ROTARY ? AT_ONCE : 1][2];  // (cos, sin) of a piece's four pairs
      if constexpr (EP::ROTARY) {
        if (g < ep.matrices) {
#pragma unroll
          for (int k = 0; k < AT_ONCE; ++k) {
            const int c = lane + 64 * (k0 + k), gm = min(m0 + wm + p * 64 + c / PIECES, M - 1), gn = min(out_n0 + c % PIECES * 8, N - 8);
            const float4_t* at = reinterpret_cast<const float4_t*>(ep.table + ((size_t)(ep.first + gm) * ep.head_dim + gn % ep.head_dim) / 2);
            turn[k][0] = at[0];
            turn[k][1] = at[1];
          }
        }
      }
#pragma unroll
      for (int k = 0; k < AT_ONCE; ++k) {
        const int c = lane + 64 * (k0 + k), gm = m0 + wm + p * 64 + c / PIECES, gn = out_n0 + c % PIECES * 8;
        const float* from = rows + (c / PIECES) * shape::OUT_LD + c % PIECES * 8;
        const float4_t lo = *reinterpret_cast<const float4_t*>(from), hi = *reinterpret_cast<const float4_t*>(from + 4);
        const float x[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        if (gm >= M || gn >= out_n) continue;
        if constexpr (SPLIT) {
          float* to = part + ((size_t)split * M + gm) * N + gn;
          if (gn + 8 <= N) {
            *reinterpret_cast<any_float4_t*>(to) = lo;
            *reinterpret_cast<any_float4_t*>(to + 4) = hi;
          } else {
            for (int e = 0; e < 8 && gn + e < N; ++e) to[e] = x[e];
          }
        } else if constexpr (EP::BF16) {
          ep.store8(gm, gn, x, out_n);
        } else {
          half_t* to = out + (size_t)gm * out_n + gn;
          if (gn + 8 <= out_n) {  // llama_cu.cu:208-215: fp16(acc + beta * old)
            half8_t y;
#pragma unroll
            for (int e = 0; e < 8; ++e) y[e] = round_f16(beta != 0.0f ? fmaf(beta, (float)old[k][e], x[e]) : x[e]);
            if constexpr (EP::ROTARY) {
              if (g < ep.matrices) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                  const float real = (float)y[2 * e], imag = (float)y[2 * e + 1], cs = turn[k][e / 2][e % 2 * 2], sn = turn[k][e / 2][e % 2 * 2 + 1];
                  y[2 * e] = round_f16(fmaf(real, cs, -(imag * sn)));
                  y[2 * e + 1] = round_f16(fmaf(real, sn, imag * cs));
                }
              }
            }
            *reinterpret_cast<any_half8_t*>(to) = y;
          } else {
            for (int e = 0; e < 8 && gn + e < out_n; ++e) to[e] = round_f16(beta != 0.0f ? fmaf(beta, (float)to[e], x[e]) : x[e]);
          }
        }
      }
    }
  };
  static_for<shape::WR / 64>(pass);
}

}  // namespace lcu
