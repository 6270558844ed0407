// Matrix products of 2 to 64 rows: the weight stream is what counts.  fp16 or bfloat16 weights, or uint8 codes; fp32 sums
// of a run of K stages (64 of K) per output to part[matrix][split][M][N].
//
// What bounds it: a compute unit has so many cache lines on their way, 24 to 28 GB/s of cold ones, so each has
// to be given the same number of bytes, in whole lines, and asked for them without a pause.  A wavefront owns 16
// columns of W and brings 128 bytes of each of its rows at a time into an LDS ring of its own, three ahead, with no
// barrier; it shares nothing but lhs, which lies in LDS in one piece or in chunks.  One workgroup runs per compute unit, with
// as many wavefronts as give every compute unit one (stream_waves): 128-column tiles with a common ring left 288 workgroups
// of Wq, Wk, Wv for 256 compute units.  (Loaded into registers as the matrix instructions want them, sixteen rows
// per 16 lanes, a line takes four requests: slower for fp16 than the common ring.)
// M = 8 with a launch that adds the splits, fp16 three times (4096, 4096) 26.0 -> 22.7 us, twice (N, K) = (11008, 4096) 45 -> 42,
// (4096, 4096) 12.1 -> 12.4; uint8 three times (6656, 6656) 61 -> 35, twice (17920, 6656) 104 -> 57, (6656, 17920) 62 -> 37.  Rows of
// 8 KB meet in the same memory channels: K = 4224 takes a tenth less than 4096.
// ONCE: weights that come from memory, 64 MB of them and more in a launch, are marked as read once (nt; stream_once).  8 rows, twice 11008 columns
// of K 4096 36.8 -> 33.7 us (4.9 -> 5.35 TB/s), 16x4096x11008 22.4 -> 20.9, 60x6656x17920 53.6 -> 50.0; eight sequences of eight 7B layers, 45 + 16 tokens
// 23.4 -> 22.1 ms.
#pragma once
#include <algorithm>

#include "gemm_plan.hpp"
#include "gemm_tile.hpp"

namespace lcu {

constexpr int STREAM_RING = 4;
constexpr int STREAM_LHS = 64 * 1024;  // bytes of lhs in LDS: one chunk, or two of half of it
// a unit is 16 rows of 128 bytes; uint8: and a word with the scales of each row
constexpr int stream_unit(bool u8) { return 2048 + (u8 ? 256 : 0); }
constexpr int stream_lds(bool u8, int waves) { return STREAM_LHS + waves * STREAM_RING * stream_unit(u8); }
// JOINED: lhs whole, and behind the product the sums of every wavefront in its place, [wavefront][row][16]; the rest for the rings
constexpr int stream_joined_lhs(int waves, int row_tiles, int M, int K) {
  return std::max((M * K * 2 + 1023) / 1024 * 1024, waves * row_tiles * 1024);
}
constexpr int STREAM_LDS = 160 * 1024;
// K extent of a chunk of lhs: the longest run, counted from the 128 of K that it begins in, or what two chunks leave
inline int stream_chunk(int rows, int stages_in_all, int splits) {
  long longest = 0;
  for (long i = 0; i < splits; ++i) longest = std::max(longest, (i + 1) * stages_in_all / splits - (i * stages_in_all / splits & ~1L));
  const int whole = (int)(longest + 1) / 2 * 128;
  return rows * whole * 2 <= STREAM_LHS ? whole : STREAM_LHS / 4 / rows / 128 * 128;
}

// at most BASE requests outstanding, and `more` (0 .. 4) younger ones of another kind besides; this wavefront's LDS reads done
template <int BASE>
__device__ __forceinline__ void wait_requests(int more) {
  switch (more) {
    case 1: asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(BASE + 1) : "memory"); break;
    case 2: asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(BASE + 2) : "memory"); break;
    case 3: asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(BASE + 3) : "memory"); break;
    case 4: asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(BASE + 4) : "memory"); break;
    default: asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(BASE) : "memory"); break;
  }
}

// JOIN: what becomes of the sums.  separate_sums: they go to part, and another launch adds them up.  Otherwise a workgroup has every split of its
// columns (MATRICES 2: of those of both matrices), a wavefront each, and lhs lies in LDS whole; the sums meet in LDS, are added in the order of
// the splits, and join(matrix, row, first of two columns, sums of the two [MATRICES]) makes outputs of them.  What bounded the second launch was its
// start and its first loads, 2 to 4 us for a few hundred KB.  us, two launches / one, 8 rows: fp16 (K, N) = (4096, 4096) three times and the rotary
// 24.4 / 21.0, (4096, 11008) twice and the SiLU 44.2 / 41.2, (2048, 2048) three times 12.3 / 8.2, uint8 (4096, 4096) three times 19.8 / 15.7; alone, fp16
// 13x2048x6656 12.0 / 9.1, 40x256x16384 9.5 / 6.4, uint8 20x1408x6656 11.5 / 7.3; over 80 drawn shapes of 2 to 62 rows 12 to 58 % sooner where one launch does it.
// The rings take only what their wavefronts need, so that lhs may have more than STREAM_LHS: 34x1408x4096 10.3 -> 7.8, 10 rows of 4096 three times and the
// rotary 24.2 -> 21.3.
// GATED: the two are blocks of 32 columns of one matrix, a gate's and behind it an up block; the columns are those of the outputs.
struct separate_sums {
  static constexpr bool JOINED = false, GATED = false;
  static constexpr int MATRICES = 1;
};

template <int TM, bool U8, bool BF16, bool ONCE, class JOIN = separate_sums>
__global__ __launch_bounds__(64 * stream_max_waves(U8), 3) void gemm_stream_kernel(const half_t* __restrict__ A, const void* __restrict__ W0,
                                                                               const half_t* __restrict__ S0, int block_shift, int M, int K,
                                                                               int N, int tiles, int kc, float* __restrict__ part, int splits,
                                                                               more_matrices_t more, JOIN join) {
  constexpr int RING = STREAM_RING, UNIT = stream_unit(U8), P = U8 ? 3 : 2;  // requests per unit
  constexpr int PER = U8 ? 2 : 1;                                           // stages per unit
  extern __shared__ __attribute__((aligned(16))) unsigned char stream_mem[];
  const int waves = blockDim.x >> 6;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Tiles of one matrix, then of the next; the same for the next split.  Consecutive workgroups go round the eight XCDs: each
  // gets one run of the tiles, the same of every split, so that what adds the splits up may find them in one L2 (bfloat16,
  // 8 rows, 4096x2048, both launches: 11.9 us with the tiles dealt one by one, 8.3 so; fp16 4096x32000 66 / 61).
  constexpr bool JOINED = JOIN::JOINED;
  // JOINED: the sixteens of columns of all matrices are dealt, `groups` to a workgroup, `per` wavefronts to one of them.
  const int outs = JOIN::GATED ? N / 2 : N, sixteens = (outs + 15) / 16, per = JOINED ? splits * JOIN::MATRICES : 1, groups = waves / per;
  const int mats = more.tiles_n_per, nb = JOINED ? tiles : tiles * mats;
  const int split = JOINED ? wave % splits : blockIdx.x / nb, bx = JOINED ? blockIdx.x : blockIdx.x - split * nb, xcd = bx % 8;
  const int rest = xcd * (nb / 8) + min(xcd, nb % 8) + bx / 8, sixteen = rest * groups + wave / per;
  const int x = wave % per / splits;  // MATRICES 2: which of them
  const int g = !JOINED ? rest / tiles : JOIN::GATED ? 0 : JOIN::MATRICES == 2 ? x : sixteen / sixteens;
  const void* W = g == 0 ? W0 : (g == 1 ? more.W[0] : more.W[1]);
  const half_t* S = g == 0 ? S0 : (g == 1 ? more.S[0] : more.S[1]);
  const int of_matrix = !JOINED ? (rest - g * tiles) * waves + wave : JOIN::MATRICES == 2 ? sixteen : sixteen - g * sixteens;
  const int n0 = JOIN::GATED ? of_matrix / 2 * 64 + x * 32 + of_matrix % 2 * 16 : of_matrix * 16;
  const bool mine = of_matrix < sixteens && g < mats;
  const int nt_all = K / 64;
  const int stage0 = (int)((long)split * nt_all / splits), stage1 = (int)((long)(split + 1) * nt_all / splits);
  // stages are counted from an even one, so that units of two are whole lines of codes
  const int base = stage0 & ~1, first = stage0 - base, end = stage1 - base;
  const int units = (end + PER - 1) / PER;

  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)stream_mem;
  // lhs: rows of kc, 16-byte piece p of row r at p ^ r % 16 (within 16 pieces), so that the sixteen rows of a
  // fragment meet in no bank.
  const uint32_t row_bytes = (uint32_t)kc * 2, chunk_bytes = (uint32_t)(M * row_bytes + 1023) / 1024 * 1024;
  const auto request_chunk = [&](int chunk) {
    const int pieces = kc / 8;
    for (int u = wave; u * 64 < M * pieces; u += waves) {
      const int piece = min(u * 64 + lane, M * pieces - 1), row = piece / pieces, at = piece - row * pieces;
      const int k = min(((JOINED ? 0 : base * 64) + chunk * kc) + ((at & ~15) | ((at ^ row) & 15)) * 8, K - 8);
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(A + (size_t)row * K + k),
                   "s"(lds0 + (chunk & 1) * chunk_bytes + u * 1024)
                   : "memory", "m0");
    }
    return (M * pieces - wave * 64 + waves * 64 - 1) / (waves * 64);
  };

  // this wavefront's columns: rows of 128 bytes, 16-byte piece p of row r at p ^ (r / 2) % 8
  const uint32_t lhs_room = JOINED ? (uint32_t)stream_joined_lhs(waves, TM, M, K) : STREAM_LHS;
  const uint32_t ring0 = lds0 + lhs_room + wave * RING * UNIT;
  uint4_t rw = operand_resource(W, (uint32_t)N * (uint32_t)K * (U8 ? 1u : 2u)), rs = rw;
  if constexpr (U8) rs = operand_resource(S, (uint32_t)N * ((uint32_t)K >> (6 + block_shift)) * 2u);
  uint32_t w_off[2], s_first = 0;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int row = j * 8 + (lane >> 3), piece = (lane & 7) ^ ((row / 2) % 8);
    w_off[j] = row_piece(n0 + row, N, (uint32_t)K * (U8 ? 1u : 2u), piece);
  }
  const int col = lane & 15, group = lane >> 4;
  if constexpr (U8) s_first = (uint32_t)min(n0 + col, N - 1) * ((uint32_t)K >> (6 + block_shift));
  const auto request = [&](int u) {
    if (u == units) rw[2] = rs[2] = 0;  // behind the last unit: requests that count and touch no memory (stage_offset)
    const uint32_t slot = ring0 + (u % RING) * UNIT, along = stage_offset(rw[2], (uint32_t)(base * (U8 ? 64 : 128) + u * 128));
    if constexpr (ONCE) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen nt lds" ::"v"(w_off[j]), "s"(rw), "s"(along),
                     "s"(slot + j * 1024)
                     : "memory", "m0");
      }
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(w_off[j]), "s"(rw), "s"(along),
                     "s"(slot + j * 1024)
                     : "memory", "m0");
      }
    }
    if constexpr (U8) {  // the word that holds the row's scales of both stages
      const uint32_t at = s_first + ((uint32_t)(base + 2 * u) >> block_shift);
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dword %0, %1, 0 offen lds" ::"v"(scale_word(at)), "s"(rs), "s"(slot + 2048)
                   : "memory", "m0");
    }
  };

  float4_t acc[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) acc[i] = (float4_t)(0.0f);
  const int turn = (col / 2) % 8;
  uint32_t lhs_row[TM];  // rows past M: the last one, whose sums nobody stores there
  int lhs_turn[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int row = min(i * 16 + col, M - 1);
    lhs_row[i] = (uint32_t)row * row_bytes;
    lhs_turn[i] = row & 15;
  }
  // Stage s of chunk c, whose columns lie in `slot` (U8: in its first or second half).  Every fragment is asked for before the first product: left to
  // itself the compiler reads one, waits for it and multiplies it, eight times with 64 rows, and there are one or two wavefronts to a SIMD (us, so / here:
  // uint8 60x6656x17920 83.5 / 72.5, 40 rows 74.6 / 65.3, 20x6656x17920 37.6 / 35.1, 14x4096x11008 19.1 / 17.8; fp16 60x6656x17920 50.2 / 49.2).
  const auto multiply = [&](const unsigned char* slot, int s, int c) {
    half8_t w[2], a[2][TM];
    uint2_t codes[2];
    uint32_t word = 0;
    const unsigned char* row = slot + col * 128;
    if constexpr (U8) {
      word = *reinterpret_cast<const uint32_t*>(slot + 2048 + lane * 4);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int byte = (s & 1) * 64 + h * 32 + group * 8;
        codes[h] = *reinterpret_cast<const uint2_t*>(row + (((byte >> 4) ^ turn) << 4) + (byte & 8));
      }
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h) w[h] = *reinterpret_cast<const half8_t*>(row + (((4 * h + group) ^ turn) << 4));
    }
    const int p0 = JOINED ? (base + s) * 8 : (s * 64 - c * kc) / 8;
    const unsigned char* lhs = stream_mem + (JOINED ? 0 : (c & 1) * chunk_bytes);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int p = p0 + 4 * h + group;
#pragma unroll
      for (int i = 0; i < TM; ++i) a[h][i] = *reinterpret_cast<const half8_t*>(lhs + lhs_row[i] + ((p & ~15) | ((p ^ lhs_turn[i]) & 15)) * 16);
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (U8) {
      const uint32_t at = s_first + ((uint32_t)(base + s) >> block_shift);
      const half_t s2 = __builtin_bit_cast(half_t, (uint16_t)((at & 1) ? word >> 16 : word)) * (half_t)2.0f;
      const half2_t s2v = {s2, s2};
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const half2_t lo = dequant2(__builtin_amdgcn_perm(0u, codes[h][i], 0x0c010c00u), s2v);
          const half2_t hi = dequant2(__builtin_amdgcn_perm(0u, codes[h][i], 0x0c030c02u), s2v);
          w[h][4 * i] = lo.x, w[h][4 * i + 1] = lo.y, w[h][4 * i + 2] = hi.x, w[h][4 * i + 3] = hi.y;
        }
      }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        if constexpr (BF16) {
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a[h][i]), __builtin_bit_cast(bf16x8_t, w[h]), acc[i], 0, 0, 0);
        } else {
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[h][i], w[h], acc[i], 0, 0, 0);
        }
      }
    }
  };

  const int chunk_units = JOINED ? units : kc / 64 / PER, u0 = first / PER;
  request_chunk(0);
  if (mine) {
#pragma unroll
    for (int j = 0; j < RING - 1; ++j) request(u0 + j);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(P * (RING - 1)) : "memory");  // lhs, but not yet the columns
  } else {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  asm volatile("s_barrier" ::: "memory");
  for (int c = 0; c * chunk_units < units; ++c) {
    if (c > 0) {
      // chunk c was requested a chunk of units ago: before all that may still be out, if that is as long as the ring
      if (mine && chunk_units >= RING) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(P * (RING - 1)) : "memory");
      } else {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      }
      asm volatile("s_barrier" ::: "memory");
    }
    const int from = max(u0, c * chunk_units);
    int lhs_out = 0;  // requests of the next chunk, behind those of the RING - 1 units that are out
    if ((c + 1) * chunk_units < units) lhs_out = request_chunk(c + 1);  // into the half that was read before the barrier
    if (!mine) continue;
    for (int u = from; u < min(units, (c + 1) * chunk_units); ++u) {
      // unit u has landed, and the unit before it has been read: the ring may take another in its place
      wait_requests<P*(RING - 2)>(u - from < RING - 1 ? lhs_out : 0);
      request(u + RING - 1);
      const unsigned char* slot = stream_mem + lhs_room + (wave * RING + u % RING) * UNIT;
#pragma unroll
      for (int e = 0; e < PER; ++e) {
        const int s = u * PER + e;
        if (PER == 1 || (s >= first && s < end)) multiply(slot, s, c);
      }
    }
  }
  if constexpr (JOINED) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");  // everybody has read lhs, whose place the sums take
    float* sums = reinterpret_cast<float*>(stream_mem);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int e = 0; e < 4; ++e) sums[(wave * TM * 16 + i * 16 + group * 4 + e) * 16 + col] = acc[i][e];
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
    for (int at = threadIdx.x; at < groups * M * 8; at += blockDim.x) {
      const int c = at % 8 * 2, m = at / 8 % M, block = at / 8 / M, of = rest * groups + block;
      const int matrix = JOIN::MATRICES == 2 ? 0 : of / sixteens, n = (of - matrix * sixteens) * 16 + c;
      if (n >= outs || matrix >= mats) continue;
      float2 total[JOIN::MATRICES];
#pragma unroll
      for (int y = 0; y < JOIN::MATRICES; ++y) {
        const float* from = sums + ((block * per + y * splits) * TM * 16 + m) * 16 + c;
        total[y] = *reinterpret_cast<const float2*>(from);
        for (int s = 1; s < splits; ++s) {
          const float2 more_of_it = *reinterpret_cast<const float2*>(from + s * TM * 256);
          total[y].x += more_of_it.x;
          total[y].y += more_of_it.y;
        }
      }
      join(matrix, m, n, total);
    }
    return;
  }
  if (!mine) return;
  // register e of a lane is row 4 group + e, column col of its tile
  part += ((size_t)g * splits + split) * M * N;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int m = i * 16 + group * 4 + e;
      if (m < M && n0 + col < N) part[(size_t)m * N + n0 + col] = acc[i][e];
    }
  }
}

}  // namespace lcu
