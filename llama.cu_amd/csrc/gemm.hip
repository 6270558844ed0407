// Prefill matrix products on the gfx950 matrix cores: out[M,N] = lhs[M,K] * W[N,K]^T + beta*out.
//
// These replace matmul_nt_wmma_128x64x64 (llama_cu.cu:150-220) and, for uint8 weights,
// matmul_nt_wmma_16x128x256_fp16u8 at M > 1 (294-366).  Both operands are K-contiguous, which is
// the natural operand order of v_mfma_f32_32x32x16_f16: every lane feeds 8 consecutive k of one
// row of lhs (A) and of one row of W (B).
//
// Four kernels:
//   gemm_tile_kernel (gemm_tile.hpp): 256-row tiles of 128, 192 or 256 columns where these fill most of the
//     chip, 256x128 with the K range split over workgroups, 128-row tiles of up to 128 rows and where only
//     those of 128x128 fill most of the chip, else 128x64; fp16, uint8 (codes in blocks of 64 << n) and bfloat16 weights
//   gemm_stream_kernel (gemm_stream.hpp): 2..64 rows, the K range split over wavefronts that add up their sums and finish
//     the outputs, or over workgroups
//   gemm_dl_kernel (K a multiple of 128; a short K where 128x128 tiles fill the chip, other blocks of codes, splits of few rows,
//     bfloat16 experts and small tiles): both operands travel from global memory straight into a ring of 2-3 LDS
//     stages with global_load_lds_dwordx4 (no staging registers, no LDS store instructions); rows are
//     unpadded and the 16-byte chunks of a row are permuted so that neither the requests nor the fragment
//     reads meet in a bank; 4 or 8 wavefronts (a second group of four may take the other half of a 128-wide K
//     stage), chosen by how many tiles the product has; uint8 weights add a ring of codes and of scales and are
//     turned into fp16 -- exactly fp16((q - 127.5) * scale), llama_cu.cu:287-289 -- once per block tile
//   Where the K range is split over workgroups -- 2..64 rows, few large tiles and a long K -- a second launch adds the
//     fp32 partial sums in split order (launch_skinny; large_tile_splits in gemm_plan.hpp)
//   gemm_kernel (ragged K): global -> registers -> padded LDS with two LDS buffers and two
//     register stages, uint8 weights dequantised between the load and the LDS store
// All: the K loop carries no vector address arithmetic and no predication; the block index ->
// tile mapping keeps the tiles that share a slice of W on one XCD (one L2); rows >= M and columns
// >= N are masked instead of the reference's zeroed "gutter" rows (llama_cu.h:236-242).
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "gemm_plan.hpp"
#include "gemm_stream.hpp"
#include "gemm_tile.hpp"
#include "linear.hpp"

using namespace lcu;

namespace lcu {
int gemv_f16(half_t* out, const half_t* x, const half_t* W, int K, int N, float beta, hipStream_t st);
int gemv_u8(half_t* out, const half_t* x, const uint8_t* W, const half_t* S, int K, int N, int block, float beta,
            hipStream_t st);
}  // namespace lcu

namespace {

constexpr int BK = 64;        // K extent one group of four wavefronts multiplies per stage
constexpr int NUM_XCD = 8;

// KS: groups of four wavefronts per workgroup.  A stage holds KS * 64 of K; group g multiplies
// columns g*64 .. g*64+63 of it into its own accumulators, and the groups' accumulators are added
// through LDS at the end (group 0 + group 1, a fixed order).  With KS = 2 every SIMD holds two
// wavefronts of the same tile, so one can wait for LDS while the other feeds the matrix core --
// what a second resident workgroup does when the grid has one to give, which at M = 512 it has not.
// KTAIL: K is not a multiple of the stage, so the last stage is partly out of range and is zeroed
// (costs selects in the loop; every model shape takes the KTAIL = false instantiation).
template <int BM, int BN, bool U8, bool KTAIL, int KS>
__global__ __launch_bounds__(256 * KS, KS == 1 ? 2 : 1) void gemm_kernel(
    half_t* __restrict__ out, const half_t* __restrict__ A, const void* __restrict__ Wv, const half_t* __restrict__ S,
    int M, int K, int N, int block, float beta, int tiles_m, int tiles_n) {
  constexpr int THREADS = 256 * KS;
  constexpr int BKS = BK * KS;   // K extent of a stage
  constexpr int LDK = BKS + 8;   // halves per LDS row: 16 bytes of padding keep 16-byte reads of 16 lanes in distinct banks
  constexpr int TM = BM / 64;    // 32x32 MFMA tiles per wavefront along M
  constexpr int TN = BN / 64;
  constexpr int A_ROW = BKS / 8;                  // 16-byte chunks per tile row of lhs
  constexpr int B_ROW = U8 ? BKS / 16 : BKS / 8;  // 16-byte chunks per tile row of W
  constexpr int A_CHUNKS = BM * A_ROW / THREADS;  // chunks per thread
  constexpr int B_CHUNKS = BN * B_ROW / THREADS;
  static_assert(A_CHUNKS >= 1 && B_CHUNKS >= 1, "tile too small for the workgroup");

  extern __shared__ __attribute__((aligned(16))) unsigned char gemm_lds[];
  half_t* As = reinterpret_cast<half_t*>(gemm_lds);  // [2][BM * LDK]
  half_t* Bs = As + 2 * BM * LDK;                    // [2][BN * LDK]

  // XCD-aware tile order: hardware deals consecutive workgroups round-robin to the 8 XCDs, so
  // give each XCD one contiguous run of the M-fastest tile sequence.
  const int nb = tiles_m * tiles_n;
  const int bid = blockIdx.x;
  const int q = nb / NUM_XCD, r = nb % NUM_XCD;
  const int xcd = bid % NUM_XCD, idx = bid / NUM_XCD;
  const int logical = xcd * q + min(xcd, r) + idx;
  const int tm = logical % tiles_m, tn = logical / tiles_m;
  const int m0 = tm * BM, n0 = tn * BN;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int group = wave >> 2, w4 = wave & 3;
  const int wm = (w4 & 1) * (BM / 2), wn = (w4 >> 1) * (BN / 2);
  const int nblk = U8 ? K / block : 0;

  // Per-thread byte offsets of its chunks from the operand bases; they do not change over the K
  // loop, which only advances a uniform base, so the loop carries no vector address arithmetic.
  // Rows past M or N are clamped to the last row: their products land in accumulator rows and
  // columns that the epilogue never stores, so no zero fill is needed for them.
  uint32_t a_off[A_CHUNKS], b_off[B_CHUNKS], s_off[U8 ? B_CHUNKS : 1];
  int a_k[A_CHUNKS], b_k[B_CHUNKS];
#pragma unroll
  for (int i = 0; i < A_CHUNKS; ++i) {
    const int c = tid + i * THREADS;
    a_k[i] = (c % A_ROW) * 8;
    a_off[i] = ((uint32_t)min(m0 + c / A_ROW, M - 1) * (uint32_t)K + a_k[i]) * 2u;
  }
#pragma unroll
  for (int i = 0; i < B_CHUNKS; ++i) {
    const int c = tid + i * THREADS;
    const uint32_t row = (uint32_t)min(n0 + c / B_ROW, N - 1);
    if constexpr (U8) {
      b_k[i] = (c % B_ROW) * 16;
      b_off[i] = row * (uint32_t)K + b_k[i];
      s_off[i] = row * (uint32_t)nblk;
    } else {
      b_k[i] = (c % B_ROW) * 8;
      b_off[i] = (row * (uint32_t)K + b_k[i]) * 2u;
    }
  }
  const char* Ab = (const char*)A;
  const char* Wb = (const char*)Wv;

  // one stage of both operands in registers, as loaded from global memory
  struct stage_t {
    half8_t ra[A_CHUNKS];
    half8_t rb[U8 ? 1 : B_CHUNKS];
    uint4_t rq[U8 ? B_CHUNKS : 1];
    half_t rs[U8 ? B_CHUNKS : 1];
    int k0;
  };

  // Unconditional loads: a predicated load becomes a branch, and branches make the compiler wait
  // for every outstanding load before it issues the next ones.  With KTAIL the k offset is
  // clamped into range here and the chunk is zeroed when it is stored to LDS.
  auto load_tile = [&](stage_t& st, int k0) {
    st.k0 = k0;
#pragma unroll
    for (int i = 0; i < A_CHUNKS; ++i) {
      int kk = k0;
      if constexpr (KTAIL) kk = min(k0, K - 8 - a_k[i]);
      st.ra[i] = *reinterpret_cast<const half8_t*>(Ab + (ptrdiff_t)kk * 2 + a_off[i]);
    }
    if constexpr (U8) {
#pragma unroll
      for (int i = 0; i < B_CHUNKS; ++i) {
        int kk = k0;
        if constexpr (KTAIL) kk = min(k0, K - 16 - b_k[i]);
        st.rq[i] = *reinterpret_cast<const uint4_t*>(Wb + (ptrdiff_t)kk + b_off[i]);
        st.rs[i] = S[s_off[i] + (uint32_t)(kk + b_k[i]) / (uint32_t)block];
      }
    } else {
#pragma unroll
      for (int i = 0; i < B_CHUNKS; ++i) {
        int kk = k0;
        if constexpr (KTAIL) kk = min(k0, K - 8 - b_k[i]);
        st.rb[i] = *reinterpret_cast<const half8_t*>(Wb + (ptrdiff_t)kk * 2 + b_off[i]);
      }
    }
  };

  auto store_tile = [&](const stage_t& st, int buf) {
    half_t* Ad = As + buf * BM * LDK;
    half_t* Bd = Bs + buf * BN * LDK;
#pragma unroll
    for (int i = 0; i < A_CHUNKS; ++i) {
      const int c = tid + i * THREADS;
      half8_t v = st.ra[i];
      if constexpr (KTAIL) v = (st.k0 + a_k[i] < K) ? v : (half8_t)(0.0f);
      *reinterpret_cast<half8_t*>(&Ad[(c / A_ROW) * LDK + a_k[i]]) = v;
    }
    if constexpr (U8) {
#pragma unroll
      for (int i = 0; i < B_CHUNKS; ++i) {
        const int c = tid + i * THREADS;
        half_t s2 = st.rs[i] * (half_t)2.0f;
        if constexpr (KTAIL) s2 = (st.k0 + b_k[i] < K) ? s2 : (half_t)0.0f;  // zero scale: zero weights
        const half2_t s2v = {s2, s2};
        half2_t d[8];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          d[2 * j] = dequant2(__builtin_amdgcn_perm(0u, st.rq[i][j], 0x0c010c00u), s2v);
          d[2 * j + 1] = dequant2(__builtin_amdgcn_perm(0u, st.rq[i][j], 0x0c030c02u), s2v);
        }
        half8_t lo = {d[0].x, d[0].y, d[1].x, d[1].y, d[2].x, d[2].y, d[3].x, d[3].y};
        half8_t hi = {d[4].x, d[4].y, d[5].x, d[5].y, d[6].x, d[6].y, d[7].x, d[7].y};
        half_t* dst = &Bd[(c / B_ROW) * LDK + b_k[i]];
        *reinterpret_cast<half8_t*>(dst) = lo;
        *reinterpret_cast<half8_t*>(dst + 8) = hi;
      }
    } else {
#pragma unroll
      for (int i = 0; i < B_CHUNKS; ++i) {
        const int c = tid + i * THREADS;
        half8_t v = st.rb[i];
        if constexpr (KTAIL) v = (st.k0 + b_k[i] < K) ? v : (half8_t)(0.0f);
        *reinterpret_cast<half8_t*>(&Bd[(c / B_ROW) * LDK + b_k[i]]) = v;
      }
    }
  };

  float16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      acc[i][j] = (float16_t)(0.0f);
    }
  }

  // Operand fragments are read one 16-wide K slice ahead of the matrix instructions that use
  // them (left to itself the compiler reads a fragment and waits for it in front of every
  // instruction, and the matrix core idles for the LDS latency each time).
  const int frag_row = lane & 31, frag_k = group * BK + (lane >> 5) * 8;
  auto compute = [&](int buf) {
    const half_t* Ad = As + buf * BM * LDK + (wm + frag_row) * LDK + frag_k;
    const half_t* Bd = Bs + buf * BN * LDK + (wn + frag_row) * LDK + frag_k;
    half8_t fa[2][TM], fb[2][TN];
    auto read_frags = [&](int slot, int ks) {
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[slot][i] = *reinterpret_cast<const half8_t*>(Ad + i * 32 * LDK + ks);
#pragma unroll
      for (int j = 0; j < TN; ++j) fb[slot][j] = *reinterpret_cast<const half8_t*>(Bd + j * 32 * LDK + ks);
    };
    read_frags(0, 0);
#pragma unroll
    for (int s = 0; s < BK / 16; ++s) {
      if (s + 1 < BK / 16) read_frags((s + 1) & 1, (s + 1) * 16);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[s & 1][i], fb[s & 1][j], acc[i][j], 0, 0, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // Pipeline: LDS buffer t%2 holds stage t; one register stage holds stage t+1 (requested one
  // iteration ago) and the other receives stage t+2 while the matrix cores work on stage t.
  // Two iterations per trip so that the two register stages keep fixed names.
  stage_t s0, s1;
  const int nt = (K + BKS - 1) / BKS;
  load_tile(s0, 0);
  if (nt > 1) load_tile(s1, BKS);
  store_tile(s0, 0);
  __syncthreads();
  for (int t = 0; t < nt; t += 2) {
    // stage t in LDS 0, stage t+1 in s1
    if (t + 2 < nt) load_tile(s0, (t + 2) * BKS);
    compute(0);
    if (t + 1 < nt) store_tile(s1, 1);
    __syncthreads();
    if (t + 1 >= nt) break;
    // stage t+1 in LDS 1, stage t+2 in s0
    if (t + 3 < nt) load_tile(s1, (t + 3) * BKS);
    compute(1);
    if (t + 2 < nt) store_tile(s0, 0);
    __syncthreads();
  }

  // the groups' partial sums meet in LDS (every wavefront is past its last LDS read: each compute
  // above is followed by a barrier); element (tile, v) of lane l sits at ((w4, tile, v), l)
  if constexpr (KS == 2) {
    float* part = reinterpret_cast<float*>(gemm_lds);
    if (group == 1) {
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            part[(((w4 * TM + i) * TN + j) * 16 + v) * 64 + lane] = acc[i][j][v];
          }
        }
      }
    }
    __syncthreads();
    if (group == 1) return;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          acc[i][j][v] += part[(((w4 * TM + i) * TN + j) * 16 + v) * 64 + lane];
        }
      }
    }
  }

  // epilogue, llama_cu.cu:208-215: fp16(acc + beta * old).  Accumulator register v of lane l is
  // element (row 8*(v/4) + 4*(l/32) + v%4, column l%32) of the 32x32 tile.
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int gn = n0 + wn + j * 32 + (lane & 31);
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int gm = m0 + wm + i * 32 + (v >> 2) * 8 + (lane >> 5) * 4 + (v & 3);
        if (gm < M && gn < N) {
          half_t* p = out + (size_t)gm * N + gn;
          float val = acc[i][j][v];
          if (beta != 0.0f) {
            val = fmaf(beta, (float)*p, val);
          }
          *p = round_f16(val);
        }
      }
    }
  }
}

// ---- fp16 weights, K a multiple of the stage: operands go from global memory straight into LDS
// (global_load_lds_dwordx4: no staging registers, no LDS store instructions, and the wavefront
// does not wait for a load before it can go on), through a ring of NS stages.
//
// A load instruction of one wavefront fills 1 KB of LDS, lane l at byte 16*l, so tile rows lie
// densely (ROWB bytes each, no padding) and bank conflicts are avoided by permuting the 16-byte
// chunks inside a row instead: the chunk that holds K offsets 8g..8g+7 of tile row r is stored at
// chunk position g ^ f(r), f(r) = (r / RPB) % CR.  Sixteen lanes reading the same g from sixteen
// consecutive rows then cover all 64 banks exactly once.
//
// Per iteration: wait until this wavefront's loads of stage t have landed, barrier (so everybody's
// have), request stage t+NS-1 into the slot whose reads ended before that barrier, multiply
// stage t.  The compiler does not track these loads against LDS reads; the waits are explicit.
// WM x WN wavefronts tile the block (each a (BM/WM) x (BN/WN) sub-tile of 32x32 matrix-instruction
// tiles), times KS groups along K.
//
// Tried and dropped: an extra wavefront that touches the lines of a stage several stages ahead so
// that the loaders hit L2.  About a sixth of the requests come from HBM, but the touches (64
// separate lines per instruction) cost the texture addresser more than the misses cost the ring.
//
// uint8 weights (U8): the codes travel the same way, into a ring of their own, one stage further
// ahead than the lhs tile ("batch" b of requests = lhs of stage b + codes of stage b+1).  During
// stage t the workgroup turns the codes of stage t+1 into the fp16 tile the matrix instructions
// read -- every thread one 16-code chunk, each weight exactly fp16((q - 127.5) * scale), written
// at the same permuted chunk positions a direct fp16 load would have filled -- so a weight is
// dequantised once per block tile and the fragment path is the fp16 one.  The chunk's scale comes
// by an ordinary 2-byte load one stage earlier.
//
// SPLIT (few rows that gemm_stream_kernel leaves, blocks of codes other than 64 << n): the grid holds
// `splits` workgroups per tile, each taking a contiguous run of the K stages and writing its fp32 sums to
// part[split][M][N]; splitk_reduce_kernel adds them in split order and applies the epilogue.
//
// EP: what the accumulators become.  f16_epilogue is the fp16 output described above.  The bfloat16
// epilogues (linear.hpp) take bfloat16 operands, which travel exactly like the fp16 ones, through
// v_mfma_f32_32x32x16_bf16, and end in a bias, a GELU, or a clamped gate; GROUPED ones take the
// rows of a tile and its weight matrix from a tile list on the device (lcu_experts_plan).
template <int BM, int BN, int WM, int WN, int KS, int NS, bool U8, bool SPLIT = false, class EP = f16_epilogue>
__global__ __launch_bounds__(64 * WM * WN * KS, WM * WN * KS <= 4 ? 2 : 1) void gemm_dl_kernel(
    half_t* __restrict__ out0, const half_t* __restrict__ A, const void* __restrict__ W0, const half_t* __restrict__ S0,
    int M, int K, int N, int block, float beta, int tiles_m, int tiles_n, float* __restrict__ part, int splits,
    more_matrices_t more, EP ep) {
  constexpr int NG = WM * WN;                // wavefronts of one group
  constexpr int NW = NG * KS;                // wavefronts
  constexpr int BKS = BK * KS;               // K extent of a stage
  constexpr int ROWB = BKS * 2;              // bytes of a tile row in LDS
  constexpr int CR = ROWB / 16;              // 16-byte chunks per row: 8 or 16
  constexpr int RPB = 16 / CR;               // tile rows per 256 bytes (one pass over the banks)
  constexpr int THREADS = 64 * NW;
  constexpr int CPR = BKS / 16;              // 16-code chunks per row of the code tile
  constexpr int PA = BM * CR / 64 / NW;      // load instructions per wavefront per stage, lhs
  constexpr int PB = U8 ? BN * CPR / 64 / NW : BN * CR / 64 / NW;  // and W (fp16 values or codes)
  constexpr int DC = U8 ? BN * CPR / THREADS : 1;                  // code chunks a thread dequantises per stage
  constexpr int A_BYTES = BM * ROWB, B_BYTES = BN * ROWB, C_BYTES = BN * BKS;
  constexpr int NB = U8 ? 2 : NS;            // fp16 W tiles held: written one stage ahead, or the ring itself
  // fp16: slot s of the ring holds lhs and W tile of a stage side by side; uint8: lhs ring, then the
  // two fp16 W tiles, then the code ring
  constexpr int A_STRIDE = U8 ? A_BYTES : A_BYTES + B_BYTES, B_STRIDE = U8 ? B_BYTES : A_BYTES + B_BYTES;
  constexpr int B_BASE = U8 ? NS * A_BYTES : A_BYTES, C_BASE = NS * A_BYTES + NB * B_BYTES;
  constexpr int S_BYTES = THREADS * 4 * DC;  // scale ring slot: one dword per thread and chunk
  constexpr int S_BASE = C_BASE + NS * C_BYTES;
  constexpr int LDS_BYTES = NS * A_BYTES + NB * B_BYTES + (U8 ? NS * (C_BYTES + S_BYTES) : 0);
  constexpr int TM = BM / (32 * WM), TN = BN / (32 * WN);
  static_assert(PA >= 1 && PB >= 1 && DC >= 1 && NS >= 2 && NS <= 4, "unsupported configuration");
  static_assert(!U8 || NS == 3, "the uint8 schedule is written for a ring of three");
  constexpr int P = PA + PB + (U8 ? DC : 0);  // requests per wavefront and batch
  static_assert(P * (NS - 1) < 64, "vmcnt has 6 bits");

  extern __shared__ __attribute__((aligned(16))) unsigned char gemm_lds[];

  const int nb = tiles_m * tiles_n;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int group = wave / NG, w4 = wave % NG;
  const int wm = (w4 % WM) * (BM / WM), wn = (w4 / WM) * (BN / WN);
  // XCD-aware tile order, as in gemm_kernel
  const int split = SPLIT ? blockIdx.x / nb : 0;
  const int bx = SPLIT ? blockIdx.x - split * nb : blockIdx.x;
  const int q = nb / NUM_XCD, r = nb % NUM_XCD;
  const int xcd = bx % NUM_XCD, idx = bx / NUM_XCD;
  const int logical = xcd * q + min(xcd, r) + idx;
  int tm = logical % tiles_m;
  int tn = logical / tiles_m;
  int e = 0;  // GROUPED: the group of this tile
  if constexpr (EP::GROUPED) {
    const group_tile_t at = group_tile(ep, tiles_n, bx);
    if (at.group < 0) return;
    e = at.group, tm = at.row_tile, tn = at.column_tile;
  }
  // which weight matrix this tile belongs to: chosen once, from kernel arguments (scalar selects)
  half_t* out = out0;
  const void* W = W0;
  const half_t* S = S0;
  if (more.tiles_n_per > 0) {
    const int g = tn / more.tiles_n_per;
    tn -= g * more.tiles_n_per;
    out = g == 0 ? out0 : (g == 1 ? more.out[0] : more.out[1]);
    W = g == 0 ? W0 : (g == 1 ? more.W[0] : more.W[1]);
    S = g == 0 ? S0 : (g == 1 ? more.S[0] : more.S[1]);
    if constexpr (SPLIT) {
      part += (size_t)g * splits * M * N;  // each matrix has its own partial sums
    }
  }
  int m0 = tm * BM;
  const int n0 = tn * BN;
  if constexpr (EP::GROUPED) {
    m0 = ep.tile_row[tm];
    M = ep.group_end[e];
    W = (const char*)W0 + (size_t)e * ep.group_stride;
  }

  // beta != 0: the old values of the output tile, asked for now in 16-byte pieces (tile row c / (BN / 8), eight
  // columns from 8 (c % (BN / 8))) and handed to the lanes that need them through LDS after the last stage.
  // Read lane by lane in the accumulators' layout (2-byte requests, two rows of 64 bytes per instruction) they cost
  // the 512 x 4096 x 4096 product 6 us.  Rows of N % 8 != 0 are not 16-byte aligned: those keep the 2-byte reads.
  // Only where a thread holds at most two pieces (the 128 x 64 tile of 512 threads, which carries Wo): the
  // registers that more pieces occupy through the K loop cost the 256 x 128 tile 5 % with beta = 0.
  constexpr int OC = BM * BN / 8 / THREADS;  // pieces per thread
  constexpr int OLD_LD = BN + 8;             // halves per tile row in LDS
  constexpr bool OLD_PIECES = !SPLIT && !EP::BF16 && OC <= 2;
  static_assert(!OLD_PIECES || (BM * BN / 8 % THREADS == 0 && BM * OLD_LD * 2 <= LDS_BYTES), "old tile staging");
  // 16-byte requests: rows of a multiple of 8 halves from a 16-byte aligned base (anything else keeps
  // the 2-byte reads of the epilogue)
  const bool old_by_pieces = OLD_PIECES && beta != 0.0f && N % 8 == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
  uint4_t old_piece[OC];
  if constexpr (OLD_PIECES) {
    if (old_by_pieces) {
#pragma unroll
      for (int j = 0; j < OC; ++j) {
        const int c = tid + j * THREADS;
        const int gm = m0 + c / (BN / 8), gn = n0 + (c % (BN / 8)) * 8;
        old_piece[j] = (uint4_t)(0u);
        if (gm < M && gn < N) old_piece[j] = *reinterpret_cast<const uint4_t*>(out + (size_t)gm * N + gn);
      }
    }
  }

  // loader: instruction j of this wavefront fills LDS bytes [(wave + j*NW) * 1024, +1024) of the
  // operand's region; lane l lands on tile row c / CR, chunk position c % CR, c = that index * 64 + l
  uint32_t a_off[PA], b_off[PB];
#pragma unroll
  for (int j = 0; j < PA; ++j) {
    const int c = (wave + j * NW) * 64 + lane;
    const int row = c / CR, g = (c % CR) ^ ((row / RPB) % CR);
    int gm = min(m0 + row, M - 1);
    if constexpr (EP::GROUPED) {
      if (ep.row_index) gm = ep.row_index[gm];
    }
    a_off[j] = ((uint32_t)gm * (uint32_t)K + g * 8) * 2u;
  }
#pragma unroll
  for (int j = 0; j < PB; ++j) {
    const int c = (wave + j * NW) * 64 + lane;
    if constexpr (U8) {  // codes lie densely and unpermuted: chunk c of the tile at byte 16 c
      b_off[j] = (uint32_t)min(n0 + c / CPR, N - 1) * (uint32_t)K + (c % CPR) * 16;
    } else {
      const int row = c / CR, g = (c % CR) ^ ((row / RPB) % CR);
      b_off[j] = ((uint32_t)min(n0 + row, N - 1) * (uint32_t)K + g * 8) * 2u;
    }
  }
  // this workgroup's K stages: all of them, or its share [stage0, stage0 + nt) of a split
  const int nt_all = K / BKS;
  const int stage0 = SPLIT ? (int)((long)split * nt_all / splits) : 0;
  const int nt = SPLIT ? (int)((long)(split + 1) * nt_all / splits) - stage0 : nt_all;
  const int k_base = stage0 * BKS;
  const char* Ab = (const char*)A + (size_t)k_base * 2;
  const char* Wb = (const char*)W + (size_t)k_base * (U8 ? 1 : 2);
  // uint8: the chunks this thread dequantises (tile row, chunk in the row), their scale index at
  // stage 0, and where the two fp16 chunks of a dequantised chunk go in the W tile
  int d_scale[DC];
  uint32_t d_src[DC], d_dst0[DC], d_dst1[DC];
  const bool hi_first = (tid >> 2) & 1;
  const int nblk = U8 ? K / block : 0;
  if constexpr (U8) {
#pragma unroll
    for (int i = 0; i < DC; ++i) {
      const int c = tid + i * THREADS;
      const int row = c / CPR, kc = c % CPR, f = (row / RPB) % CR;
      d_scale[i] = min(n0 + row, N - 1) * nblk;
      d_src[i] = (uint32_t)c * 16;
      d_dst0[i] = (uint32_t)row * ROWB + (uint32_t)(((2 * kc) ^ f) * 16);
      d_dst1[i] = (uint32_t)row * ROWB + (uint32_t)(((2 * kc + 1) ^ f) * 16);
      // LDS stores see 32 banks (128 bytes): eight consecutive lanes must land on eight different
      // chunk positions modulo 8.  Four lanes share a row (or half a row) and would all write even
      // positions with their first store; so every second group of four lanes writes its odd chunk
      // first (8 conflict cycles per store instruction otherwise).
      if (hi_first) {
        const uint32_t t0 = d_dst0[i];
        d_dst0[i] = d_dst1[i];
        d_dst1[i] = t0;
      }
    }
  }
  // A request is written as inline assembly (M0 = LDS address of the wavefront's 1 KB, then the
  // load), so that the compiler does not know about it: knowing, it treats the request like a FLAT
  // access and waits for every LDS read in front of each matrix instruction.  Nothing else in this
  // kernel uses M0.  The data lands in LDS, not in a register, so there is nothing here the
  // compiler could copy too early; the waits for it (vmcnt) are the explicit ones below.
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)gemm_lds;
  auto request16 = [&](const void* g, uint32_t lds_off) {
    const uint32_t m0 = __builtin_amdgcn_readfirstlane(lds0 + lds_off);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(m0) : "memory", "m0");
  };
  auto request4 = [&](const void* g, uint32_t lds_off) {
    const uint32_t m0 = __builtin_amdgcn_readfirstlane(lds0 + lds_off);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(g), "s"(m0) : "memory", "m0");
  };
  // request `idx` (0 .. P-1) of this wavefront for batch `stage` into ring slot `slot`: the lhs tile
  // of that stage, and the W tile of that stage (fp16) or the codes and scales of the stage after it
  // (uint8; past the end the last stage is fetched again and never used)
  auto issue_one = [&](int stage, int slot, int idx) {
    if (idx < PA) {
      request16(Ab + (size_t)stage * (BKS * 2) + a_off[idx], slot * A_STRIDE + (wave + idx * NW) * 1024);
    } else if constexpr (U8) {
      const int cslot = slot + 1 == NS ? 0 : slot + 1;
      const int st1 = min(stage + 1, nt - 1);
      if (idx < PA + PB) {
        request16(Wb + (size_t)st1 * BKS + b_off[idx - PA], C_BASE + cslot * C_BYTES + (wave + (idx - PA) * NW) * 1024);
      } else {
        const int i = idx - PA - PB;  // the dword that holds this thread's fp16 scale of chunk i
        const int kc = (tid + i * THREADS) % CPR;
        const int at = d_scale[i] + (k_base + st1 * BKS + kc * 16) / block;
        request4(S + (at & ~1), S_BASE + cslot * S_BYTES + (i * NW + wave) * 256);
      }
    } else {
      request16(Wb + (size_t)stage * (BKS * 2) + b_off[idx - PA], B_BASE + slot * B_STRIDE + (wave + (idx - PA) * NW) * 1024);
    }
  };
  auto issue = [&](int stage, int slot) {
#pragma unroll
    for (int idx = 0; idx < P; ++idx) issue_one(stage, slot, idx);
  };

  float16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      acc[i][j] = (float16_t)(0.0f);
    }
  }

  // reader: chunk position of K slice s (16 wide) for this lane; the row term of f() is the same
  // for every 32-row tile of the wavefront because 32 / RPB is a multiple of CR
  const int frag_row = lane & 31;
  const int fr = (frag_row / RPB) % CR;
  const int gbase = group * 8 + (lane >> 5);
  uint32_t pos[BK / 16];
#pragma unroll
  for (int s4 = 0; s4 < BK / 16; ++s4) pos[s4] = (uint32_t)(((gbase + 2 * s4) ^ fr) * 16);
  const uint32_t a_row = (uint32_t)(wm + frag_row) * ROWB, b_row = (uint32_t)B_BASE + (uint32_t)(wn + frag_row) * ROWB;

  // codes and scales in ring slot `cslot` (they belong to K stage `stage`) -> fp16 W tile `bslot`
  auto dequantise = [&](int cslot, int bslot, int stage) {
#pragma unroll
    for (int i = 0; i < DC; ++i) {
      const uint4_t q = *reinterpret_cast<const uint4_t*>(gemm_lds + C_BASE + cslot * C_BYTES + d_src[i]);
      const uint32_t pair = *reinterpret_cast<const uint32_t*>(gemm_lds + S_BASE + cslot * S_BYTES + i * THREADS * 4 + tid * 4);
      const int kc = (tid + i * THREADS) % CPR;
      const int at = d_scale[i] + (k_base + stage * BKS + kc * 16) / block;  // the request fetched the dword at (at & ~1)
      const half_t sc = __builtin_bit_cast(half_t, (uint16_t)((at & 1) ? pair >> 16 : pair & 0xffffu));
      const half_t s2 = sc * (half_t)2.0f;
      const half2_t s2v = {s2, s2};
      half2_t d[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        d[2 * j] = dequant2(__builtin_amdgcn_perm(0u, q[j], 0x0c010c00u), s2v);
        d[2 * j + 1] = dequant2(__builtin_amdgcn_perm(0u, q[j], 0x0c030c02u), s2v);
      }
      const half8_t lo = {d[0].x, d[0].y, d[1].x, d[1].y, d[2].x, d[2].y, d[3].x, d[3].y};
      const half8_t hi = {d[4].x, d[4].y, d[5].x, d[5].y, d[6].x, d[6].y, d[7].x, d[7].y};
      unsigned char* tile = gemm_lds + B_BASE + bslot * B_STRIDE;
      *reinterpret_cast<half8_t*>(tile + d_dst0[i]) = hi_first ? hi : lo;
      *reinterpret_cast<half8_t*>(tile + d_dst1[i]) = hi_first ? lo : hi;
    }
  };

  // ---- the stage loop --------------------------------------------------------------------------
  // K slice s of a stage uses fragment buffer s & 1.  Per stage and wavefront:
  //   slices 0..2: read slice s+1 | request a third of the batch NS-1 ahead | multiply slice s
  //   slice 3:     wait for this wavefront's LDS accesses (it is then done with the stage) | wait
  //                for its own requests of the next stage | barrier | read slice 0 of the next
  //                stage | multiply slice 3
  // so fragments are always requested one slice before the matrix instructions that use them, also
  // across the stage boundary.  The fragment reads are ordinary loads: the compiler counts them
  // (lgkmcnt) and waits for exactly the fragments an instruction needs.
  constexpr int S4 = BK / 16;
  static_assert(S4 == 4, "the schedule below is written for four K slices per stage");
  half8_t fa[2][TM], fb[2][TN];
  auto read_frags = [&](int buf, int slot, int bslot, int s4) {
    const unsigned char* pa = gemm_lds + slot * A_STRIDE + a_row + pos[s4];
    const unsigned char* pb = gemm_lds + bslot * B_STRIDE + b_row + pos[s4];
#pragma unroll
    for (int i = 0; i < TM; ++i) fa[buf][i] = *reinterpret_cast<const half8_t*>(pa + i * 32 * ROWB);
#pragma unroll
    for (int j = 0; j < TN; ++j) fb[buf][j] = *reinterpret_cast<const half8_t*>(pb + j * 32 * ROWB);
  };
  auto multiply = [&](int buf) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if constexpr (EP::BF16) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, fa[buf][i]),
                                                              __builtin_bit_cast(bf16x8_t, fb[buf][j]), acc[i][j], 0, 0, 0);
        } else {
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[buf][i], fb[buf][j], acc[i][j], 0, 0, 0);
        }
      }
    }
  };
  // one stage (lhs in ring slot `slot`, W tile `bslot`); FETCH: request batch `next` into slot
  // `fill`; MORE: another stage follows (slots `nslot`, `nbslot`), whose own requests are complete
  // once at most PEND younger ones are outstanding.  uint8 with MORE: between the first two slices
  // the codes of the next stage (ring slot nslot) become its fp16 tile nbslot.
  auto stage = [&](int slot, int bslot, auto fetch, int next, int fill, auto more, auto pend, int nslot, int nbslot,
                   int t) {
    constexpr bool FETCH = decltype(fetch)::value, MORE = decltype(more)::value;
    constexpr int PEND = decltype(pend)::value;
#pragma unroll
    for (int s4 = 0; s4 < 3; ++s4) {
      read_frags((s4 + 1) & 1, slot, bslot, s4 + 1);
      if constexpr (FETCH) {
#pragma unroll
        for (int idx = s4 * P / 3; idx < (s4 + 1) * P / 3; ++idx) issue_one(next, fill, idx);
      }
      __builtin_amdgcn_sched_barrier(0);
      multiply(s4 & 1);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (U8 && MORE) {
        if (s4 == 0) {
          dequantise(nslot, nbslot, t + 1);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    if constexpr (MORE) {
      // this wavefront's reads of the stage (and its writes of the next fp16 tile) are complete
      // before it lets the others overwrite the slot / read the tile
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      wait_vmcnt<PEND>();
      asm volatile("s_barrier" ::: "memory");
      read_frags(0, nslot, nbslot, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    multiply(1);
    __builtin_amdgcn_sched_barrier(0);
  };

  if constexpr (U8) {
    // codes and scales of stage 0 (batch -1, into slot 0 of their rings), then the first batches
#pragma unroll
    for (int idx = PA; idx < P; ++idx) issue_one(-1, NS - 1, idx);
#pragma unroll
    for (int s0 = 0; s0 < NS - 1; ++s0) {
      if (s0 < nt) issue(s0, s0);
    }
    if (nt > 1) {
      wait_vmcnt<(NS - 1) * P>();  // everything older than the batches: codes and scales of stage 0
    } else {
      wait_vmcnt<0>();
    }
    asm volatile("s_barrier" ::: "memory");
    dequantise(0, 0, 0);
  } else {
#pragma unroll
    for (int s0 = 0; s0 < NS - 1; ++s0) {
      if (s0 < nt) issue(s0, s0);
    }
  }
  // stage 0 has to be there before anything is read
  if (nt > 1) {
    wait_vmcnt<(NS - 2) * P>();  // with nt < NS - 1 fewer requests exist: the wait is merely stricter
  } else {
    wait_vmcnt<0>();
  }
  __syncthreads();  // also orders the fp16 tile written just above (uint8) before its first reads
  read_frags(0, 0, 0, 0);
  int slot = 0, fill = NS - 1;  // ring slots of stage t and of batch t + NS - 1
  auto next_of = [](int v) { return v + 1 == NS ? 0 : v + 1; };
  const int n_main = max(nt - (NS - 1), 0);
  for (int t = 0; t < n_main; ++t) {
    // after this stage's requests (batch t+NS-1), batches t+2 .. t+NS-1 may stay in flight when
    // batch t+1 must have landed
    stage(slot, U8 ? (t & 1) : slot, std::true_type{}, t + NS - 1, fill, std::true_type{},
          std::integral_constant<int, (NS - 2) * P>{}, next_of(slot), U8 ? ((t + 1) & 1) : next_of(slot), t);
    slot = next_of(slot);
    fill = next_of(fill);
  }
  // the last NS-1 stages: nothing left to request, so simply wait for everything
  for (int t = n_main; t < nt; ++t) {
    if (t + 1 < nt) {
      stage(slot, U8 ? (t & 1) : slot, std::false_type{}, 0, 0, std::true_type{}, std::integral_constant<int, 0>{},
            next_of(slot), U8 ? ((t + 1) & 1) : next_of(slot), t);
    } else {
      stage(slot, U8 ? (t & 1) : slot, std::false_type{}, 0, 0, std::false_type{}, std::integral_constant<int, 0>{}, 0, 0,
            t);
    }
    slot = next_of(slot);
  }
  __syncthreads();  // the last stage has been read by everybody: LDS is free for the partial sums

  if constexpr (KS == 2) {
    float* part = reinterpret_cast<float*>(gemm_lds);
    if (group == 1) {
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            part[(((w4 * TM + i) * TN + j) * 16 + v) * 64 + lane] = acc[i][j][v];
          }
        }
      }
    }
    __syncthreads();
    if (group == 0) {
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            acc[i][j][v] += part[(((w4 * TM + i) * TN + j) * 16 + v) * 64 + lane];
          }
        }
      }
    }
  }

  half_t* old_lds = reinterpret_cast<half_t*>(gemm_lds);
  if constexpr (OLD_PIECES) {
    if (old_by_pieces) {
      if constexpr (KS == 2) __syncthreads();  // the partial sums above have been read
#pragma unroll
      for (int j = 0; j < OC; ++j) {
        const int c = tid + j * THREADS;
        *reinterpret_cast<uint4_t*>(old_lds + (c / (BN / 8)) * OLD_LD + (c % (BN / 8)) * 8) = old_piece[j];
      }
      __syncthreads();
    }
  }
  if constexpr (EP::BF16) {
    static_assert(!U8, "bfloat16 operands are not quantised");
    if (group == 0) {
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int gm = m0 + wm + i * 32 + (v >> 2) * 8 + (lane >> 5) * 4 + (v & 3);
          if (gm >= M) continue;
          if constexpr (SPLIT) {  // the epilogue belongs to the launch that adds the splits
#pragma unroll
            for (int j = 0; j < TN; ++j) {
              const int gn = n0 + wn + j * 32 + (lane & 31);
              if (gn < N) part[((size_t)split * M + gm) * N + gn] = acc[i][j][v];
            }
          } else if constexpr (EP::GATED) {
            // 32 columns of gate rows, then the 32 of the up rows they belong to: one lane holds both
            static_assert(TN == 2, "a wavefront's columns are one gate / up pair of blocks");
            const int hc = (n0 + wn) / 2 + (lane & 31);
            if (n0 + wn < N) ep.store_gated(gm, hc, acc[i][0][v], acc[i][1][v]);
          } else {
#pragma unroll
            for (int j = 0; j < TN; ++j) {
              const int gn = n0 + wn + j * 32 + (lane & 31);
              if (gn < N) ep.store(gm, gn, acc[i][j][v]);
            }
          }
        }
      }
    }
    return;
  }
  // epilogue as in gemm_kernel (llama_cu.cu:208-215)
  if (group == 0) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int gn = n0 + wn + j * 32 + (lane & 31);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int lm = wm + i * 32 + (v >> 2) * 8 + (lane >> 5) * 4 + (v & 3);
          const int gm = m0 + lm;
          if (gm < M && gn < N) {
            if constexpr (SPLIT) {
              part[((size_t)split * M + gm) * N + gn] = acc[i][j][v];
            } else {
              half_t* p = out + (size_t)gm * N + gn;
              float val = acc[i][j][v];
              if (beta != 0.0f) {
                const half_t before = old_by_pieces ? old_lds[lm * OLD_LD + wn + j * 32 + (lane & 31)] : *p;
                val = fmaf(beta, (float)before, val);
              }
              *p = round_f16(val);
            }
          }
        }
      }
    }
  }
}

// out_g[m][n] = fp16(sum over splits, in split order, of part[g][s][m][n] + beta * out_g[m][n]); blockIdx.y = g
__global__ __launch_bounds__(256) void splitk_reduce_kernel(half_t* out0, half_t* out1, half_t* out2,
                                                            const float* __restrict__ part, size_t mn, int splits,
                                                            float beta) {
  const int g = blockIdx.y;
  half_t* out = g == 0 ? out0 : (g == 1 ? out1 : out2);
  part += (size_t)g * splits * mn;
  const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= mn) {
    return;
  }
  if (i + 4 <= mn && mn % 4 == 0) {
    float4 sum = *reinterpret_cast<const float4*>(part + i);
    for (int s = 1; s < splits; ++s) {
      const float4 v = *reinterpret_cast<const float4*>(part + (size_t)s * mn + i);
      sum.x += v.x;
      sum.y += v.y;
      sum.z += v.z;
      sum.w += v.w;
    }
    const float v4[4] = {sum.x, sum.y, sum.z, sum.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float val = v4[e];
      if (beta != 0.0f) {
        val = fmaf(beta, (float)out[i + e], val);
      }
      out[i + e] = round_f16(val);
    }
    return;
  }
  for (size_t j = i; j < min(i + 4, mn); ++j) {
    float val = part[j];
    for (int s = 1; s < splits; ++s) {
      val += part[(size_t)s * mn + j];
    }
    if (beta != 0.0f) {
      val = fmaf(beta, (float)out[j], val);
    }
    out[j] = round_f16(val);
  }
}

// the arguments of one launch: matrix 0 and, for fused launches, up to two more of the same shape
struct operands_t {
  half_t* out;
  const void* W;
  const half_t* S;
  more_matrices_t more;
  int n_mats;
};

inline operands_t single_matrix(half_t* out, const void* W, const half_t* S) {
  return operands_t{out, W, S, more_matrices_t{{nullptr, nullptr}, {nullptr, nullptr}, {nullptr, nullptr}, 0}, 1};
}

inline operands_t last_matrix(operands_t op) {
  return op.n_mats == 1 ? op : single_matrix(op.more.out[op.n_mats - 2], op.more.W[op.n_mats - 2], op.more.S[op.n_mats - 2]);
}

template <int BM, int BN, int WM, int WN, int KS, int NS, bool U8>
int launch_dl(operands_t op, const half_t* A, int M, int K, int N, int block, float beta, hipStream_t st) {
  constexpr int ROWB = BK * KS * 2;
  constexpr int DCH = U8 ? BN * (BK * KS / 16) / (64 * WM * WN * KS) : 0;  // scale dwords per thread and stage
  constexpr size_t lds = (size_t)NS * BM * ROWB + (size_t)(U8 ? 2 : NS) * BN * ROWB +
                         (U8 ? (size_t)NS * (BN * BK * KS + 64 * WM * WN * KS * 4 * DCH) : 0);
  static_assert(lds <= 160 * 1024, "rings do not fit LDS");
  static_assert(KS == 1 || lds >= (size_t)BM * BN * 4 / 2, "LDS must hold one group's accumulators");
  const int tiles_m = (M + BM - 1) / BM, tiles_n_per = (N + BN - 1) / BN, tiles_n = tiles_n_per * op.n_mats;
  op.more.tiles_n_per = op.n_mats > 1 ? tiles_n_per : 0;
  auto kernel = gemm_dl_kernel<BM, BN, WM, WN, KS, NS, U8>;
  if constexpr (lds > 64 * 1024) {
    static bool raised[16] = {};  // per device, once
    int dev = 0;
    LCU_HIP(hipGetDevice(&dev));
    if (!raised[dev & 15]) {
      LCU_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
      raised[dev & 15] = true;
    }
  }
  kernel<<<tiles_m * tiles_n, 64 * WM * WN * KS, lds, st>>>(op.out, A, op.W, op.S, M, K, N, block, beta, tiles_m,
                                                            tiles_n, nullptr, 1, op.more, f16_epilogue{});
  LCU_LAUNCH_CHECK();
  return LCU_OK;
}

// 64 << shift = block, -1 for blocks that gemm_tile_kernel does not take (0: no codes)
inline int block_shift(int block) {
  for (int shift = 0; shift < 16; ++shift) {
    if (block == 64 << shift) return shift;
  }
  return -1;
}

// A launch of gemm_tile_kernel; splits > 1: the K stages of every tile dealt to that many workgroups, fp32 sums to part.
template <int BM, int BN, int WM, int WN, int NA, int NB, bool U8, bool SPLIT, class EP, int CHAINS = 1>
int launch_tile(EP const& ep, operands_t op, const void* A, int M, int K, int N, int block, float beta, hipStream_t st, int splits = 1,
                float* part = nullptr, columns_t which = {}, int step = 1) {
  using shape = tile_shape<BM, BN, WM, WN, NA, NB, U8, SPLIT, EP>;
  const int tiles_m = (M + BM - 1) / BM;
  if (which.from > 0) op = last_matrix(op);
  const int tiles_n_per = (N - which.from + BN - 1) / BN, tiles_n = which.tiles > 0 ? which.tiles : tiles_n_per * op.n_mats;
  op.more.tiles_n_per = op.n_mats > 1 ? tiles_n_per : 0;
  auto kernel = gemm_tile_kernel<BM, BN, WM, WN, NA, NB, U8, SPLIT, EP, CHAINS>;
  static bool raised[16] = {};  // per device, once
  int dev = 0;
  LCU_HIP(hipGetDevice(&dev));
  if (!raised[dev & 15]) {
    LCU_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, shape::LDS));
    raised[dev & 15] = true;
  }
  kernel<<<tiles_m * tiles_n * splits, 64 * WM * WN, shape::LDS, st>>>(op.out, (const half_t*)A, op.W, op.S, block_shift(block), M, K, N, beta,
                                                                       tiles_m, tiles_n, which.from, part, splits, step, op.more, ep);
  LCU_LAUNCH_CHECK();
  return LCU_OK;
}

// tiles of 256 rows
template <bool U8, class EP>
int launch_columns(EP const& ep, operands_t op, const void* A, int M, int K, int N, int block, float beta, hipStream_t st, int columns,
                   columns_t which) {
  if constexpr (U8) {
    if (columns == 256) return launch_tile<256, 256, 1, 4, 3, 3, true, false>(ep, op, A, M, K, N, block, beta, st, 1, nullptr, which);
    if (columns == 192) return launch_tile<256, 192, 1, 4, 3, 3, true, false>(ep, op, A, M, K, N, block, beta, st, 1, nullptr, which);
    return launch_tile<256, 128, 1, 4, 3, 3, true, false>(ep, op, A, M, K, N, block, beta, st, 1, nullptr, which);
  } else {
    if (columns == 256) return launch_tile<256, 256, 2, 2, 2, 3, false, false>(ep, op, A, M, K, N, 0, beta, st, 1, nullptr, which);
    if (columns == 192) {
      return launch_tile<256, 192, EP::GATED ? 4 : 2, EP::GATED ? 1 : 2, 2, 4, false, false>(ep, op, A, M, K, N, 0, beta, st, 1, nullptr, which);
    }
    return launch_tile<256, 128, 4, 2, 3, 3, false, false>(ep, op, A, M, K, N, 0, beta, st, 1, nullptr, which);
  }
}

// the columns of the last matrix that whole rounds of large tiles leave
template <bool U8, class EP>
int launch_rest(EP const& ep, large_tiles_t const& plan, operands_t op, const void* A, int M, int K, int N, int block, float beta, hipStream_t st) {
  if (plan.rest_rows == 256) return launch_columns<U8>(ep, op, A, M, K, N, block, beta, st, plan.rest_columns, plan.rest);
  return launch_tile<128, 128, U8 ? 1 : 2, U8 ? 4 : 2, 4, 4, U8, false>(ep, op, A, M, K, N, block, beta, st, 1, nullptr, plan.rest);
}

template <bool U8, class EP>
int launch_large(EP const& ep, operands_t op, const void* A, int M, int K, int N, int block, float beta, hipStream_t st) {
  device_state* ds = current_device_state();
  bool ragged = N % 8 != 0;
  if constexpr (EP::BF16) ragged = ep.ldo % 8 != 0;
  const product_type type = U8 ? product_type::u8 : !EP::BF16 ? product_type::f16 : EP::GATED ? product_type::bf16_gated : product_type::bf16;
  const large_tiles_t plan = plan_large(type, M, K, N, op.n_mats, ds && ds->compute_units > 0 ? ds->compute_units : 256, ragged);
  if (M <= 128) {
    if constexpr (U8) {
      if (plan.columns == 256) return launch_tile<128, 256, 1, 4, 3, 3, true, false>(ep, op, A, M, K, N, block, beta, st);
      return launch_tile<128, 128, 1, 4, 4, 4, true, false>(ep, op, A, M, K, N, block, beta, st);
    } else {
      if (plan.columns == 256) return launch_tile<128, 256, 2, 4, 3, 3, false, false>(ep, op, A, M, K, N, 0, beta, st);
      return launch_tile<128, 128, 2, 2, 4, 4, false, false>(ep, op, A, M, K, N, 0, beta, st);
    }
  }
  const int rc = launch_columns<U8>(ep, op, A, M, K, N, block, beta, st, plan.columns, plan.first);
  if (rc != LCU_OK || plan.rest.from == 0) return rc;
  if constexpr (EP::ROTARY) {  // columns of the last matrix only, which are values
    LCU_REQUIRE(ep.matrices < op.n_mats, "large tiles: the last of %d matrices is not rotated", op.n_mats);
    return launch_rest<U8>(f16_epilogue{}, plan, op, A, M, K, N, block, beta, st);
  } else {
    return launch_rest<U8>(ep, plan, op, A, M, K, N, block, beta, st);
  }
}

template <bool U8>
size_t weight_bytes(const operands_t& op, int K, int N) {
  return (size_t)N * K * (U8 ? 1 : 2) * op.n_mats;
}

// whether an output lies over lhs
inline bool over_lhs(const operands_t& op, const void* A, int M, int K, int N) {
  for (const void* o : {(const void*)op.out, (const void*)op.more.out[0], (const void*)op.more.out[1]}) {
    if (o != nullptr && overlap(o, (size_t)M * N * 2, A, (size_t)M * K * 2)) return true;
  }
  return false;
}
template <bool GATED>
bool over_lhs(linear_epilogue<false, GATED> const& ep, const void* A, int M, int K, int N) {
  const size_t lhs_bytes = (size_t)M * K * 2, row = GATED ? N / 2 : N;
  return overlap(ep.out, ((size_t)(M - 1) * ep.ldo + row) * (ep.out_f32 ? 4 : 2), A, lhs_bytes) ||
         (ep.tail && overlap(ep.tail, ((size_t)(M - 1) * ep.ld_tail + (N - ep.tail_from)) * 4, A, lhs_bytes));
}

// where a split-K launch left its partial sums: part[matrix][split][M][N] fp32
struct partial_sums_t {
  const float* part;
  int splits;
};

// BM x BN tiles of WM x WN wavefronts, the K stages of every tile dealt to `splits` workgroups
// (gemm_dl_kernel<.., SPLIT = true>), fp32 partial sums in the stream's workspace, then
// splitk_reduce_kernel -- or the caller's own kernel when `leave` is given.
template <int BM, int BN, int WM, int WN, bool U8>
int launch_split(operands_t op, const half_t* A, int M, int K, int N, int block, float beta, hipStream_t st, int splits,
                 float* part, partial_sums_t* leave = nullptr) {
  constexpr int KS = 1, NS = 3;
  constexpr int ROWB = BK * KS * 2;
  constexpr int DCH = U8 ? BN * (BK * KS / 16) / (64 * WM * WN * KS) : 0;
  constexpr size_t lds = (size_t)NS * BM * ROWB + (size_t)(U8 ? 2 : NS) * BN * ROWB +
                         (U8 ? (size_t)NS * (BN * BK * KS + 64 * WM * WN * KS * 4 * DCH) : 0);
  static_assert(lds <= 160 * 1024, "LDS");
  const int tiles_m = (M + BM - 1) / BM, tiles_n_per = (N + BN - 1) / BN, tiles_n = tiles_n_per * op.n_mats;
  op.more.tiles_n_per = op.n_mats > 1 ? tiles_n_per : 0;
  const size_t mn = (size_t)M * N;
  auto kernel = gemm_dl_kernel<BM, BN, WM, WN, KS, NS, U8, true>;
  if constexpr (lds > 64 * 1024) {
    static bool raised[16] = {};  // per device, once
    int dev = 0;
    LCU_HIP(hipGetDevice(&dev));
    if (!raised[dev & 15]) {
      LCU_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
      raised[dev & 15] = true;
    }
  }
  kernel<<<tiles_m * tiles_n * splits, 64 * WM * WN * KS, lds, st>>>(op.out, A, op.W, op.S, M, K, N, block, beta, tiles_m,
                                                                     tiles_n, part, splits, op.more, f16_epilogue{});
  LCU_LAUNCH_CHECK();
  if (leave) {  // the caller's own kernel adds the partial sums up (fused with what follows the product)
    leave->part = part;
    leave->splits = splits;
  } else {
    splitk_reduce_kernel<<<dim3((unsigned)((mn + 1023) / 1024), op.n_mats), 256, 0, st>>>(
        op.out, op.more.out[0], op.more.out[1], part, mn, splits, beta);
    LCU_LAUNCH_CHECK();
  }
  return LCU_OK;
}

// Workgroups that have every split of their columns: wavefronts of one (0: more than a round of them, too few wavefronts for the splits, or no room for lhs)
// and workgroups in all.  As few sixteens of columns as leave one round, four wavefronts at least.
struct stream_join_t {
  int waves, tiles;
};
inline stream_join_t plan_stream_join(int M, int K, int N, int n_mats, int joined, int splits, long cus, bool u8) {
  const int per = splits * joined;
  const long sixteens = (long)(N + 15) / 16 * (n_mats / joined);
  const int row_tiles = M <= 16 ? 1 : M <= 32 ? 2 : 4;
  if ((size_t)M * K * 2 > (size_t)STREAM_LDS) return {0, 0};
  for (int each = 1; each * per <= stream_max_waves(u8); ++each) {
    const int waves = each * per;
    const long tiles = (sixteens + each - 1) / each;
    if (stream_joined_lhs(waves, row_tiles, M, K) + waves * STREAM_RING * stream_unit(u8) > STREAM_LDS) break;
    if (tiles <= cus && waves >= 4) return {waves, (int)tiles};
  }
  return {0, 0};
}

template <int TM, bool U8, bool BF16, bool ONCE>
int launch_stream_rows(operands_t op, const void* A, int M, int K, int N, int block, hipStream_t st, int splits, float* part, long cus) {
  long rounds = 1;
  const int waves = stream_waves(N, op.n_mats, splits, cus, stream_max_waves(U8), &rounds), tiles = ((N + 15) / 16 + waves - 1) / waves;
  op.more.tiles_n_per = op.n_mats;
  auto kernel = gemm_stream_kernel<TM, U8, BF16, ONCE>;
  static bool raised[16] = {};  // per device, once
  int dev = 0;
  LCU_HIP(hipGetDevice(&dev));
  if (!raised[dev & 15]) {
    LCU_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, stream_lds(U8, stream_max_waves(U8))));
    raised[dev & 15] = true;
  }
  const int kc = stream_chunk(M, K / BK, splits);
  kernel<<<tiles * op.n_mats * splits, 64 * waves, stream_lds(U8, waves), st>>>((const half_t*)A, op.W, op.S, block_shift(block), M, K, N, tiles,
                                                                                kc, part, splits, op.more, separate_sums{});
  LCU_LAUNCH_CHECK();
  return LCU_OK;
}

// 1 .. 64 rows, K a multiple of 64: fp32 sums of every split's K stages to part[matrix][split][M][N]
template <bool U8, bool BF16>
int launch_stream(operands_t op, const void* A, int M, int K, int N, int block, hipStream_t st, int splits, float* part, long cus, bool memory) {
  const auto rows = [&](auto once) {
    constexpr bool ONCE = decltype(once)::value;
    if (M <= 16) return launch_stream_rows<1, U8, BF16, ONCE>(op, A, M, K, N, block, st, splits, part, cus);
    if (M <= 32) return launch_stream_rows<2, U8, BF16, ONCE>(op, A, M, K, N, block, st, splits, part, cus);
    return launch_stream_rows<4, U8, BF16, ONCE>(op, A, M, K, N, block, st, splits, part, cus);
  };
  return stream_once(memory, weight_bytes<U8>(op, K, N)) ? rows(std::true_type{}) : rows(std::false_type{});
}

// The direct-to-LDS kernels fetch a thread's fp16 scale as the aligned 4-byte word that holds it:
// every scale array must then start on a 4-byte boundary and hold an even number of scales (the
// word of the last scale must not reach past the array).  Otherwise the register-staged kernel runs.
template <bool U8>
bool scale_words_ok(const operands_t& op, int K, int N, int block) {
  if constexpr (!U8) {
    return true;
  } else {
    if (((size_t)N * (size_t)(K / block)) % 2 != 0) {
      return false;
    }
    const half_t* all[3] = {op.S, op.n_mats > 1 ? op.more.S[0] : nullptr, op.n_mats > 2 ? op.more.S[1] : nullptr};
    for (const half_t* p : all) {
      if (p != nullptr && (reinterpret_cast<uintptr_t>(p) & 3) != 0) {
        return false;
      }
    }
    return true;
  }
}

template <int TM, bool U8, bool BF16, bool ONCE, class JOIN>
int launch_joined_rows(JOIN const& join, operands_t op, const half_t* A, int M, int K, int N, int block, hipStream_t st, int splits, int waves, int tiles) {
  auto kernel = gemm_stream_kernel<TM, U8, BF16, ONCE, JOIN>;
  static bool raised[16] = {};  // per device, once
  int dev = 0;
  LCU_HIP(hipGetDevice(&dev));
  if (!raised[dev & 15]) {
    LCU_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, STREAM_LDS));
    raised[dev & 15] = true;
  }
  op.more.tiles_n_per = op.n_mats;
  const int lds = stream_joined_lhs(waves, TM, M, K) + waves * STREAM_RING * stream_unit(U8);
  kernel<<<tiles, 64 * waves, lds, st>>>(A, op.W, op.S, block_shift(block), M, K, N, tiles, K, nullptr,
                                                                                         splits, op.more, join);
  LCU_LAUNCH_CHECK();
  return LCU_OK;
}

template <bool U8, bool BF16, class JOIN>
int launch_joined_shape(JOIN const& join, operands_t op, const half_t* A, int M, int K, int N, int block, hipStream_t st, int splits, stream_join_t shape,
                        bool memory) {
  const auto rows = [&](auto once) {
    constexpr bool ONCE = decltype(once)::value;
    if (M <= 16) return launch_joined_rows<1, U8, BF16, ONCE>(join, op, A, M, K, N, block, st, splits, shape.waves, shape.tiles);
    if (M <= 32) return launch_joined_rows<2, U8, BF16, ONCE>(join, op, A, M, K, N, block, st, splits, shape.waves, shape.tiles);
    return launch_joined_rows<4, U8, BF16, ONCE>(join, op, A, M, K, N, block, st, splits, shape.waves, shape.tiles);
  };
  return stream_once(memory, weight_bytes<U8>(op, K, N)) ? rows(std::true_type{}) : rows(std::false_type{});
}

// A product of few rows and what follows it in one launch, with the splits of plan_skinny.  *done = false, with nothing launched, where lhs does not fit
// LDS whole, the workgroups would take a second round, or an output (an operand's, or `out`) lies over lhs, which other workgroups still read.
template <bool U8, class JOIN>
int launch_joined(JOIN const& join, operands_t op, const half_t* A, int M, int K, int N, int block, hipStream_t st, const void* out, bool* done) {
  *done = false;
  const device_state* ds = current_device_state();
  const workspace_t ws = workspace_for(st);
  if (ds == nullptr || ws.ptr == nullptr || K % 128 != 0 || N % 2 != 0 || M < 2 || M > 64 ||
      (U8 && block_shift(block) < 0) || !scale_words_ok<U8>(op, K, N, block)) {
    return LCU_OK;
  }
  if (over_lhs(op, A, M, K, N) || (out != nullptr && overlap(out, (size_t)M * N * 2, A, (size_t)M * K * 2))) return LCU_OK;
  const skinny_plan_t plan = plan_skinny(M <= 32 || U8 ? 32 : 64, M, K, N, op.n_mats, ds->compute_units, ws.bytes);
  if (plan.splits == 0) return LCU_OK;
  const stream_join_t shape = plan_stream_join(M, K, N, op.n_mats, JOIN::MATRICES, plan.splits, ds->compute_units, U8);
  if (shape.waves == 0) return LCU_OK;
  const int rc = launch_joined_shape<U8, false>(join, op, A, M, K, N, block, st, plan.splits, shape, from_memory(ws.weights, weight_bytes<U8>(op, K, N)));
  *done = rc == LCU_OK;
  return rc;
}

// what splitk_reduce_kernel makes of the sums
struct f16_join {
  static constexpr bool JOINED = true, GATED = false;
  static constexpr int MATRICES = 1;
  half_t* out[3];
  int N;
  float beta;
  __device__ __forceinline__ void operator()(int matrix, int row, int c, const float2 (&x)[1]) const {
    half_t* to = (matrix == 0 ? out[0] : matrix == 1 ? out[1] : out[2]) + (size_t)row * N + c;
    to[0] = round_f16(beta != 0.0f ? fmaf(beta, (float)to[0], x[0].x) : x[0].x);
    to[1] = round_f16(beta != 0.0f ? fmaf(beta, (float)to[1], x[0].y) : x[0].y);
  }
};

// Few rows (2 .. 64: short prompts, where the reference takes its 16-row tile, llama_cu.cu:1481-1484):
// the K stages split as BM x 128 tiles would need to give every compute unit one workgroup; gemm_stream_kernel
// walks the splits, in one launch with what follows (launch_joined) or for another to add up, or such tiles with four
// wavefronts do (`streams`; blocks of codes other than 64 << n).
// Returns LCU_OK with *done = false when the shape does not suit it.
template <int BM, bool U8>
int launch_skinny(operands_t op, const half_t* A, int M, int K, int N, int block, float beta, hipStream_t st,
                  bool* done, partial_sums_t* leave = nullptr) {
  // a ring of six stages and 128-wide stages with eight wavefronts measured no faster
  constexpr int BN = 128;
  *done = false;
  device_state* ds = current_device_state();
  const workspace_t ws = workspace_for(st);
  if (ds == nullptr || ws.ptr == nullptr) {
    return LCU_OK;
  }
  int rc;
  if (leave == nullptr) {
    rc = launch_joined<U8>(f16_join{{op.out, op.more.out[0], op.more.out[1]}, N, beta}, op, A, M, K, N, block, st, nullptr, done);
    if (rc != LCU_OK || *done) return rc;
  }
  const skinny_plan_t plan = plan_skinny(BM, M, K, N, op.n_mats, ds->compute_units, ws.bytes);
  if (plan.splits == 0) return LCU_OK;
  const int splits = plan.splits;
  const size_t mn = (size_t)M * N;
  const bool memory = from_memory(ws.weights, weight_bytes<U8>(op, K, N));
  if ((U8 && block_shift(block) < 0) || !streams(M, N, op.n_mats, splits, K / BK, plan.tiles, ds->compute_units, U8, false, memory)) {
    rc = launch_split<BM, BN, 1, 4, U8>(op, A, M, K, N, block, beta, st, splits, (float*)ws.ptr, leave);
    *done = rc == LCU_OK;
    return rc;
  }
  rc = launch_stream<U8, false>(op, A, M, K, N, block, st, splits, (float*)ws.ptr, ds->compute_units, memory);
  if (rc == LCU_OK && leave) {
    leave->part = (float*)ws.ptr;
    leave->splits = splits;
  } else if (rc == LCU_OK) {
    splitk_reduce_kernel<<<dim3((unsigned)((mn + 1023) / 1024), op.n_mats), 256, 0, st>>>(op.out, op.more.out[0], op.more.out[1],
                                                                                          (const float*)ws.ptr, mn, splits, beta);
    LCU_LAUNCH_CHECK();
  }
  *done = rc == LCU_OK;
  return rc;
}

// Sums of every split to part, in tiles of 256x128 (128x128 up to 128 rows or where `small`), or of fewer where these leave compute units idle
// (plan_tile_size).  us, those / so: fp16 66x11008x4096 33.5 / 27.2, 128 rows 38.8 / 32.8, 66x6656x6656 35.7 / 29.4, 200x5632x2048 42.1 / 19.1; uint8
// 36.6 / 27.5, 41.9 / 34.2, 40.9 / 28.2, 49.0 / 21.7.
template <bool U8>
int launch_partial(operands_t op, const half_t* A, int M, int K, int N, int block, hipStream_t st, int splits, float* part, bool small, int step, long cus) {
  const tile_size_t tile = plan_tile_size(M, N, splits * op.n_mats, small || M <= 128 ? tile_size_t{128, 128} : tile_size_t{256, 128}, false, cus);
  const f16_epilogue ep{};
  if (tile.rows == 64) return launch_tile<64, 64, 1, 4, 4, 4, U8, true>(ep, op, A, M, K, N, block, 0.0f, st, splits, part, {}, step);
  if (tile.columns == 64) return launch_tile<128, 64, U8 ? 1 : 2, U8 ? 4 : 2, 4, 4, U8, true>(ep, op, A, M, K, N, block, 0.0f, st, splits, part, {}, step);
  if (tile.rows == 128) return launch_tile<128, 128, U8 ? 1 : 2, U8 ? 4 : 2, 4, 4, U8, true>(ep, op, A, M, K, N, block, 0.0f, st, splits, part, {}, step);
  return launch_tile<256, 128, U8 ? 1 : 4, U8 ? 4 : 2, 3, 3, U8, true>(ep, op, A, M, K, N, block, 0.0f, st, splits, part, {}, step);
}

template <bool U8>
int launch_large_split(operands_t op, const half_t* A, int M, int K, int N, int block, float beta, hipStream_t st, int splits, float* part, long cus) {
  const int rc = launch_partial<U8>(op, A, M, K, N, block, st, splits, part, false, 1, cus);
  if (rc != LCU_OK) return rc;
  const size_t mn = (size_t)M * N;
  splitk_reduce_kernel<<<dim3((unsigned)((mn + 1023) / 1024), op.n_mats), 256, 0, st>>>(op.out, op.more.out[0], op.more.out[1], part, mn,
                                                                                        splits, beta);
  LCU_LAUNCH_CHECK();
  return LCU_OK;
}

// the split-K product of a few rows with its partial sums left in the workspace; *done = false when
// the shape does not take that path (nothing has been launched then)
template <bool U8>
int skinny_partial(operands_t op, const half_t* A, int M, int K, int N, int block, hipStream_t st, bool* done,
                   partial_sums_t* res) {
  *done = false;
  if (K % 128 != 0 || M > 64 || M < 1 || !scale_words_ok<U8>(op, K, N, block)) {
    return LCU_OK;
  }
  if constexpr (U8) {
    return launch_skinny<32, true>(op, A, M, K, N, block, 0.0f, st, done, res);
  } else {
    return M <= 32 ? launch_skinny<32, false>(op, A, M, K, N, block, 0.0f, st, done, res)
                   : launch_skinny<64, false>(op, A, M, K, N, block, 0.0f, st, done, res);
  }
}

// the same for more than 64 rows of one matrix (plan_left_sums)
template <bool U8>
int many_rows_partial(operands_t op, const half_t* A, int M, int K, int N, int block, hipStream_t st, bool* done, partial_sums_t* res) {
  *done = false;
  device_state* ds = current_device_state();
  const workspace_t ws = workspace_for(st);
  if (K % 128 != 0 || M <= 64 || ds == nullptr || ws.ptr == nullptr || !scale_words_ok<U8>(op, K, N, block) || (U8 && block_shift(block) < 0) ||
      (size_t)M * K * 2 >= (size_t)1 << 32 || (size_t)N * K * (U8 ? 1 : 2) >= (size_t)1 << 32) {
    return LCU_OK;
  }
  const long cus = ds->compute_units > 0 ? ds->compute_units : 256;
  const left_sums_t left = plan_left_sums(U8, M, K, N, cus, ws.bytes, ws.owned);
  if (left.splits == 0) return LCU_OK;
  const int rc = launch_partial<U8>(op, A, M, K, N, block, st, left.splits, (float*)ws.ptr, left.step == 2, left.step, cus);
  res->part = (float*)ws.ptr;
  res->splits = left.splits;
  *done = rc == LCU_OK;
  return rc;
}

// ---- kernels that add the partial sums up and go on with what follows the product in a batched
// decode step (llama_cu.cu:1144-1156, 1174-1176, 1180-1185), one row per sequence ----

// In split order, four splits asked for at a time: with a runtime count the compiler waits for each before the next.  A last one by itself, as
// with two splits (46x512x5632 twice in uint8, product and SiLU: asked for four times over 12.7 us, once 10.9).
__device__ __forceinline__ float2 sum_pair(const float* __restrict__ part, size_t at, size_t mn, int splits) {
  float2 v = *reinterpret_cast<const float2*>(part + at);
  for (int s = 1; s < splits; s += 4) {
    if (s + 1 == splits) {
      const float2 w = *reinterpret_cast<const float2*>(part + (size_t)s * mn + at);
      v.x += w.x;
      v.y += w.y;
      break;
    }
    float2 w[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) w[u] = *reinterpret_cast<const float2*>(part + (size_t)min(s + u, splits - 1) * mn + at);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (s + u < splits) {
        v.x += w[u].x;
        v.y += w[u].y;
      }
    }
  }
  return v;
}

// the rotary of a pair whose products are rounded to fp16 before it reads them (1144-1153)
__device__ __forceinline__ half2_t rotated_pair(float2 x, float2 cs) {
  const float real = (float)round_f16(x.x), imag = (float)round_f16(x.y);
  half2_t w;
  w.x = round_f16(fmaf(real, cs.x, -(imag * cs.y)));
  w.y = round_f16(fmaf(real, cs.y, imag * cs.x));
  return w;
}

// Wq, Wk, Wv products -> fp16 -> rotary of q (to q_out) and k.  Sequences: at pos[b], rotated k and v into row
// pos[b] of sequence b's caches (what splitk_reduce_kernel + rope_store_batch_kernel do).  A prompt: at first + row, into the rows of k_out, v_out.
struct sequence_rows {
  half_t* const* __restrict__ k_ptrs;
  half_t* const* __restrict__ v_ptrs;
  const int* __restrict__ pos_dev;
  int max_pos;
  __device__ __forceinline__ int position(int b) const { return min(max(pos_dev[b], 0), max_pos); }
  __device__ __forceinline__ half_t* k(int b, int pos, int dim) const { return k_ptrs[b] + (size_t)pos * dim; }
  __device__ __forceinline__ half_t* v(int b, int pos, int dim) const { return v_ptrs[b] + (size_t)pos * dim; }
};
struct prompt_rows {
  half_t* k_out;
  half_t* v_out;
  int first;
  __device__ __forceinline__ int position(int row) const { return first + row; }
  __device__ __forceinline__ half_t* k(int row, int, int dim) const { return k_out + (size_t)row * dim; }
  __device__ __forceinline__ half_t* v(int row, int, int dim) const { return v_out + (size_t)row * dim; }
};
template <class ROWS>
__global__ __launch_bounds__(256) void reduce_rope_store_kernel(half_t* __restrict__ q_out, const float* __restrict__ part, int splits, int n_seq,
                                                                int dim, ROWS rows, int head_dim, const float2* __restrict__ table) {
  const int pair = blockIdx.x * 256 + threadIdx.x;
  const int b = blockIdx.y;
  if (pair * 2 >= dim) return;
  const int c = pair * 2;
  const size_t mn = (size_t)n_seq * dim, at = (size_t)b * dim + c;
  const int pos = rows.position(b);
  const float2 cs = table[(size_t)pos * (head_dim / 2) + (c % head_dim) / 2];
  const float2 qf = sum_pair(part, at, mn, splits);
  const float2 kf = sum_pair(part + (size_t)splits * mn, at, mn, splits);
  const float2 vf = sum_pair(part + (size_t)2 * splits * mn, at, mn, splits);
  *reinterpret_cast<half2_t*>(q_out + at) = rotated_pair(qf, cs);
  *reinterpret_cast<half2_t*>(rows.k(b, pos, dim) + c) = rotated_pair(kf, cs);
  *reinterpret_cast<half2_t*>(rows.v(b, pos, dim) + c) = half2_t{round_f16(vf.x), round_f16(vf.y)};
}

// the same, two products and SiLU, and the bare sums, where the product's workgroups have all the splits of their columns (gemm_stream_kernel)
template <class ROWS>
struct rope_join {
  static constexpr bool JOINED = true, GATED = false;
  static constexpr int MATRICES = 1;
  half_t* q_out;
  ROWS rows;
  const float2* table;
  int dim, head_dim;
  __device__ __forceinline__ void operator()(int matrix, int row, int c, const float2 (&x)[1]) const {
    const int pos = rows.position(row);
    const float2 cs = table[(size_t)pos * (head_dim / 2) + (c % head_dim) / 2];
    half_t* to = (matrix == 0 ? q_out + (size_t)row * dim : matrix == 1 ? rows.k(row, pos, dim) : rows.v(row, pos, dim)) + c;
    *reinterpret_cast<half2_t*>(to) = matrix < 2 ? rotated_pair(x[0], cs) : half2_t{round_f16(x[0].x), round_f16(x[0].y)};
  }
};
struct silu_join {
  static constexpr bool JOINED = true, GATED = false;
  static constexpr int MATRICES = 2;
  half_t* out;
  int ffn;
  __device__ __forceinline__ void operator()(int, int row, int c, const float2 (&x)[2]) const {
    half2_t w;
    w.x = silu_mul(round_f16(x[0].x), round_f16(x[1].x));
    w.y = silu_mul(round_f16(x[0].y), round_f16(x[1].y));
    *reinterpret_cast<half2_t*>(out + (size_t)row * ffn + c) = w;
  }
};

struct sum_join {
  static constexpr bool JOINED = true, GATED = false;
  static constexpr int MATRICES = 1;
  float* part;
  int N;
  __device__ __forceinline__ void operator()(int, int row, int c, const float2 (&x)[1]) const {
    *reinterpret_cast<float2*>(part + (size_t)row * N + c) = x[0];
  }
};

// W1, W3 products -> fp16 each -> fp16(silu(w1) * w3)  (1180-1183, 533-539)
__global__ __launch_bounds__(256) void reduce_silu_kernel(half_t* __restrict__ out, const float* __restrict__ part,
                                                          int splits, size_t mn) {
  const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 2;
  if (i >= mn) return;
  const float2 a = sum_pair(part, i, mn, splits);
  const float2 g = sum_pair(part + (size_t)splits * mn, i, mn, splits);
  half2_t w;
  w.x = silu_mul(round_f16(a.x), round_f16(g.x));
  w.y = silu_mul(round_f16(a.y), round_f16(g.y));
  *reinterpret_cast<half2_t*>(out + i) = w;
}

// x += product (one rounding of the fp32 sum, 1174 / 1185), then rms_norm of the new row with the
// next norm's weights (1176 / 1129 of the next layer / 1191).  One 1024-thread workgroup per row
// (up to 8192 columns: four pairs per thread, every partial sum requested before the first is
// used -- the launch is a handful of workgroups and nothing but latency); the norm as in
// rmsnorm_kernel, its sum of squares taken by the first 256 threads in the reference's association.
// 8 rows of 4096, eight splits: 7.4 us with a wait per split, 6.0 with four asked for at a time; 512 rows, four splits 9.1 (the sums' 46 MB),
// where the sum and the norm took 9.5 and 5.5 in launches of their own.
constexpr int RN_THREADS = 1024, RN_PAIRS = 4;
template <int PAIRS>
__global__ __launch_bounds__(RN_THREADS) void reduce_residual_norm_kernel(half_t* __restrict__ x,
                                                                          half_t* __restrict__ norm_out,
                                                                          const float* __restrict__ part, int splits,
                                                                          int n_seq, int cols,
                                                                          const half_t* __restrict__ norm_w, float eps) {
  extern __shared__ half_t row_lds[];
  __shared__ float red[8];
  const int b = blockIdx.x, tid = threadIdx.x;
  const size_t mn = (size_t)n_seq * cols;
  half_t* xr = x + (size_t)b * cols;
  float2 acc[PAIRS];
  half2_t old[PAIRS], wv[PAIRS];
#pragma unroll
  for (int j = 0; j < PAIRS; ++j) {
    const int c = min((tid + j * RN_THREADS) * 2, cols - 2);
    acc[j] = *reinterpret_cast<const float2*>(part + (size_t)b * cols + c);
    old[j] = *reinterpret_cast<const half2_t*>(xr + c);
    wv[j] = *reinterpret_cast<const half2_t*>(norm_w + c);
  }
  for (int s = 1; s < splits; s += 4) {
    float2 w[4][PAIRS];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
#pragma unroll
      for (int j = 0; j < PAIRS; ++j) {
        const int c = min((tid + j * RN_THREADS) * 2, cols - 2);
        w[u][j] = *reinterpret_cast<const float2*>(part + (size_t)min(s + u, splits - 1) * mn + (size_t)b * cols + c);
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (s + u >= splits) break;
#pragma unroll
      for (int j = 0; j < PAIRS; ++j) {
        acc[j].x += w[u][j].x;
        acc[j].y += w[u][j].y;
      }
    }
  }
  half2_t val[PAIRS];
#pragma unroll
  for (int j = 0; j < PAIRS; ++j) {
    const int c = (tid + j * RN_THREADS) * 2;
    val[j].x = round_f16(fmaf(1.0f, (float)old[j].x, acc[j].x));
    val[j].y = round_f16(fmaf(1.0f, (float)old[j].y, acc[j].y));
    if (c < cols) {
      *reinterpret_cast<half2_t*>(xr + c) = val[j];
      *reinterpret_cast<half2_t*>(row_lds + c) = val[j];
    }
  }
  __syncthreads();
  float s = 0.0f;
  if (tid < 256) {
    for (int i = tid; i < cols; i += 256) {
      const float v = (float)row_lds[i];
      s = fmaf(v, v, s);
    }
  }
  // block256_sum_ref_order for the first 256 threads of a larger workgroup
#pragma unroll
  for (int off = 16; off > 0; off >>= 1) {
    s += __shfl_xor(s, off, WAVE);
  }
  if (tid < 256 && (tid & 31) == 0) {
    red[tid >> 5] = s;
  }
  __syncthreads();
  float total = red[tid & 7];
#pragma unroll
  for (int off = 4; off > 0; off >>= 1) {
    total += __shfl_xor(total, off, WAVE);
  }
  const float rms_inv = 1.0f / sqrtf(total / (float)cols + eps);
  half_t* y = norm_out + (size_t)b * cols;
#pragma unroll
  for (int j = 0; j < PAIRS; ++j) {
    const int c = (tid + j * RN_THREADS) * 2;
    if (c < cols) {
      half2_t r;
      r.x = round_f16((float)wv[j].x * (float)round_f16((float)val[j].x * rms_inv));
      r.y = round_f16((float)wv[j].y * (float)round_f16((float)val[j].y * rms_inv));
      *reinterpret_cast<half2_t*>(y + c) = r;
    }
  }
}

template <int BM, int BN, int KS>
constexpr size_t gemm_lds_bytes() {
  return (size_t)2 * (BM + BN) * (BK * KS + 8) * sizeof(half_t);
}

template <int BM, int BN, bool U8, bool KTAIL, int KS>
int launch_one(half_t* out, const half_t* A, const void* W, const half_t* S, int M, int K, int N, int block,
               float beta, int tiles_m, int tiles_n, hipStream_t st) {
  constexpr size_t lds = gemm_lds_bytes<BM, BN, KS>();
  static_assert(lds >= (size_t)BM * BN * 4 / 2 || KS == 1, "LDS must hold one group's accumulators");
  auto kernel = gemm_kernel<BM, BN, U8, KTAIL, KS>;
  if constexpr (lds > 64 * 1024) {
    static bool raised[16] = {};  // per device, once
    int dev = 0;
    LCU_HIP(hipGetDevice(&dev));
    if (!raised[dev & 15]) {
      LCU_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
      raised[dev & 15] = true;
    }
  }
  kernel<<<tiles_m * tiles_n, 256 * KS, lds, st>>>(out, A, W, S, M, K, N, block, beta, tiles_m, tiles_n);
  LCU_LAUNCH_CHECK();
  return LCU_OK;
}

template <int BM, int BN, bool U8, int KS>
int launch_gemm(half_t* out, const half_t* A, const void* W, const half_t* S, int M, int K, int N, int block,
                float beta, hipStream_t st) {
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  if (K % (BK * KS) == 0) {
    return launch_one<BM, BN, U8, false, KS>(out, A, W, S, M, K, N, block, beta, tiles_m, tiles_n, st);
  }
  return launch_one<BM, BN, U8, true, KS>(out, A, W, S, M, K, N, block, beta, tiles_m, tiles_n, st);
}

// rotary: rotates the outputs where the product takes gemm_tile_kernel without a split; *rotated then says so.
template <bool U8>
int dispatch_gemm(operands_t op, const half_t* A, int M, int K, int N, int block, float beta, hipStream_t st,
                  const rotary_epilogue* rotary = nullptr, bool* rotated = nullptr) {
  // Tile choice.  Large tiles read fewer operand bytes per multiply-add and pay per output for fewer
  // barriers.  So: tiles of 256 rows when those of 256x128 still give 160 workgroups, or with few of them
  // and a long K the splits of each (large_tile_splits); 128x128 when these give 160; 128x64 with a ring of
  // three stages when there are more of them than compute units (two fit); else 128x64 with a longer ring, the
  // even and the odd stages summed apart.
  // gemm_tile_kernel pays about 1 us more per tile before its first and behind its last stage than gemm_dl_kernel (a longer ring
  // to fill, outputs through LDS) and less per stage: over a short K the other kernels stay, by the lines below.
  // Several matrices of one shape (op.n_mats > 1) count as one product with n_mats * N columns; only uint8
  // weights in blocks other than 64 << n, whose kernel has one width of large tiles, take a launch each where
  // a matrix fills the chip with 256x128 tiles and fusing saves no round of workgroups.
  const bool whole_stages = K % 128 == 0 && scale_words_ok<U8>(op, K, N, block);
  if (U8 && block_shift(block) < 0 && op.n_mats > 1 && M > 64 && whole_stages) {
    device_state* ds = current_device_state();
    const long cus = ds && ds->compute_units > 0 ? ds->compute_units : 256;
    const long per = (long)((M + 255) / 256) * ((N + 127) / 128);
    if (per >= 160 && (per * op.n_mats + cus - 1) / cus >= op.n_mats * ((per + cus - 1) / cus)) {
      for (int g = 0; g < op.n_mats; ++g) {
        const operands_t one = single_matrix(g == 0 ? op.out : op.more.out[g - 1], g == 0 ? op.W : op.more.W[g - 1],
                                             g == 0 ? op.S : op.more.S[g - 1]);
        const int rc = dispatch_gemm<U8>(one, A, M, K, N, block, beta, st);
        if (rc != LCU_OK) {
          return rc;
        }
      }
      return LCU_OK;
    }
  }
  const long nm = op.n_mats;
  const long tiles128 = (long)((M + 127) / 128) * ((N + 127) / 128) * nm;
  const long tiles64 = (long)((M + 127) / 128) * ((N + 63) / 64) * nm;
  if (whole_stages && M <= 64) {  // short prompts: the weight stream is what counts
    bool done = false;
    int rc;
    if constexpr (U8) {  // 64-row tiles with the code ring would leave LDS for one workgroup only
      rc = launch_skinny<32, true>(op, A, M, K, N, block, beta, st, &done);
    } else {
      rc = M <= 32 ? launch_skinny<32, false>(op, A, M, K, N, block, beta, st, &done)
                   : launch_skinny<64, false>(op, A, M, K, N, block, beta, st, &done);
    }
    if (rc != LCU_OK || done) {
      return rc;
    }
  }
  if (whole_stages) {  // whole stages: the direct-to-LDS kernels
    device_state* ds = current_device_state();
    const long cus = ds && ds->compute_units > 0 ? ds->compute_units : 256;
    const workspace_t ws = workspace_for(st);
    const row_plan_t plan = plan_rows(M, K, N, op.n_mats, cus, ds != nullptr && ws.ptr != nullptr ? ws.bytes : 0);
    if (plan.tiles == row_tiles::large) {
      if constexpr (U8) {
        // over a short K gemm_dl_kernel is done sooner (us, it / gemm_tile_kernel, K 256, 512, 768: 512 rows of 12288 columns 11.2 / 12.4,
        // 15.1 / 16.2, 18.7 / 18.3; several rounds of workgroups, 1015 rows, three times 4096 columns of K 256 20.2 / 22.0, 1805
        // rows, three times 8256 of K 384 85.6 / 90.3, 1987 rows, three times 4096 of K 512 52.2 / 46.9)
        const bool one_round = tiles_of(M, N, 256, 128) * nm <= cus;
        if (block_shift(block) < 0 || (M > 128 && K < (one_round ? 640 : 448))) {
          return launch_dl<256, 128, 4, 2, 1, 3, U8>(op, A, M, K, N, block, beta, st);
        }
      }
      if (rotary && N % 8 == 0) {
        *rotated = true;
        return launch_large<U8>(*rotary, op, A, M, K, N, block, beta, st);
      }
      return launch_large<U8>(f16_epilogue{}, op, A, M, K, N, block, beta, st);
    }
    if (plan.tiles == row_tiles::split_large) {
      if constexpr (U8) {
        if (block_shift(block) < 0) return launch_split<256, 128, 4, 2, U8>(op, A, M, K, N, block, beta, st, plan.splits, (float*)ws.ptr);
      }
      return launch_large_split<U8>(op, A, M, K, N, block, beta, st, plan.splits, (float*)ws.ptr, cus);
    }
    // Tiles of 128x128, the ring of four stages filled by address-free requests: us here against a two-stage ring with two
    // workgroups per compute unit (from 256 tiles up) or eight wavefronts and three stages (below), M x K x N: 256 tiles
    // 1000x4096x4096 71 -> 41, 1024x2048x4096 39 -> 24; 288 tiles 1100x4096x4096 55 -> 47; 160 and 192 tiles the same
    // (512x4096x5120 40, 384x4096x4096 twice 42).  uint8, against eight wavefronts with a
    // ring of codes or, from 256 tiles up, the register-staged kernel: 1000x4096x4096 67 -> 44, 1100 rows 69 -> 56, 200 rows of
    // three matrices 55 -> 41, 512x4096x5120 54 -> 39.
    if (plan.tiles == row_tiles::medium) {
      if constexpr (U8) {
        // Several matrices, each with so few tiles that a call of its own would sum the even and the odd stages apart: so does their common
        // launch, on gemm_dl_kernel.  us, weights from memory, separate calls / here: blocks of 32, which such calls take to the same kernel,
        // 512 rows, three times 3072x3072 78 / 73, 1000 rows, twice 2048 columns of K 4608 74 / 73.  Blocks of 64 << n, which they take to the
        // two chains of gemm_tile_kernel below, 67 / 73 and 63 / 72, 768 rows, three times 2048x2048 49 / 51: there this launch is behind.
        const bool one_chain = tiles128 < 256 || tiles128 / nm >= 256 || tiles64 / nm > 256;
        if (!one_chain) return launch_dl<128, 64, 2, 2, 2, 3, true>(op, A, M, K, N, block, beta, st);
        // us, the older kernel / here, K 256, 512, 1024, 2048: 512 rows of 5120 columns 7.6 / 7.8, 10.5 / 9.8, 16.3 / 13.7; one matrix with
        // more tiles than compute units, which the register-staged kernel puts two to a compute unit, 1000 rows of 4608 columns
        // 11.4 / 14.0, 15.8 / 17.8, 24.5 / 25.6, 41.9 / 41.6
        const bool long_enough = tiles128 < 256 ? K >= 384 : tiles128 / nm <= 256 || K >= 1536;
        if (block_shift(block) >= 0 && long_enough) {
          if (rotary && N % 8 == 0) {
            *rotated = true;
            return launch_tile<128, 128, 1, 4, 4, 4, true, false>(*rotary, op, A, M, K, N, block, beta, st);
          }
          return launch_tile<128, 128, 1, 4, 4, 4, true, false>(f16_epilogue{}, op, A, M, K, N, block, beta, st);
        }
        if (tiles128 < 256) return launch_dl<128, 128, 4, 2, 1, 3, true>(op, A, M, K, N, block, beta, st);
      } else {
        // us, K 256, 512, 1024, 1536, 2048: eight wavefronts / here, 512 rows of 5120 columns 6.2 / 7.1, 7.8 / 8.5, 10.9 / 11.2, 16.1 / 15.2, 22.0 / 22.3;
        // two workgroups per compute unit / here, 1000 rows of 4608 columns 9.6 / 12.4, 13.2 / 15.7, 20.8 / 21.4, 29.3 / 27.9, 39.5 / 35.1
        if (K < 1280 && tiles128 < 256) return launch_dl<128, 128, 4, 2, 1, 3, false>(op, A, M, K, N, block, beta, st);
        // with weights from memory the second workgroup also hides the second round's first requests: K 1280, 1536, 1792, 512 rows of
        // 10000 columns 30.3 / 34.4, 34.2 / 38.2, 38.9 / 42.0, 896 rows of 4992 26.6 / 28.3, 30.4 / 31.0, 34.6 / 34.1
        if (K < 1536 && tiles128 > 256) return launch_dl<128, 128, 2, 2, 1, 2, false>(op, A, M, K, N, block, beta, st);
        if (rotary && N % 8 == 0) {
          *rotated = true;
          return launch_tile<128, 128, 2, 2, 4, 4, false, false>(*rotary, op, A, M, K, N, 0, beta, st);
        }
        return launch_tile<128, 128, 2, 2, 4, 4, false, false>(f16_epilogue{}, op, A, M, K, N, 0, beta, st);
      }
    } else {
      // More 128x64 tiles than compute units, two to a compute unit: against gemm_dl_kernel 40 drawn products of K 256 to 5000 take 0.98 of the time
      // (0.92 to 1.02; 1038x4096x2048 37.5 / 34.8 us), uint8 0.78 (0.70 to 0.86; 559x1792x3352 25.6 / 18.0): every code converted once, not twice.
      if (plan.tiles == row_tiles::narrow) {
        if constexpr (U8) {
          if (block_shift(block) >= 0) return launch_tile<128, 64, 1, 4, 3, 3, true, false>(f16_epilogue{}, op, A, M, K, N, block, beta, st);
          return launch_dl<128, 64, 2, 2, 1, 3, true>(op, A, M, K, N, block, beta, st);
        } else {
          return launch_tile<128, 64, 2, 2, 3, 3, false, false>(f16_epilogue{}, op, A, M, K, N, 0, beta, st);
        }
      }
      // us, two groups of four wavefronts that halve the stages on gemm_dl_kernel / four that sum them in turn here: 300x4096x4096 25.1 / 23.8,
      // 1000x2048x2048 17.2 / 15.7; 512 rows of 4096 columns, K 256, 512, 1024, 2048 6.3 / 5.2, 7.2 / 6.1, 10.9 / 9.7, 15.4 / 15.0, but K 4096 28.9 / 29.3:
      // 24 KB a stage on their way into LDS bound it over a long K, and the rest is what it gains.  70 drawn products 0.91 of the time (0.82 to
      // 1.03), 45 in uint8 0.84 (0.79 to 0.88).
      // Smaller ones where these would leave compute units idle: 90 rows of 2048 columns eight fp16 layers 0.90 -> 0.71 ms.
      // Outputs over lhs keep the tiles whose workgroup, where all columns are one tile, has read its rows before it stores them.
      const tile_size_t tile = over_lhs(op, A, M, K, N) ? tile_size_t{128, 64} : plan_tile_size(M, N, op.n_mats, {128, 64}, !U8, cus);
      const f16_epilogue ep{};
      if constexpr (U8) {
        if (block_shift(block) < 0) return launch_dl<128, 64, 2, 2, 2, 3, true>(op, A, M, K, N, block, beta, st);
        if (tile.rows == 64) return launch_tile<64, 64, 1, 4, 4, 4, true, false, f16_epilogue, 2>(ep, op, A, M, K, N, block, beta, st);
        return launch_tile<128, 64, 1, 4, 4, 4, true, false, f16_epilogue, 2>(ep, op, A, M, K, N, block, beta, st);
      } else {
        if (tile.columns == 32) return launch_tile<64, 32, 1, 2, 4, 4, false, false, f16_epilogue, 2>(ep, op, A, M, K, N, 0, beta, st);
        if (tile.rows == 64) return launch_tile<64, 64, 1, 4, 4, 4, false, false, f16_epilogue, 2>(ep, op, A, M, K, N, 0, beta, st);
        return launch_tile<128, 64, 2, 2, 4, 4, false, false, f16_epilogue, 2>(ep, op, A, M, K, N, 0, beta, st);
      }
    }
  }
  // ragged K: the register-staged kernel, one matrix per launch
  for (int g = 0; g < op.n_mats; ++g) {
    half_t* out = g == 0 ? op.out : op.more.out[g - 1];
    const void* W = g == 0 ? op.W : op.more.W[g - 1];
    const half_t* S = g == 0 ? op.S : op.more.S[g - 1];
    const long t128 = tiles128 / nm, t64 = tiles64 / nm;
    int rc;
    if (t128 >= 256) {
      rc = launch_gemm<128, 128, U8, 1>(out, A, W, S, M, K, N, block, beta, st);
    } else if (t64 > 256) {
      rc = launch_gemm<128, 64, U8, 1>(out, A, W, S, M, K, N, block, beta, st);
    } else {
      rc = launch_gemm<128, 64, U8, 2>(out, A, W, S, M, K, N, block, beta, st);
    }
    if (rc != LCU_OK) {
      return rc;
    }
  }
  return LCU_OK;
}

// ---- bfloat16 operands ----
// splits > 1: the K stages of every tile dealt to that many workgroups, fp32 sums to part (no epilogue)
template <int BM, int BN, int WM, int WN, int KS, int NS, bool SPLIT = false, class EP>
int launch_bf16(EP const& ep, const void* A, const void* W, int tiles_m, int M, int K, int N, hipStream_t st, int splits = 1,
                float* part = nullptr) {
  constexpr int ROWB = BK * KS * 2;
  constexpr size_t lds = (size_t)NS * (BM + BN) * ROWB;
  static_assert(lds <= 160 * 1024, "rings do not fit LDS");
  static_assert(KS == 1 || lds >= (size_t)BM * BN * 4 / 2, "LDS must hold one group's accumulators");
  auto kernel = gemm_dl_kernel<BM, BN, WM, WN, KS, NS, false, SPLIT, EP>;
  if constexpr (lds > 64 * 1024) {
    static bool raised[16] = {};  // per device, once
    int dev = 0;
    LCU_HIP(hipGetDevice(&dev));
    if (!raised[dev & 15]) {
      LCU_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
      raised[dev & 15] = true;
    }
  }
  const int tiles_n = (N + BN - 1) / BN;
  const more_matrices_t none{{nullptr, nullptr}, {nullptr, nullptr}, {nullptr, nullptr}, 0};
  kernel<<<tiles_m * tiles_n * splits, 64 * WM * WN * KS, lds, st>>>(nullptr, (const half_t*)A, W, nullptr, M, K, N, 0, 0.0f,
                                                                     tiles_m, tiles_n, part, splits, none, ep);
  LCU_LAUNCH_CHECK();
  return LCU_OK;
}

// the splits' sums in split order, then the epilogue; a thread per output
template <bool GATED>
__global__ __launch_bounds__(256) void splitk_epilogue_kernel(linear_epilogue<false, GATED> ep, const float* __restrict__ part, int M,
                                                              int N, int splits) {
  const int outs = GATED ? N / 2 : N, i = blockIdx.x * 256 + threadIdx.x;
  if (i >= M * outs) return;
  const int m = i / outs, n = i - m * outs;
  const auto sum = [&](int c) {
    float s = 0.0f;
    for (int k = 0; k < splits; ++k) s += part[((size_t)k * M + m) * N + c];
    return s;
  };
  if constexpr (GATED) {
    const int c = n / 32 * 64 + n % 32;
    ep.store_gated(m, n, sum(c), sum(c + 32));
  } else {
    ep.store(m, n, sum(n));
  }
}

template <bool GATED_>
struct linear_join {
  static constexpr bool JOINED = true, GATED = GATED_;
  static constexpr int MATRICES = GATED ? 2 : 1;
  linear_epilogue<false, GATED> ep;
  int N;
  __device__ __forceinline__ void operator()(int, int row, int c, const float2 (&x)[MATRICES]) const {
    if constexpr (GATED) {
      ep.store_gated(row, c, x[0].x, x[1].x);
      ep.store_gated(row, c + 1, x[0].y, x[1].y);
    } else {
      ep.store(row, c, x[0].x);
      if (c + 1 < N) ep.store(row, c + 1, x[0].y);
    }
  }
};

// The same in one launch (launch_joined; us, two / one: 6x2048x2048 6.8 / 5.6, 13x2048x6656 12.5 / 9.2, 42x768x6656 11.4 / 7.4, 11x2048x256 7.7 / 4.9; 40
// drawn shapes of 2 to 62 rows 7 to 71 % sooner where K is split).  *done = false, with nothing launched, where lhs does not fit LDS whole, the workgroups would take a
// second round, or the outputs lie over lhs.
template <bool GATED>
int bf16_joined(linear_epilogue<false, GATED> const& ep, const void* A, const void* W, int M, int K, int N, int splits, long cus, bool memory,
                hipStream_t st, bool* done) {
  *done = false;
  const int outs = GATED ? N / 2 : N;
  if (K % 128 != 0 || (GATED && outs % 32 != 0) || over_lhs(ep, A, M, K, N)) return LCU_OK;
  const int mats = GATED ? 2 : 1;
  const stream_join_t shape = plan_stream_join(M, K, outs, mats, mats, splits, cus, false);
  if (shape.waves == 0) return LCU_OK;
  const int rc = launch_joined_shape<false, true>(linear_join<GATED>{ep, N}, single_matrix(nullptr, W, nullptr), (const half_t*)A, M, K, N, 0, st, splits, shape,
                                                memory);
  *done = rc == LCU_OK;
  return rc;
}

// Few rows: the weight stream is what counts (see launch_skinny).  *done = false when the shape gives no second
// workgroup to a tile.
template <bool GATED>
int bf16_skinny(linear_epilogue<false, GATED> const& ep, const void* A, const void* W, int M, int K, int N, hipStream_t st, bool* done) {
  *done = false;
  device_state* ds = current_device_state();
  const workspace_t ws = workspace_for(st);
  if (ds == nullptr || ws.ptr == nullptr) return LCU_OK;
  const int tiles = (N + 127) / 128;
  int splits = std::min((ds->compute_units + tiles - 1) / tiles, K / BK / 4);
  while (splits > 1 && (size_t)splits * M * N * sizeof(float) > ws.bytes) --splits;
  if (splits < 2) return LCU_OK;
  const bool memory = from_memory(ws.weights, (size_t)N * K * 2);
  int rc = bf16_joined<GATED>(ep, A, W, M, K, N, splits, ds->compute_units, memory, st, done);
  if (rc != LCU_OK || *done) return rc;
  float* part = (float*)ws.ptr;
  if (streams(M, N, 1, splits, K / BK, (long)tiles * splits, ds->compute_units, false, true, memory)) {
    rc = launch_stream<false, true>(single_matrix(nullptr, W, nullptr), A, M, K, N, 0, st, splits, part, ds->compute_units, memory);
  } else {
    rc = M <= 32 ? launch_bf16<32, 128, 1, 4, 1, 3, true>(ep, A, W, 1, M, K, N, st, splits, part)
                 : launch_bf16<64, 128, 1, 4, 1, 3, true>(ep, A, W, 1, M, K, N, st, splits, part);
  }
  if (rc != LCU_OK) return rc;
  const int outs = M * (GATED ? N / 2 : N);
  splitk_epilogue_kernel<GATED><<<(outs + 255) / 256, 256, 0, st>>>(ep, part, M, N, splits);
  LCU_LAUNCH_CHECK();
  *done = true;
  return LCU_OK;
}

}  // namespace

namespace lcu {

// One product with every row of lhs: the tile choice of dispatch_gemm.  GATED tiles give a wavefront 64
// columns (a 32-wide gate block and its up block).
template <bool GATED>
int gemm_bf16(linear_epilogue<false, GATED> const& ep, const void* A, const void* W, int M, int K, int N, hipStream_t st) {
  const auto tm = [&](int bm) { return (M + bm - 1) / bm; };
  const auto tn = [&](int bn) { return (long)((N + bn - 1) / bn); };
  const device_state* ds = current_device_state();
  const long cus = ds && ds->compute_units > 0 ? ds->compute_units : 256;
  if (M <= 64) {
    bool done = false;
    const int rc = bf16_skinny<GATED>(ep, A, W, M, K, N, st, &done);
    if (rc != LCU_OK || done) return rc;
    return launch_bf16<64, 64, 2, GATED ? 1 : 2, 1, 3>(ep, A, W, tm(64), M, K, N, st);
  }
  if (tm(256) * tn(128) >= 160) return launch_large<false>(ep, single_matrix(nullptr, W, nullptr), A, M, K, N, 0, 0.0f, st);
  if constexpr (GATED) {  // 1000 rows of 4608 columns, K 512, 1024, 2048: 17.2 us, 24.5, 43.1 with two workgroups per compute unit, else 17.8, 24.8, 39.7
    if (K < 1280 && tm(128) * tn(128) > 256) return launch_bf16<128, 128, 2, 2, 1, 2>(ep, A, W, tm(128), M, K, N, st);
  }
  if (tm(128) * tn(128) >= 160) return launch_tile<128, 128, 2, 2, 4, 4, false, false>(ep, single_matrix(nullptr, W, nullptr), A, M, K, N, 0, 0.0f, st);
  if constexpr (GATED) {
    if (gated_on_tiles(M, K, N, cus, from_memory(workspace_for(st).weights, (size_t)N * K * 2))) {
      return launch_tile<128, 64, 2, 1, 4, 4, false, false>(ep, single_matrix(nullptr, W, nullptr), A, M, K, N, 0, 0.0f, st);
    }
    if (tm(128) * tn(64) > 128) return launch_bf16<128, 64, 4, 1, 1, 3>(ep, A, W, tm(128), M, K, N, st);
    return launch_bf16<64, 64, 2, 1, 1, 3>(ep, A, W, tm(64), M, K, N, st);
  } else {
    if (tm(128) * tn(64) > 256) return launch_tile<128, 64, 2, 2, 3, 3, false, false>(ep, single_matrix(nullptr, W, nullptr), A, M, K, N, 0, 0.0f, st);
    if (K % 128 == 0 && tm(128) * tn(64) > 128) {
      return launch_tile<128, 64, 2, 2, 4, 4, false, false, linear_epilogue<false, GATED>, 2>(ep, single_matrix(nullptr, W, nullptr), A, M, K, N, 0, 0.0f, st);
    }
    // us, on gemm_dl_kernel / here: 100x2048x2048 16.3 / 11.0, 200x4096x4096 29.4 / 20.9, 66x4096x8192 30.5 / 24.2
    const operands_t op = single_matrix(nullptr, W, nullptr);
    const tile_size_t tile = over_lhs(ep, A, M, K, N) ? tile_size_t{64, 64} : plan_tile_size(M, N, 1, {64, 64}, true, cus);  // over lhs: as in dispatch_gemm
    if (tile.columns == 32) return launch_tile<64, 32, 1, 2, 4, 4, false, false>(ep, op, A, M, K, N, 0, 0.0f, st);
    return launch_tile<64, 64, 1, 4, 4, 4, false, false>(ep, op, A, M, K, N, 0, 0.0f, st);
  }
}
template int gemm_bf16<false>(linear_epilogue<false, false> const&, const void*, const void*, int, int, int, hipStream_t);
template int gemm_bf16<true>(linear_epilogue<false, true> const&, const void*, const void*, int, int, int, hipStream_t);

// Products of groups of rows with one matrix each, from the tile list in ep (row tiles of ep.tile_rows rows, at
// most max_tiles of them).
// What bounds them is the weight stream, up to some 100 rows a group: 24 GB/s to a compute unit, those lines included that two row tiles of
// a group both ask for.  So a group's rows go into one tile where they fit: 512 tokens, top 2 of 16 experts of 4096 x 5632 and 2816 x 4096,
// tiles of 64 rows 183 and 101 us, of 128 152 and 86 (159 and 89 on gemm_dl_kernel), of 256 178 and 94; 340 tokens 146 and 75, 150 and 80, 170 and
// 90; 1000 tokens 225 and 121, 192 and 115, 185 and 104 (gemm_dl_kernel 219 and 117); 2010 tokens 353 and 187, 302 and 168, 250 and 145 (281 and
// 160).  Over 12 600 drawn products tiles of 128 rows take 0.97 (gated) and 0.95 of their time on gemm_dl_kernel, where rings of three stages of
// lhs and seven of W took 1.04 and 1.03.
// A few rows to a tile and a short K are left to that kernel: the gated epilogue of a whole tile through LDS is what counts then (up to 8
// tokens a tile, tiles of 128 / 256 rows, here against it: K 512 1.16 and 1.11 times as long, 1024 1.08 and 1.01, 2048 1.04 and 0.97, 4096 0.99 and 0.92).
template <bool GATED>
int gemm_bf16_grouped(linear_epilogue<true, GATED> const& ep, const void* A, const void* W, int max_tiles, int K, int N,
                      hipStream_t st) {
  const operands_t op = single_matrix(nullptr, W, nullptr);
  if constexpr (GATED) {
    const bool few = ep.lhs_rows <= 8 * max_tiles;  // tokens to a tile: rows, where a token takes one expert
    if (few && ep.tile_rows == 256 && K <= 512) return launch_bf16<256, 128, 4, 2, 1, 3>(ep, A, W, max_tiles, 0, K, N, st);
    if (few && ep.tile_rows == 128 && K <= 2048) return launch_bf16<128, 128, 4, 2, 1, 3>(ep, A, W, max_tiles, 0, K, N, st);
  }
  if (ep.tile_rows == 64) return launch_bf16<64, 128, 2, 2, 1, 3>(ep, A, W, max_tiles, 0, K, N, st);
  const auto tiles = [&](auto const& e) {
    if (ep.tile_rows == 256) return launch_tile<256, 128, 4, 2, 3, 3, false, false>(e, op, A, max_tiles * 256, K, N, 0, 0.0f, st);
    return launch_tile<128, 128, 2, 2, 4, 4, false, false>(e, op, A, max_tiles * 128, K, N, 0, 0.0f, st);
  };
  // Weights that come from memory are marked as read once, whatever the rows to an expert: one that takes two row tiles asks for its lines in both at the same
  // time.  us, both products, unmarked / marked, from memory: top 2 of 16 of 2816, 4096 wide, 512 tokens 240 / 230, 1000 291 / 285, 2010 412 / 395, 4000 (500
  // rows to an expert) 636 / 617; top 4 of 64 of 704, 2048 wide, 1000 161 / 151, 4000 259 / 248.  Those that may lie in the cache are not: top 2 of 8 of 512,
  // 1024 wide (25 MB), again and again 1000 27.0 / 28.5, 2010 35.3 / 37.4, 4000 65 / 70.
  if (!from_memory(workspace_for(st).weights, 0)) return tiles(ep);
  read_once<GATED> marked;
  static_cast<linear_epilogue<true, GATED>&>(marked) = ep;
  return tiles(marked);
}
template int gemm_bf16_grouped<false>(linear_epilogue<true, false> const&, const void*, const void*, int, int, int, hipStream_t);
template int gemm_bf16_grouped<true>(linear_epilogue<true, true> const&, const void*, const void*, int, int, int, hipStream_t);

}  // namespace lcu

extern "C" {

int lcu_gemm_f16_nt(void* out_dev, const void* lhs_dev, const void* rhs_dev, int M, int K, int N, float beta,
                    void* stream) {
  LCU_REQUIRE(out_dev && lhs_dev && rhs_dev, "lcu_gemm_f16_nt: null pointer");
  LCU_REQUIRE(M >= 0 && N > 0 && K > 0 && K % 8 == 0, "lcu_gemm_f16_nt: bad shape M %d K %d N %d (K %% 8 == 0)", M, K,
              N);
  if (M == 0) return LCU_OK;
  LCU_REQUIRE((size_t)M * K * 2 < ((size_t)1 << 32) && (size_t)N * K * 2 < ((size_t)1 << 32),
              "lcu_gemm_f16_nt: operands of 4 GiB or more are not supported");
  if (M == 1 && K <= 24576) {
    return gemv_f16((half_t*)out_dev, (const half_t*)lhs_dev, (const half_t*)rhs_dev, K, N, beta, as_stream(stream));
  }
  return dispatch_gemm<false>(single_matrix((half_t*)out_dev, rhs_dev, nullptr), (const half_t*)lhs_dev, M, K, N, 0, beta,
                              as_stream(stream));
}

int lcu_gemm_f16_nt_multi(void* const* out_dev, const void* lhs_dev, const void* const* rhs_dev, int n_mats, int M,
                          int K, int N, float beta, void* stream) {
  LCU_REQUIRE(out_dev && lhs_dev && rhs_dev && n_mats >= 1 && n_mats <= 3, "lcu_gemm_f16_nt_multi: bad arguments");
  for (int g = 0; g < n_mats; ++g) {
    LCU_REQUIRE(out_dev[g] && rhs_dev[g], "lcu_gemm_f16_nt_multi: null pointer");
  }
  if (M == 1 || n_mats == 1) {  // matrix-vector products and single matrices: the ordinary entry point
    for (int g = 0; g < n_mats; ++g) {
      const int rc = lcu_gemm_f16_nt(out_dev[g], lhs_dev, rhs_dev[g], M, K, N, beta, stream);
      if (rc != LCU_OK) return rc;
    }
    return LCU_OK;
  }
  LCU_REQUIRE(M >= 0 && N > 0 && K > 0 && K % 8 == 0, "lcu_gemm_f16_nt_multi: bad shape M %d K %d N %d (K %% 8 == 0)", M,
              K, N);
  if (M == 0) return LCU_OK;
  LCU_REQUIRE((size_t)M * K * 2 < ((size_t)1 << 32) && (size_t)N * K * 2 < ((size_t)1 << 32),
              "lcu_gemm_f16_nt_multi: operands of 4 GiB or more are not supported");
  operands_t op = single_matrix((half_t*)out_dev[0], rhs_dev[0], nullptr);
  op.n_mats = n_mats;
  for (int g = 1; g < n_mats; ++g) {
    op.more.out[g - 1] = (half_t*)out_dev[g];
    op.more.W[g - 1] = rhs_dev[g];
  }
  return dispatch_gemm<false>(op, (const half_t*)lhs_dev, M, K, N, 0, beta, as_stream(stream));
}

int lcu_gemm_f16u8_nt(void* out_dev, const void* lhs_dev, const void* codes_dev, const void* scales_dev, int M,
                      int K, int N, int block, float beta, void* stream) {
  LCU_REQUIRE(out_dev && lhs_dev && codes_dev && scales_dev, "lcu_gemm_f16u8_nt: null pointer");
  LCU_REQUIRE(M >= 0 && N > 0 && K > 0 && K % 16 == 0 && block >= 16 && block % 16 == 0 && K % block == 0,
              "lcu_gemm_f16u8_nt: bad shape M %d K %d N %d block %d (K %% 16 == 0, block %% 16 == 0, K %% block == 0)",
              M, K, N, block);
  if (M == 0) return LCU_OK;
  LCU_REQUIRE((size_t)M * K * 2 < ((size_t)1 << 32) && (size_t)N * K < ((size_t)1 << 32),
              "lcu_gemm_f16u8_nt: operands of 4 GiB or more are not supported");
  if (M == 1 && K <= 24576) {
    return gemv_u8((half_t*)out_dev, (const half_t*)lhs_dev, (const uint8_t*)codes_dev, (const half_t*)scales_dev, K,
                   N, block, beta, as_stream(stream));
  }
  return dispatch_gemm<true>(single_matrix((half_t*)out_dev, codes_dev, (const half_t*)scales_dev), (const half_t*)lhs_dev,
                             M, K, N, block, beta, as_stream(stream));
}

int lcu_gemm_f16u8_nt_multi(void* const* out_dev, const void* lhs_dev, const void* const* codes_dev,
                            const void* const* scales_dev, int n_mats, int M, int K, int N, int block, float beta,
                            void* stream) {
  LCU_REQUIRE(out_dev && lhs_dev && codes_dev && scales_dev && n_mats >= 1 && n_mats <= 3,
              "lcu_gemm_f16u8_nt_multi: bad arguments");
  for (int g = 0; g < n_mats; ++g) {
    LCU_REQUIRE(out_dev[g] && codes_dev[g] && scales_dev[g], "lcu_gemm_f16u8_nt_multi: null pointer");
  }
  if (M == 1 || n_mats == 1) {
    for (int g = 0; g < n_mats; ++g) {
      const int rc = lcu_gemm_f16u8_nt(out_dev[g], lhs_dev, codes_dev[g], scales_dev[g], M, K, N, block, beta, stream);
      if (rc != LCU_OK) return rc;
    }
    return LCU_OK;
  }
  LCU_REQUIRE(M >= 0 && N > 0 && K > 0 && K % 16 == 0 && block >= 16 && block % 16 == 0 && K % block == 0,
              "lcu_gemm_f16u8_nt_multi: bad shape M %d K %d N %d block %d", M, K, N, block);
  if (M == 0) return LCU_OK;
  LCU_REQUIRE((size_t)M * K * 2 < ((size_t)1 << 32) && (size_t)N * K < ((size_t)1 << 32),
              "lcu_gemm_f16u8_nt_multi: operands of 4 GiB or more are not supported");
  operands_t op = single_matrix((half_t*)out_dev[0], codes_dev[0], (const half_t*)scales_dev[0]);
  op.n_mats = n_mats;
  for (int g = 1; g < n_mats; ++g) {
    op.more.out[g - 1] = (half_t*)out_dev[g];
    op.more.W[g - 1] = codes_dev[g];
    op.more.S[g - 1] = (const half_t*)scales_dev[g];
  }
  return dispatch_gemm<true>(op, (const half_t*)lhs_dev, M, K, N, block, beta, as_stream(stream));
}

// ---- fused steps of a batched decode (one row per sequence) ----

static operands_t make_operands(void* const* outs, const void* const* values, const void* const* scales, int count) {
  operands_t op = single_matrix((half_t*)(outs ? outs[0] : nullptr), values[0], (const half_t*)(scales ? scales[0] : nullptr));
  op.n_mats = count;
  for (int g = 1; g < count; ++g) {
    op.more.out[g - 1] = (half_t*)(outs ? outs[g] : nullptr);
    op.more.W[g - 1] = values[g];
    op.more.S[g - 1] = (const half_t*)(scales ? scales[g] : nullptr);
  }
  return op;
}

int lcu_batch_qkv(void* q_out_dev, void* k_tmp_dev, void* v_tmp_dev, const void* lhs_dev, const void* const* w_dev,
                  const void* const* scales_dev, int block, int n_seq, int dim, int n_heads,
                  const void* k_cache_ptrs_dev, const void* v_cache_ptrs_dev, const void* pos_dev,
                  const void* table_dev, int table_positions, void* stream) {
  LCU_REQUIRE(q_out_dev && k_tmp_dev && v_tmp_dev && lhs_dev && w_dev && w_dev[0] && w_dev[1] && w_dev[2] &&
                  k_cache_ptrs_dev && v_cache_ptrs_dev && pos_dev && table_dev,
              "lcu_batch_qkv: null pointer");
  LCU_REQUIRE(n_seq >= 0 && dim > 0 && n_heads > 0 && dim % n_heads == 0 && (dim / n_heads) % 2 == 0 && dim % 16 == 0 &&
                  table_positions > 0,
              "lcu_batch_qkv: bad shape n_seq %d dim %d heads %d", n_seq, dim, n_heads);
  LCU_REQUIRE(block == 0 || (scales_dev && scales_dev[0] && scales_dev[1] && scales_dev[2] && block % 16 == 0 &&
                             dim % block == 0),
              "lcu_batch_qkv: quantised weights need scales and a block dividing dim");
  if (n_seq == 0) return LCU_OK;
  hipStream_t st = as_stream(stream);
  void* const outs[3] = {q_out_dev, k_tmp_dev, v_tmp_dev};
  const sequence_rows rows{(half_t* const*)k_cache_ptrs_dev, (half_t* const*)v_cache_ptrs_dev, (const int*)pos_dev, table_positions - 1};
  bool done = false;
  partial_sums_t ps{};
  if (n_seq > 1) {
    const operands_t op = make_operands(outs, w_dev, block ? scales_dev : nullptr, 3);
    const half_t* lhs = (const half_t*)lhs_dev;
    const rope_join<sequence_rows> join{(half_t*)q_out_dev, rows, (const float2*)table_dev, dim, dim / n_heads};
    int rc = block ? launch_joined<true>(join, op, lhs, n_seq, dim, dim, block, st, nullptr, &done) : launch_joined<false>(join, op, lhs, n_seq, dim, dim, 0, st, nullptr, &done);
    if (rc != LCU_OK || done) return rc;
    rc = block ? skinny_partial<true>(op, lhs, n_seq, dim, dim, block, st, &done, &ps) : skinny_partial<false>(op, lhs, n_seq, dim, dim, 0, st, &done, &ps);
    if (rc != LCU_OK) return rc;
  }
  if (done) {
    reduce_rope_store_kernel<<<dim3((dim / 2 + 255) / 256, n_seq), 256, 0, st>>>((half_t*)q_out_dev, ps.part, ps.splits, n_seq, dim, rows,
                                                                                 dim / n_heads, (const float2*)table_dev);
    LCU_LAUNCH_CHECK();
    return LCU_OK;
  }
  // any other shape: the three products, then rotary and cache append
  const int rc = block ? lcu_gemm_f16u8_nt_multi(outs, lhs_dev, w_dev, scales_dev, 3, n_seq, dim, dim, block, 0.0f, stream)
                       : lcu_gemm_f16_nt_multi(outs, lhs_dev, w_dev, 3, n_seq, dim, dim, 0.0f, stream);
  if (rc != LCU_OK) return rc;
  return lcu_rope_store_batch(q_out_dev, k_tmp_dev, v_tmp_dev, k_cache_ptrs_dev, v_cache_ptrs_dev, pos_dev, n_seq, dim,
                              n_heads, table_dev, table_positions, stream);
}

int lcu_prompt_qkv(void* q_out_dev, void* k_out_dev, void* v_out_dev, const void* lhs_dev, const void* const* w_dev, const void* const* scales_dev,
                   int block, int rows, int dim, int n_heads, int first_position, const void* table_dev, int table_positions, void* stream) {
  LCU_REQUIRE(q_out_dev && k_out_dev && v_out_dev && lhs_dev && w_dev && w_dev[0] && w_dev[1] && w_dev[2] && table_dev, "lcu_prompt_qkv: null pointer");
  LCU_REQUIRE(rows >= 0 && rows <= 65535 && dim > 0 && n_heads > 0 && dim % n_heads == 0 && (dim / n_heads) % 2 == 0 && dim % 16 == 0,
              "lcu_prompt_qkv: bad shape rows %d dim %d heads %d", rows, dim, n_heads);
  LCU_REQUIRE(first_position >= 0 && first_position + rows <= table_positions, "lcu_prompt_qkv: positions %d..%d outside the table of %d",
              first_position, first_position + rows, table_positions);
  LCU_REQUIRE(block == 0 || (scales_dev && scales_dev[0] && scales_dev[1] && scales_dev[2] && block % 16 == 0 && dim % block == 0),
              "lcu_prompt_qkv: quantised weights need scales and a block dividing dim");
  LCU_REQUIRE((size_t)rows * dim * 2 < ((size_t)1 << 32) && (size_t)dim * dim * (block ? 1 : 2) < ((size_t)1 << 32),
              "lcu_prompt_qkv: operands of 4 GiB or more are not supported");
  if (rows == 0) return LCU_OK;
  hipStream_t st = as_stream(stream);
  void* const outs[3] = {q_out_dev, k_out_dev, v_out_dev};
  const half_t* lhs = (const half_t*)lhs_dev;
  const int head_dim = dim / n_heads;
  bool done = false;
  if (rows > 1) {
    const operands_t op = make_operands(outs, w_dev, block ? scales_dev : nullptr, 3);
    partial_sums_t ps{};
    const prompt_rows to{(half_t*)k_out_dev, (half_t*)v_out_dev, first_position};
    const rope_join<prompt_rows> join{(half_t*)q_out_dev, to, (const float2*)table_dev, dim, head_dim};
    int rc = block ? launch_joined<true>(join, op, lhs, rows, dim, dim, block, st, nullptr, &done) : launch_joined<false>(join, op, lhs, rows, dim, dim, 0, st, nullptr, &done);
    if (rc != LCU_OK || done) return rc;
    rc = block ? skinny_partial<true>(op, lhs, rows, dim, dim, block, st, &done, &ps) : skinny_partial<false>(op, lhs, rows, dim, dim, 0, st, &done, &ps);
    if (rc != LCU_OK) return rc;
    if (done) {
      reduce_rope_store_kernel<<<dim3((dim / 2 + 255) / 256, rows), 256, 0, st>>>((half_t*)q_out_dev, ps.part, ps.splits, rows, dim, to, head_dim,
                                                                                  (const float2*)table_dev);
      LCU_LAUNCH_CHECK();
      return LCU_OK;
    }
    const rotary_epilogue turn{(const float2*)table_dev, head_dim, first_position, 2};
    const rotary_epilogue* rotary = head_dim % 8 == 0 && (reinterpret_cast<uintptr_t>(table_dev) & 15) == 0 ? &turn : nullptr;
    rc = block ? dispatch_gemm<true>(op, lhs, rows, dim, dim, block, 0.0f, st, rotary, &done) : dispatch_gemm<false>(op, lhs, rows, dim, dim, 0, 0.0f, st, rotary, &done);
    if (rc != LCU_OK) return rc;
  } else {
    const int rc = block ? lcu_gemm_f16u8_nt_multi(outs, lhs_dev, w_dev, scales_dev, 3, rows, dim, dim, block, 0.0f, stream)
                         : lcu_gemm_f16_nt_multi(outs, lhs_dev, w_dev, 3, rows, dim, dim, 0.0f, stream);
    if (rc != LCU_OK) return rc;
  }
  return done ? LCU_OK : lcu_rope_pair(q_out_dev, k_out_dev, rows, dim, n_heads, first_position, table_dev, table_positions, stream);
}

int lcu_batch_ffn_up(void* out_dev, void* w1_tmp_dev, void* w3_tmp_dev, const void* lhs_dev, const void* const* w_dev,
                     const void* const* scales_dev, int block, int n_seq, int dim, int ffn, void* stream) {
  LCU_REQUIRE(out_dev && w1_tmp_dev && w3_tmp_dev && lhs_dev && w_dev && w_dev[0] && w_dev[1], "lcu_batch_ffn_up: null pointer");
  LCU_REQUIRE(n_seq >= 0 && dim > 0 && ffn > 0 && dim % 16 == 0 && ffn % 2 == 0, "lcu_batch_ffn_up: bad shape n_seq %d dim %d ffn %d",
              n_seq, dim, ffn);
  LCU_REQUIRE(block == 0 || (scales_dev && scales_dev[0] && scales_dev[1] && block % 16 == 0 && dim % block == 0),
              "lcu_batch_ffn_up: quantised weights need scales and a block dividing dim");
  if (n_seq == 0) return LCU_OK;
  hipStream_t st = as_stream(stream);
  void* const outs[2] = {w1_tmp_dev, w3_tmp_dev};
  bool done = false;
  partial_sums_t ps{};
  if (n_seq > 1) {
    const operands_t op = make_operands(outs, w_dev, block ? scales_dev : nullptr, 2);
    const half_t* lhs = (const half_t*)lhs_dev;
    const silu_join join{(half_t*)out_dev, ffn};
    int rc = block ? launch_joined<true>(join, op, lhs, n_seq, dim, ffn, block, st, out_dev, &done) : launch_joined<false>(join, op, lhs, n_seq, dim, ffn, 0, st, out_dev, &done);
    if (rc != LCU_OK || done) return rc;
    rc = block ? skinny_partial<true>(op, lhs, n_seq, dim, ffn, block, st, &done, &ps) : skinny_partial<false>(op, lhs, n_seq, dim, ffn, 0, st, &done, &ps);
    if (rc != LCU_OK) return rc;
  }
  if (done) {
    const size_t mn = (size_t)n_seq * ffn;
    reduce_silu_kernel<<<(unsigned)((mn / 2 + 255) / 256), 256, 0, st>>>((half_t*)out_dev, ps.part, ps.splits, mn);
    LCU_LAUNCH_CHECK();
    return LCU_OK;
  }
  if (block == 0 && n_seq > 64 && dim % 128 == 0 && ffn % 16 == 0 && (size_t)n_seq * dim * 2 < ((size_t)1 << 32) &&
      (size_t)ffn * dim * 2 < ((size_t)1 << 32) && ffn < 1 << 30 && tiles_of(n_seq, ffn, 256, 128) * 2 >= 160 &&  // those of plan_rows' large tiles
      !overlap(out_dev, (size_t)n_seq * ffn * 2, lhs_dev, (size_t)n_seq * dim * 2)) {  // other workgroups, or the launch for the rest, still read lhs
    operands_t op = single_matrix((half_t*)out_dev, w_dev[0], nullptr);
    op.more.W[0] = w_dev[1];
    return launch_large<false>(silu_epilogue{}, op, lhs_dev, n_seq, dim, 2 * ffn, 0, 0.0f, st);
  }
  const int rc = block ? lcu_gemm_f16u8_nt_multi(outs, lhs_dev, w_dev, scales_dev, 2, n_seq, dim, ffn, block, 0.0f, stream)
                       : lcu_gemm_f16_nt_multi(outs, lhs_dev, w_dev, 2, n_seq, dim, ffn, 0.0f, stream);
  if (rc != LCU_OK) return rc;
  return lcu_silu_mul(out_dev, w1_tmp_dev, w3_tmp_dev, (size_t)n_seq * ffn, stream);
}

int lcu_batch_proj_norm(void* x_dev, void* norm_out_dev, const void* lhs_dev, const void* w_dev, const void* scales_dev,
                        int block, int n_seq, int K, int dim, const void* norm_w_dev, float eps, void* stream) {
  LCU_REQUIRE(x_dev && norm_out_dev && lhs_dev && w_dev && norm_w_dev, "lcu_batch_proj_norm: null pointer");
  LCU_REQUIRE(n_seq >= 0 && dim > 0 && K > 0 && K % 16 == 0 && dim % 2 == 0 && dim <= 24576,
              "lcu_batch_proj_norm: bad shape n_seq %d K %d dim %d", n_seq, K, dim);
  LCU_REQUIRE(block == 0 || (scales_dev && block % 16 == 0 && K % block == 0),
              "lcu_batch_proj_norm: quantised weights need scales and a block dividing K");
  if (n_seq == 0) return LCU_OK;
  hipStream_t st = as_stream(stream);
  bool done = false;
  partial_sums_t ps{};
  if (n_seq > 1 && dim <= RN_THREADS * RN_PAIRS * 2) {
    const operands_t op = single_matrix((half_t*)x_dev, w_dev, (const half_t*)(block ? scales_dev : nullptr));
    const half_t* lhs = (const half_t*)lhs_dev;
    int rc;
    if (n_seq > 64) {
      rc = block ? many_rows_partial<true>(op, lhs, n_seq, K, dim, block, st, &done, &ps) : many_rows_partial<false>(op, lhs, n_seq, K, dim, 0, st, &done, &ps);
    } else {
      const workspace_t ws = workspace_for(st);
      // the norm's launch, a workgroup to a row, then asks for one sum and not eight (8x4096x4096, both launches 14.5 -> 13.1 us)
      const sum_join join{(float*)ws.ptr, dim};
      rc = block ? launch_joined<true>(join, op, lhs, n_seq, K, dim, block, st, nullptr, &done) : launch_joined<false>(join, op, lhs, n_seq, K, dim, 0, st, nullptr, &done);
      if (done) ps = {(float*)ws.ptr, 1};
      if (rc == LCU_OK && !done) rc = block ? skinny_partial<true>(op, lhs, n_seq, K, dim, block, st, &done, &ps) : skinny_partial<false>(op, lhs, n_seq, K, dim, 0, st, &done, &ps);
    }
    if (rc != LCU_OK) return rc;
  }
  if (done) {
    auto kernel = dim <= RN_THREADS * 2 ? reduce_residual_norm_kernel<1> : dim <= RN_THREADS * 4 ? reduce_residual_norm_kernel<2> : reduce_residual_norm_kernel<RN_PAIRS>;
    kernel<<<n_seq, RN_THREADS, (size_t)dim * 2, st>>>((half_t*)x_dev, (half_t*)norm_out_dev, ps.part, ps.splits, n_seq, dim,
                                                       (const half_t*)norm_w_dev, eps);
    LCU_LAUNCH_CHECK();
    return LCU_OK;
  }
  const int rc = block ? lcu_gemm_f16u8_nt(x_dev, lhs_dev, w_dev, scales_dev, n_seq, K, dim, block, 1.0f, stream)
                       : lcu_gemm_f16_nt(x_dev, lhs_dev, w_dev, n_seq, K, dim, 1.0f, stream);
  if (rc != LCU_OK) return rc;
  return lcu_rmsnorm(norm_out_dev, x_dev, norm_w_dev, n_seq, dim, eps, stream);
}

}  // extern "C"
