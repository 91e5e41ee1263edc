// bf16 grouped GEMM for groups of a few rows (a decode step, the shared experts of a small batch): the
// matrices stream straight from memory into MFMA operands, without LDS in between.
//
//   C[rows of e, :] = A[rows of e, :] @ B[e]                          (kDual = false)
//   C = silu(round(A @ B0[e])) * round(A @ B1[e])                     (kDual = true)
//
// Bound: HBM (a matrix element is used by a handful of rows), through what one CU can draw: 50 to 60 GB/s from
// memory and twice that from the L2, however many loads its waves have in flight, so that the chip's 6 TB/s
// take a hundred of its CUs or more.  A launch of the LDS kernels at these sizes has 8 to 100 tiles, and a
// 32-deep step of a tile costs 0.65 us whatever the depth of its pipeline (wait, barrier, LDS reads and
// products of 64 mostly empty rows with one wave per SIMD: 1500 cycles for 16 KB).  Hence here
//   * narrow tiles: 128 / FOLD columns of one matrix, or of each of two (kDual);
//   * a wave owns its loads: a lane fetches 16 bytes (8 columns) of eight consecutive k rows, the wave a block
//     of the matrix as it is stored, and 32 byte permutes turn it into the B operands of eight
//     v_mfma_f32_16x16x32_bf16 (operand j: column 8 (lane % 16) + j, whose eight k values the lane holds);
//   * FOLD = 2: the upper eight of sixteen lanes hold the same columns 32 k rows further on, so that a tile of half
//     the columns still reads whole 128-byte lines.  Operands 0 .. 3 then take columns j of the lower lanes and
//     j + 4 of the upper ones, for either half of the k rows, the other half's values a lane rotation away;
//   * D = 2 blocks of 8 KB are in flight per wave in a ring of registers, up to three workgroups to a CU.  (Four
//     blocks leave room for one workgroup per CU, and longer turns: 10 to 20 % slower throughout; the next
//     blocks requested before the turn instead of in it, with registers for both: as fast with one workgroup to
//     a CU, 5 to 30 % slower with more.)
//   * the four waves of a workgroup (two of them per matrix when kDual) take turns of D blocks on the k range and
//     hand the accumulators on through LDS, so that every sum is ONE chain in k order, as in the LDS kernels: a row's
//     result has the same bits whichever kernel takes it, and does not depend on what shares its call.  (A
//     16x16x32 instruction adds its 32 products as two 32x32x16 ones in a row do: no bit of 2048-deep chains
//     differed on operands of 12, 24 and 48 bits of range.)  A wave turns its blocks into operands before its
//     turn comes, which leaves 8 D products and 16 bytes per lane and accumulator each way in it.
//     The turns cost 0 to 6 % against partial sums of each wave's own (shared experts of 2816 at 64 tokens 36 us
//     against 34, 64 experts at 4 tokens 100 against 100); only tiles of 32 rows and 128 columns, with twice the
//     accumulators to hand on, lost more (gate/up at 256 tokens 6 us) and are gone.
// RB = blocks of 16 rows per tile.  Rows past the end of a group, columns past N and k past K read as zeros.
//
// Requirements: K % 8 == 0, N % 8 == 0, 16-byte aligned pointers, K*N*2 < 2^31, a_rows*K*2 < 2^31.
#pragma once

#include "grouped_gemm_dma.hpp"

namespace jtmoe {

template <int RB_, int FOLD_, bool kDual_>
struct SkinnyCfg {
  static constexpr int RB = RB_, FOLD = FOLD_, BM = 16 * RB, BN = 128 / FOLD, NT = 256, BK = 32 * FOLD;
  static constexpr bool kDual = kDual_;
  static constexpr int D = 2;                                  // blocks per turn, and in flight per wave
  static constexpr int KWAVES = kDual ? 2 : 4;                 // waves that take turns on the k range of a matrix
  static constexpr int NJ = 8 / FOLD;                          // accumulators per 16 rows
  static constexpr int MIN_WAVES_PER_EU = RB == 1 ? 2 : 1;
  static constexpr int GROUP_M = 4;
  static constexpr int SMEM_BYTES = (kDual ? 2 : 1) * RB * NJ * 64 * 16;  // the accumulators of each matrix
  static_assert(FOLD == 1 || FOLD == 2, "columns per tile");
};

struct SkinnyProblem {
  const uint16_t *A, *B0, *B1;
  uint16_t *C, *save0, *save1;  // save0 / save1: the two rounded products of a dual launch, or null
  const int32_t *group_sizes, *offsets;  // null: one group of dense_rows rows
  const int32_t* row_map;  // tile row j reads row row_map[j] / row_div of A (a_rows rows), or null
  int E, dense_rows, Kdim, N, mtiles, ntiles_n, row_div, a_rows;
  int a_group_rows;  // > 0: A holds a block of a_group_rows rows per group, and the map's rows are rows of it
};

template <typename Cfg>
__device__ __forceinline__ void grouped_gemm_skinny_tile(const SkinnyProblem& pr, int block, int launch_blocks) {
  constexpr int RB = Cfg::RB, FOLD = Cfg::FOLD, BM = Cfg::BM, BN = Cfg::BN, BK = Cfg::BK, D = Cfg::D;
  constexpr int LF = 16 / FOLD;  // lanes (of sixteen) that hold different columns
  constexpr bool kDual = Cfg::kDual;
  extern __shared__ __align__(16) unsigned char smem_raw[];

  const int Kdim = pr.Kdim, N = pr.N;
  TileCoord tc;
  TileRows tr;
  if (pr.group_sizes) {
    const GroupScan scan = group_scan(BM, pr.group_sizes, pr.E);
    tc = xcd_tile_order_balanced(scan.total, pr.ntiles_n, Cfg::GROUP_M, block);
    if (tc.mt < 0) return;
    tr = locate_tile(scan, tc.mt, BM, pr.offsets);
  } else {
    tc = xcd_tile_order(pr.mtiles, pr.ntiles_n, Cfg::GROUP_M, block, launch_blocks);
    if (tc.mt < 0) return;
    tr = find_tile_wave(tc.mt, BM, nullptr, nullptr, pr.E, pr.dense_rows);
  }
  tr.expert = __builtin_amdgcn_readfirstlane(tr.expert);
  tr.row0 = __builtin_amdgcn_readfirstlane(tr.row0);
  tr.rows = __builtin_amdgcn_readfirstlane(tr.rows);
  if (tr.rows <= 0) return;
  const int n0 = tc.nt * BN;
  const size_t wofs = (size_t)tr.expert * Kdim * N;

  const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int which = kDual ? wave & 1 : 0, kw = kDual ? wave >> 1 : wave;  // matrix, and share of the k range

  const bool gather = pr.row_map != nullptr;
  const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(pr.A + (gather ? (size_t)tr.expert * pr.a_group_rows : (size_t)tr.row0) * Kdim), 0,
      (gather ? pr.a_rows : tr.rows) * Kdim * 2, kBufferFlags);
  const __amdgpu_buffer_rsrc_t b_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>((which ? pr.B1 : pr.B0) + wofs), 0, Kdim * N * 2, kBufferFlags);
  int a_voff[RB];
#pragma unroll
  for (int b = 0; b < RB; ++b) {
    const int r = b * 16 + c16;
    const int src = gather && r < tr.rows ? pr.row_map[tr.row0 + r] / pr.row_div : r;
    a_voff[b] = r < tr.rows ? (src * Kdim + g * 8) * 2 : kOutside;
  }
  const int col = n0 + c16 % LF * 8, b_k = c16 / LF * 32 + g * 8;  // this lane's columns, and first k row of a block
  const int b_voff = col < N ? (b_k * N + col) * 2 : kOutside;

  constexpr int KW = Cfg::KWAVES, NJ = Cfg::NJ;
  const int blocks = (Kdim + BK - 1) / BK;
  const int rounds = (blocks + KW * D - 1) / (KW * D);  // turns of every wave

  u32x4_t b_ring[D][8], a_ring[D][FOLD][RB];
  // Every load is issued on every path (a block past the end, like a chunk past the end of K, takes an offset
  // outside the operand: zeros, no traffic), so that the compiler's wait counts stay exact: with the loads of the
  // last blocks behind a branch it waits for all loads in flight in front of every block.
  auto load = [&](int slot, int block) {
    const int k0 = block < blocks ? block * BK : 0;
    const int k_end = block < blocks ? Kdim - k0 : 0;  // k rows from k0 on
#pragma unroll
    for (int f = 0; f < FOLD; ++f)
#pragma unroll
      for (int b = 0; b < RB; ++b)
        a_ring[slot][f][b] = __builtin_amdgcn_raw_buffer_load_b128(
            a_rsrc, f * 32 + g * 8 >= k_end ? kOutside : a_voff[b], (k0 + f * 32) * 2, 0);
#pragma unroll
    for (int r = 0; r < 8; ++r)  // non-temporal: few other workgroups read these bytes
      b_ring[slot][r] = __builtin_amdgcn_raw_buffer_load_b128(b_rsrc, b_k >= k_end ? kOutside : b_voff, (k0 + r) * N * 2, 2);
  };
  // operand jj for k half f of the block in `slot`: column 8 (c16 % LF) + jj (+ 4 in the upper lanes of a folded one)
  auto operand = [&](int slot, int j) {
    u32x4_t v;
#pragma unroll
    for (int p = 0; p < 4; ++p)  // k = 8 g + 2 p (low half) and 2 p + 1 of column j of the lane's eight
      v[p] = __builtin_amdgcn_perm(b_ring[slot][2 * p + 1][j / 2], b_ring[slot][2 * p][j / 2],
                                   j % 2 ? 0x07060302u : 0x05040100u);
    return v;
  };
  u32x4_t frag[D][FOLD][NJ];
  auto prepare = [&](int slot) {
#pragma unroll
    for (int jj = 0; jj < NJ; ++jj) {
      const u32x4_t lo = operand(slot, jj);
      if constexpr (FOLD == 1) {
        frag[slot][0][jj] = lo;
      } else {
        const u32x4_t hi = operand(slot, jj + 4);
#pragma unroll
        for (int p = 0; p < 4; ++p) {  // rotations by 8 of 16 lanes, into the upper eight and into the lower eight
          frag[slot][0][jj][p] = __builtin_amdgcn_update_dpp(lo[p], hi[p], 0x128, 0xf, 0xc, false);
          frag[slot][FOLD - 1][jj][p] = __builtin_amdgcn_update_dpp(hi[p], lo[p], 0x128, 0xf, 0x3, false);
        }
      }
    }
  };
  typedef __attribute__((ext_vector_type(4))) float f32x4;
  f32x4* const sums = reinterpret_cast<f32x4*>(smem_raw);  // [matrix][16-row block][operand][lane]
  f32x4* const mine = sums + which * (RB * NJ * 64) + lane;
  auto turn_ends = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  if (kw == 0)
#pragma unroll
    for (int i = 0; i < RB * NJ; ++i) mine[i * 64] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int d = 0; d < D; ++d) {
    load(d, kw * D + d);
    __builtin_amdgcn_sched_barrier(0);
  }
  for (int round = 0; round < rounds; ++round) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      prepare(d);
      __builtin_amdgcn_sched_barrier(0);  // (one block's operands at a time: mixed, they do not fit the registers)
    }
    for (int w = 0; w < kw; ++w) turn_ends();  // the waves before this one
    f32x4 acc[RB][NJ];
#pragma unroll
    for (int i = 0; i < RB * NJ; ++i) acc[i / NJ][i % NJ] = mine[i * 64];
#pragma unroll
    for (int d = 0; d < D; ++d) {  // (blocks past the end multiply zeros)
#pragma unroll
      for (int f = 0; f < FOLD; ++f)
#pragma unroll
        for (int b = 0; b < RB; ++b)
#pragma unroll
          for (int jj = 0; jj < NJ; ++jj)
            acc[b][jj] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a_ring[d][f][b]),
                                                                 __builtin_bit_cast(bf16x8_t, frag[d][f][jj]), acc[b][jj], 0, 0, 0);
      load(d, ((round + 1) * KW + kw) * D + d);
      __builtin_amdgcn_sched_barrier(0);  // (else the loads of all D blocks gather at the end of the loop body)
    }
#pragma unroll
    for (int i = 0; i < RB * NJ; ++i) mine[i * 64] = acc[i / NJ][i % NJ];
    for (int w = kw; w < KW; ++w) turn_ends();  // this wave, and those behind it
  }

  // value i of lane (c16, g) of accumulator (b, jj) is row 16 b + 4 g + i, column 8 (c16 % LF) + jj (+ 4 in the
  // upper lanes of a folded tile)
  const float* const values = reinterpret_cast<const float*>(smem_raw);
  for (int c = tid; c < BM * (BN / 8); c += Cfg::NT) {  // one 16-byte piece of a result row per thread
    const int r = c / (BN / 8), q = c - r * (BN / 8), c8 = q * 8;
    if (r >= tr.rows || n0 + c8 >= N) continue;
    const float* p = values + ((r / 16) * NJ * 64 + r % 16 / 4 * 16 + q) * 4 + r % 4;
    float v[2][8];  // the two products, or the only one
#pragma unroll
    for (int m = 0; m < (kDual ? 2 : 1); ++m)
#pragma unroll
      for (int j = 0; j < 8; ++j) v[m][j] = p[(m * RB * NJ * 64 + j % NJ * 64 + j / NJ * LF) * 4];
    const size_t at = (size_t)(tr.row0 + r) * N + n0 + c8;
    auto store8 = [&](uint16_t* out, const float* f) {
      const u32x4_t q = {pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3]), pack_bf16x2(f[4], f[5]), pack_bf16x2(f[6], f[7])};
      *reinterpret_cast<u32x4_t*>(out + at) = q;
    };
    if (kDual) {
      float h[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float gate = bf16_round_fast(v[0][j]);
        h[j] = (Kdim % 64 != 0 ? silu_gate<true>(gate) : silu_gate<false>(gate)) * bf16_round_fast(v[1][j]);
      }
      store8(pr.C, h);
      if (pr.save0) {
        store8(pr.save0, v[0]);
        store8(pr.save1, v[1]);
      }
    } else {
      store8(pr.C, v[0]);
    }
  }
}

template <typename Cfg>
__global__ __launch_bounds__(Cfg::NT) __attribute__((amdgpu_waves_per_eu(Cfg::MIN_WAVES_PER_EU))) void grouped_gemm_skinny_kernel(
    SkinnyProblem p) {
  grouped_gemm_skinny_tile<Cfg>(p, (int)blockIdx.x, (int)gridDim.x);
}

// The shared experts' down product of a few tokens beside a routed product: its tiles are the launch's first
// beside_blocks workgroups.  Neither needs the other's result, and either alone leaves CUs or bandwidth idle.
using BesideCfg = SkinnyCfg<1, 2, false>;
struct Beside {
  SkinnyProblem p;
  int blocks;  // a multiple of 8
};

template <typename Cfg>
__global__ __launch_bounds__(Cfg::NT) __attribute__((amdgpu_waves_per_eu(Cfg::MIN_WAVES_PER_EU))) void grouped_gemm_skinny_beside_kernel(
    SkinnyProblem p, Beside beside) {
  if ((int)blockIdx.x < beside.blocks)
    grouped_gemm_skinny_tile<BesideCfg>(beside.p, (int)blockIdx.x, beside.blocks);
  else
    grouped_gemm_skinny_tile<Cfg>(p, (int)blockIdx.x - beside.blocks, (int)gridDim.x - beside.blocks);
}

// (three workgroups per CU: the streaming tile takes more registers than the 64-row one)
template <typename Cfg>
__global__ __launch_bounds__(Cfg::NT) __attribute__((amdgpu_waves_per_eu(3))) void grouped_gemm_dma_beside_kernel(
    const uint16_t* __restrict__ A, const uint16_t* __restrict__ B0, const uint16_t* __restrict__ B1,
    uint16_t* __restrict__ C, const int32_t* __restrict__ group_sizes, const int32_t* __restrict__ offsets, int E,
    int rows, int Kdim, int N, int mtiles, int ntiles_n, const int32_t* __restrict__ row_map, int row_div, int a_rows,
    uint16_t* __restrict__ save0, uint16_t* __restrict__ save1, int a_group_rows, Beside beside) {
  if ((int)blockIdx.x < beside.blocks)
    grouped_gemm_skinny_tile<BesideCfg>(beside.p, (int)blockIdx.x, beside.blocks);
  else
    grouped_gemm_dma_tile<Cfg>(A, B0, B1, C, group_sizes, offsets, E, rows, Kdim, N, mtiles, ntiles_n, row_map, row_div,
                               a_rows, save0, save1, 0, a_group_rows, (int)blockIdx.x - beside.blocks,
                               (int)gridDim.x - beside.blocks);
}

// One dense group of T rows.
inline SkinnyProblem dense_skinny(const void* a, const void* b0, const void* b1, void* c, void* save0, void* save1,
                                  int64_t T, int64_t Kdim, int64_t N, int BM, int BN) {
  return SkinnyProblem{static_cast<const uint16_t*>(a), static_cast<const uint16_t*>(b0),
                       static_cast<const uint16_t*>(b1), static_cast<uint16_t*>(c), static_cast<uint16_t*>(save0),
                       static_cast<uint16_t*>(save1), nullptr, nullptr, nullptr, 1, (int)T, (int)Kdim, (int)N,
                       (int)((T + BM - 1) / BM), (int)((N + BN - 1) / BN), 1, 0, 0};
}

}  // namespace jtmoe
