// Single-precision grouped GEMMs on v_mfma_f32_32x32x2_f32 (inputs, sums and results in fp32):
//
//   "NN"  C[rows of e, :] = A[rows of e, :] @ B[e]            B[e] [K, N]      (forward products; kDual: gate and
//         up share the A tile and the SwiGLU runs in the epilogue)
//   "NT"  C[rows of e, :] = sum over segments A_s[rows of e, :] @ B_s[e]^T,    B_s[e] [N, K]   (data gradients)
//   "TN"  C[e] = P[rows of e, :]^T @ D[rows of e, :]                           (weight gradients)
//
// Bound: the fp32 matrix rate (157 TFLOP/s: 64 cycles per 32 x 32 x 2 product), sixteen times below bf16's, so
// operand traffic is cheap by comparison and the design only has to keep every SIMD's matrix core busy: four
// waves (2 x 2) per workgroup, 32-deep k steps, two LDS stages filled by buffer_load ... lds while the other is
// multiplied, and two to four workgroups per CU so that one's barrier runs under another's products.  A step
// of a 64 x 64 wave tile is 4096 matrix cycles against 16 ds_read_b128 and 64 ds_read_b32.
// k-contiguous tiles (A, and B of NT) hold rows of eight 16-byte chunks, chunk c of row r in slot
// c ^ ((r / 2) % 8), and one ds_read_b128 feeds four MFMAs (lane half h takes k = 8 q + 4 h + i in product i:
// any assignment of k to products serves as long as both operands use it).  Row-major tiles ([k][n]) are read
// one word per MFMA, 32 consecutive words per half wave.
// Two tile heights and widths (128 and 64): the launcher takes the one with the fewer rounds over the CUs.
// Three stages instead of two measured the same (46.4 against 45.6 us for a product of 4096 rows in one group, K = 1024,
// N = 512): the loads arrive in time, and the LDS is better spent on more workgroups per CU.
// What costs rate beside the products, and what is done about it in the two forms with a row per group row:
//   - the accumulators have to stay where they are.  A wave that skips its products inside the step loop makes the
//     compiler carry them through ordinary registers, a write and a read of each per step: 16 to 64 writes among 16 to 64
//     products.  The waves without rows have a loop of their own instead (4096 rows in one group, K = 4096, N = 512:
//     168.9 -> 162.5 us; gate/up with K = 2048, N = 1024: 270.7 -> 253.4).
//   - the first fragments of a step are requested in front of the last products of the one before (162.5 -> 159.8).
//   - 64-row tiles, whose steps are short: the loads lie between those products.  In one piece behind the barrier the
//     loads of all waves queue up and hold the products back (159.8 -> 150.9).  In the tiles with four blocks per wave
//     that costs 2 % (gate/up above 253 -> 259).
// Measured at 4096 rows in 8 groups, 512 x 1024: gate/up 100.5 -> 95.4 us, down 60.8 -> 56.1, data gradients 54.2 -> 52.1
// and 114.6 -> 107.9, weight gradients 47 and 83 in launches of their own; the element-wise staged kernels, which still take other
// widths, 143 to 424.  What is left is the last, partly filled round (2.1 rounds of tiles for the down product) and
// the fixed cost of launches this short; with long reductions the large tiles reach 136 TFLOP/s of the 154 that the
// matrix cores reach from registers.
//
// Requirements: K, N (KA) multiples of 4, 16-byte aligned pointers, operands of a group below 2 GiB.
#pragma once

#include "grouped_gemm_dma.hpp"

namespace jtmoe {

template <int BM_, int BN_, bool kDual_, bool kBT_>
struct F32Cfg {
  static constexpr int BM = BM_, BN = BN_, BK = 32, NT = 256;
  static constexpr bool kDual = kDual_, kBT = kBT_;
  static constexpr int NSUB = kDual ? 2 : 1;           // matrices per B tile
  static constexpr int TM = BM / 64, TN = NSUB * BN / 64;  // 32 x 32 blocks per wave
  static constexpr int A_BYTES = BM * BK * 4, B_BYTES = BN * BK * 4;
  static constexpr int STAGE_BYTES = A_BYTES + NSUB * B_BYTES;
  static constexpr int SMEM_BYTES = 2 * STAGE_BYTES;
  static constexpr int A_LOADS = BM * 8 / NT, B_LOADS = BN * 8 / NT;
  static constexpr int GROUP_M = 4;
  static constexpr bool kSpread = BM == 64;  // the loads lie between the products
  static_assert(BM % 64 == 0 && BN % 64 == 0 && !(kDual && (kBT || BN != 64)), "2 x 2 waves of 32 x 32 blocks");
};

// 16 bytes per lane into LDS at base + lane * 16; the whole offset in the vector part (ends of rows and
// matrices are recognised by the descriptor's bound)
__device__ __forceinline__ void f32_load(i32x4_t rsrc, unsigned base, int voffset) {
  buffer_load_lds16(rsrc, base, voffset, 0);
}

// (block / blocks: this workgroup's index among those that share out the tiles, and their number, a multiple of 8)
template <typename Cfg>
__device__ __forceinline__ void f32_rows_body(
    int block, int blocks, unsigned char* smem_raw, const float* __restrict__ A0, const float* __restrict__ A1,
    const float* __restrict__ B0, const float* __restrict__ B1, float* __restrict__ C,
    const int32_t* __restrict__ group_sizes, const int32_t* __restrict__ offsets, int E, int dense_rows, int Kdim, int N,
    int mtiles, int ntiles_n, const int32_t* __restrict__ row_map, int row_div, int a_rows, int segs,
    float* __restrict__ save0, float* __restrict__ save1) {
  constexpr int BM = Cfg::BM, BN = Cfg::BN, BK = Cfg::BK, NT = Cfg::NT, TM = Cfg::TM, TN = Cfg::TN;
  constexpr bool kDual = Cfg::kDual, kBT = Cfg::kBT;

  TileCoord tc;
  TileRows tr;
  if (group_sizes) {
    const GroupScan scan = group_scan(BM, group_sizes, E);
    tc = xcd_tile_order_balanced(scan.total, ntiles_n, Cfg::GROUP_M, block);
    if (tc.mt < 0) return;
    tr = locate_tile(scan, tc.mt, BM, offsets);
  } else {
    tc = xcd_tile_order(mtiles, ntiles_n, Cfg::GROUP_M, block, blocks);
    if (tc.mt < 0) return;
    tr = find_tile_wave(tc.mt, BM, nullptr, nullptr, E, dense_rows);
  }
  tr.expert = __builtin_amdgcn_readfirstlane(tr.expert);
  tr.row0 = __builtin_amdgcn_readfirstlane(tr.row0);
  tr.rows = __builtin_amdgcn_readfirstlane(tr.rows);
  if (tr.rows <= 0) return;
  const int n0 = tc.nt * BN;
  const size_t wofs = (size_t)tr.expert * Kdim * N;

  const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const bool gather = row_map != nullptr;

  // ---- load plan ----
  const i32x4_t a_rsrc0 = gather ? make_rsrc(A0, a_rows * Kdim * 4) : make_rsrc(A0 + (size_t)tr.row0 * Kdim, tr.rows * Kdim * 4);
  const i32x4_t a_rsrc1 = segs > 1 ? make_rsrc(A1 + (size_t)tr.row0 * Kdim, tr.rows * Kdim * 4) : a_rsrc0;
  const i32x4_t b_rsrc0 = make_rsrc(B0 + wofs, Kdim * N * 4);
  const i32x4_t b_rsrc1 = (kDual || segs > 1) ? make_rsrc(B1 + wofs, Kdim * N * 4) : b_rsrc0;
  // k-contiguous tiles: load j of this thread is row l_r + 32 j, source chunk l_c
  const int l_r = tid >> 3, l_c = (tid & 7) ^ ((l_r >> 1) & 7);
  int a_voff[Cfg::A_LOADS];
#pragma unroll
  for (int j = 0; j < Cfg::A_LOADS; ++j) {
    const int r = l_r + j * 32;
    const int src = gather && r < tr.rows ? row_map[tr.row0 + r] / row_div : r;
    a_voff[j] = r < tr.rows ? (src * Kdim + l_c * 4) * 4 : kOutside;
  }
  int b_voff[Cfg::B_LOADS];
#pragma unroll
  for (int j = 0; j < Cfg::B_LOADS; ++j) {
    const int c = tid + j * NT;
    b_voff[j] = kBT ? ((n0 + l_r + j * 32) * Kdim + l_c * 4) * 4 : (c / (BN / 4) * N + n0 + c % (BN / 4) * 4) * 4;
  }
  const unsigned wave_lds = lds_byte_addr(smem_raw) + wave * 1024;
  const int nk1 = (Kdim + BK - 1) / BK, nk = max(nk1 * segs, 1);
  constexpr int LOADS = Cfg::A_LOADS + Cfg::NSUB * Cfg::B_LOADS;
  // load `i` of step kt; past the last step everything lies outside and reads as zeros
  auto issue = [&](int kt, int i) {
    const unsigned base = __builtin_amdgcn_readfirstlane(wave_lds + (kt & 1) * Cfg::STAGE_BYTES);
    const bool second = kt >= nk1;
    const int k0 = (second ? kt - nk1 : kt) * BK;
    const bool past_k = kt >= nk || k0 + l_c * 4 >= Kdim;  // this lane's chunk lies past the end of a row
    if (i < Cfg::A_LOADS) {
      f32_load(second ? a_rsrc1 : a_rsrc0, base + i * NT * 16, past_k ? kOutside : a_voff[i] + k0 * 4);
      return;
    }
    const int u = (i - Cfg::A_LOADS) / Cfg::B_LOADS, j = (i - Cfg::A_LOADS) % Cfg::B_LOADS;
    const unsigned to = base + Cfg::A_BYTES + u * Cfg::B_BYTES + j * NT * 16;
    if (kBT)
      f32_load(second ? b_rsrc1 : b_rsrc0, to, past_k ? kOutside : b_voff[j] + k0 * 4);
    else
      f32_load(u ? b_rsrc1 : b_rsrc0, to, kt >= nk ? kOutside : b_voff[j] + k0 * N * 4);
  };

  f32x16_t acc[TM][TN];
#pragma unroll
  for (int mi = 0; mi < TM; ++mi)
#pragma unroll
    for (int jj = 0; jj < TN; ++jj)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[mi][jj][i] = 0.0f;

  typedef float f32x4 __attribute__((ext_vector_type(4)));
  const int sw = ((lane & 31) >> 1) & 7;
  const int a_off = (wm * 32 * TM + (lane & 31)) * (BK * 4);
  const int bt_off = Cfg::A_BYTES + (wn * 32 * TN + (lane & 31)) * (BK * 4);
  // fragments of an 8-deep sub-step: value i of this lane belongs to k = 8 q + 4 half + i
  auto load_frags = [&](const unsigned char* st, int q, f32x4* a, f32x4* b) {
    const int chunk = ((2 * q + half) ^ sw) << 4;
#pragma unroll
    for (int mi = 0; mi < TM; ++mi)
      a[mi] = *reinterpret_cast<const f32x4*>(st + a_off + mi * 32 * BK * 4 + chunk);
#pragma unroll
    for (int jj = 0; jj < TN; ++jj) {
      if constexpr (kBT) {
        b[jj] = *reinterpret_cast<const f32x4*>(st + bt_off + jj * 32 * BK * 4 + chunk);
      } else {
        const int u = kDual ? jj : 0, col = (kDual ? wn : wn * TN + jj) * 32 + (lane & 31);
        const float* p = reinterpret_cast<const float*>(st + Cfg::A_BYTES + u * Cfg::B_BYTES) + (8 * q + 4 * half) * BN + col;
#pragma unroll
        for (int i = 0; i < 4; ++i) b[jj][i] = p[i * BN];
      }
    }
  };
  // (the scheduling barriers keep the fragments' requests in front of the products, under which they arrive, and spread
  // loads between them)
  f32x4 a[2][TM], b[2][TN];
  auto products = [&](int set, bool loads, int kt) {  // with `loads`: and the loads of step kt
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int mi = 0; mi < TM; ++mi)
#pragma unroll
        for (int jj = 0; jj < TN; ++jj)
          acc[mi][jj] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[set][mi][i], b[set][jj][i], acc[mi][jj], 0, 0, 0);
      if (loads) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = LOADS * i / 4; j < LOADS * (i + 1) / 4; ++j) issue(kt, j);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr int QS = BK / 8;
#pragma unroll
  for (int i = 0; i < LOADS; ++i) issue(0, i);
  wait_and_barrier<0>();
#pragma unroll
  for (int i = 0; i < LOADS; ++i) issue(1, i);
  if (wm * 32 * TM >= tr.rows) {  // rows past the end of the group: loads and barriers only
    for (int kt = 0; kt + 1 < nk; ++kt) {
      wait_and_barrier<0>();
#pragma unroll
      for (int i = 0; i < LOADS; ++i) issue(kt + 2, i);
    }
    wait_vmcnt<0>();
    return;
  }
  load_frags(smem_raw, 0, a[0], b[0]);
  for (int kt = 0; kt + 1 < nk; ++kt) {
    const unsigned char* st = smem_raw + (kt & 1) * Cfg::STAGE_BYTES;
#pragma unroll
    for (int q = 0; q < QS - 1; ++q) {
      load_frags(st, q + 1, a[(q + 1) & 1], b[(q + 1) & 1]);
      products(q & 1, false, 0);
    }
    // all waves have read stage kt and their loads of stage kt + 1 are there: its first fragments are on their way
    // while the last products of this step run
    wait_and_barrier<0>();
    if (!Cfg::kSpread && kt + 2 < nk) {
#pragma unroll
      for (int i = 0; i < LOADS; ++i) issue(kt + 2, i);
    }
    load_frags(smem_raw + ((kt + 1) & 1) * Cfg::STAGE_BYTES, 0, a[0], b[0]);
    products((QS - 1) & 1, Cfg::kSpread, kt + 2);
  }
  {
    const unsigned char* st = smem_raw + ((nk - 1) & 1) * Cfg::STAGE_BYTES;
#pragma unroll
    for (int q = 0; q < QS; ++q) {
      if (q + 1 < QS) load_frags(st, q + 1, a[(q + 1) & 1], b[(q + 1) & 1]);
      products(q & 1, false, 0);
    }
  }
  wait_vmcnt<0>();  // the loads past the last step

  // value i of lane l of a block is row 8 (i / 4) + 4 (l / 32) + i % 4, column l % 32: the 32 lanes of a
  // half wave store 128 contiguous bytes
#pragma unroll
  for (int mi = 0; mi < TM; ++mi)
#pragma unroll
    for (int jj = 0; jj < (kDual ? 1 : TN); ++jj) {
      const int col = n0 + (kDual ? wn : wn * TN + jj) * 32 + (lane & 31);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int r = (wm * TM + mi) * 32 + 8 * (i >> 2) + 4 * half + (i & 3);
        if (r < tr.rows && col < N) {
          const size_t at = (size_t)(tr.row0 + r) * N + col;
          if constexpr (kDual) {
            const float g = acc[mi][0][i], u = acc[mi][1][i];
            C[at] = silu_fast(g) * u;
            if (save0) {
              save0[at] = g;
              save1[at] = u;
            }
          } else {
            C[at] = acc[mi][jj][i];
          }
        }
      }
    }
}

template <typename Cfg>
__global__ __launch_bounds__(Cfg::NT) void grouped_gemm_f32_kernel(
    const float* __restrict__ A0, const float* __restrict__ A1, const float* __restrict__ B0,
    const float* __restrict__ B1, float* __restrict__ C, const int32_t* __restrict__ group_sizes,
    const int32_t* __restrict__ offsets, int E, int dense_rows, int Kdim, int N, int mtiles, int ntiles_n,
    const int32_t* __restrict__ row_map, int row_div, int a_rows, int segs, float* __restrict__ save0,
    float* __restrict__ save1) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  f32_rows_body<Cfg>((int)blockIdx.x, (int)gridDim.x, smem_raw, A0, A1, B0, B1, C, group_sizes, offsets, E, dense_rows,
                     Kdim, N, mtiles, ntiles_n, row_map, row_div, a_rows, segs, save0, save1);
}

// Weight gradients.  One workgroup per (matrix, group, tile); D1 / C1 (if `matrices` is 2) is a second
// product with the same P.  split_chunk > 0 (one dense group): "group" e is the e-th run of split_chunk rows
// and C holds partial sums [matrix][E][KA, N] that the caller adds up in order.
template <int BMO, int BNO>
__device__ __forceinline__ void f32_tn_body(int block, unsigned char* smem_raw, const float* __restrict__ P,
                                            const float* __restrict__ D0, const float* __restrict__ D1,
                                            float* __restrict__ C0, float* __restrict__ C1,
                                            const int32_t* __restrict__ group_sizes, const int32_t* __restrict__ offsets,
                                            int E, int dense_rows, int KA, int N, int mtiles_o, int ntiles_o,
                                            int split_chunk) {
  constexpr int BK = 32, NT = 256, TM = BMO / 64, TN = BNO / 64;
  constexpr int P_BYTES = BK * BMO * 4, STAGE_BYTES = P_BYTES + BK * BNO * 4;
  const int per_group = mtiles_o * ntiles_o;
  const int which = block / (E * per_group);
  block -= which * E * per_group;
  const int e = block / per_group;
  const int in_e = block - e * per_group;
  const int nt = in_e / mtiles_o, m0 = (in_e - nt * mtiles_o) * BMO, n0 = nt * BNO;
  int row0 = 0, rows = dense_rows;
  if (group_sizes) {
    row0 = __builtin_amdgcn_readfirstlane(offsets[e]);
    rows = __builtin_amdgcn_readfirstlane(group_sizes[e]);
  } else if (split_chunk > 0) {
    row0 = e * split_chunk;
    rows = max(0, min(split_chunk, dense_rows - row0));
  }
  const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  // rows past the end of the group lie outside the descriptors and read as zeros
  const i32x4_t p_rsrc = make_rsrc(P + (size_t)row0 * KA, rows * KA * 4);
  const i32x4_t d_rsrc = make_rsrc((which ? D1 : D0) + (size_t)row0 * N, rows * N * 4);
  const unsigned wave_lds = lds_byte_addr(smem_raw) + wave * 1024;
  auto issue = [&](int kt) {
    const unsigned base = wave_lds + (kt & 1) * STAGE_BYTES;
#pragma unroll
    for (int j = 0; j < BMO / 32; ++j) {
      const int s = tid + j * NT, k = s / (BMO / 4), c = s % (BMO / 4);
      f32_load(p_rsrc, base + j * NT * 16, ((kt * BK + k) * KA + m0 + c * 4) * 4);
    }
#pragma unroll
    for (int j = 0; j < BNO / 32; ++j) {
      const int s = tid + j * NT, k = s / (BNO / 4), c = s % (BNO / 4);
      f32_load(d_rsrc, base + P_BYTES + j * NT * 16, ((kt * BK + k) * N + n0 + c * 4) * 4);
    }
  };
  f32x16_t acc[TM][TN];
#pragma unroll
  for (int mi = 0; mi < TM; ++mi)
#pragma unroll
    for (int jj = 0; jj < TN; ++jj)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[mi][jj][i] = 0.0f;
  const int nk = (rows + BK - 1) / BK;
  if (nk > 0) issue(0);
  for (int kt = 0; kt < nk; ++kt) {
    wait_vmcnt<0>();
    __syncthreads();
    if (kt + 1 < nk) issue(kt + 1);
    const float* ps = reinterpret_cast<const float*>(smem_raw + (kt & 1) * STAGE_BYTES) + half * BMO + wm * 32 * TM + (lane & 31);
    const float* ds = reinterpret_cast<const float*>(smem_raw + (kt & 1) * STAGE_BYTES + P_BYTES) + half * BNO + wn * 32 * TN + (lane & 31);
    // two k rows (one per half wave) per product, four products' worth of fragments ahead
    constexpr int KS = 4;
    float a[2][KS][TM], b[2][KS][TN];
    auto load_frags = [&](int set, int k2) {
#pragma unroll
      for (int i = 0; i < KS; ++i) {
#pragma unroll
        for (int mi = 0; mi < TM; ++mi) a[set][i][mi] = ps[2 * (k2 + i) * BMO + mi * 32];
#pragma unroll
        for (int jj = 0; jj < TN; ++jj) b[set][i][jj] = ds[2 * (k2 + i) * BNO + jj * 32];
      }
    };
    load_frags(0, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < BK / 2 / KS; ++g) {
      if (g + 1 < BK / 2 / KS) load_frags((g + 1) & 1, (g + 1) * KS);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < KS; ++i)
#pragma unroll
        for (int mi = 0; mi < TM; ++mi)
#pragma unroll
          for (int jj = 0; jj < TN; ++jj)
            acc[mi][jj] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[g & 1][i][mi], b[g & 1][i][jj], acc[mi][jj], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  float* const Ce = (which ? C1 : C0) + (size_t)e * KA * N;
#pragma unroll
  for (int mi = 0; mi < TM; ++mi)
#pragma unroll
    for (int jj = 0; jj < TN; ++jj) {
      const int col = n0 + (wn * TN + jj) * 32 + (lane & 31);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int r = m0 + (wm * TM + mi) * 32 + 8 * (i >> 2) + 4 * half + (i & 3);
        if (r < KA && col < N) Ce[(size_t)r * N + col] = acc[mi][jj][i];
      }
    }
}

template <int BMO, int BNO>
__global__ __launch_bounds__(256) void grouped_gemm_f32_tn_kernel(
    const float* __restrict__ P, const float* __restrict__ D0, const float* __restrict__ D1, float* __restrict__ C0,
    float* __restrict__ C1, const int32_t* __restrict__ group_sizes, const int32_t* __restrict__ offsets, int E,
    int dense_rows, int KA, int N, int mtiles_o, int ntiles_o, int split_chunk) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  f32_tn_body<BMO, BNO>((int)blockIdx.x, smem_raw, P, D0, D1, C0, C1, group_sizes, offsets, E, dense_rows, KA, N,
                        mtiles_o, ntiles_o, split_chunk);
}

// The three products behind the SwiGLU's backward pass, none of which needs another's result, in one launch of 64 x 64
// tiles: dXp = dG Wg^T + dU Wu^T first, whose tiles are the longest, then dWg = Xp^T dG, dWu = Xp^T dU and
// dWd = HW^T dYp.  Launches of their own each end in a round that is partly empty: at 4096 rows in 8 groups, 512 x 1024,
// 108 + 83 + 47 us (2.1 rounds of tiles for dXp, and two and one of the large tiles of the weight gradients at 102 and
// 92 TFLOP/s), 192 us in one.
struct F32BackwardProducts {
  const float *dg, *du, *hw, *xp, *dyp, *gate, *up;  // [rows, I] x 3, [rows, H] x 2, [E, H, I] x 2
  float *dxp, *d_gate, *d_up, *d_down;               // [rows, H], [E, H, I] x 2, [E, I, H]
  const int32_t *group_sizes, *offsets;
  int rows, H, I, E, mtiles, dx_blocks;  // m-tiles and workgroups of dXp
};

__global__ __launch_bounds__(256) void grouped_gemm_f32_backward_kernel(F32BackwardProducts p) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int th = (p.H + 63) / 64, ti = (p.I + 63) / 64, per_matrix = p.E * th * ti;
  int block = (int)blockIdx.x;
  if (block < p.dx_blocks) {
    f32_rows_body<F32Cfg<64, 64, false, true>>(block, p.dx_blocks, smem_raw, p.dg, p.du, p.gate, p.up, p.dxp,
                                               p.group_sizes, p.offsets, p.E, p.rows, p.I, p.H, p.mtiles, th, nullptr, 1,
                                               0, 2, nullptr, nullptr);
    return;
  }
  block -= p.dx_blocks;
  const bool down = block >= 2 * per_matrix;
  f32_tn_body<64, 64>(down ? block - 2 * per_matrix : block, smem_raw, down ? p.hw : p.xp, down ? p.dyp : p.dg, p.du,
                      down ? p.d_down : p.d_gate, p.d_up, p.group_sizes, p.offsets, p.E, p.rows, down ? p.I : p.H,
                      down ? p.H : p.I, down ? ti : th, down ? th : ti, 0);
}

}  // namespace jtmoe
