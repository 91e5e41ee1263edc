// The grouped bf16 GEMM of grouped_gemm_dma.hpp (same tiles, same LDS layouts, same LDS-DMA operand
// loads) as ONE software pipeline that runs through all the tiles of a workgroup:
//
//   * NSTAGE operand stages are in flight.  The loads of k step c + NSTAGE are issued during step c,
//     as soon as the stage they overwrite has been read for the last time, so a load has NSTAGE - 1
//     steps to arrive instead of one, and the wait in front of the barrier (s_waitcnt vmcnt(n),
//     n > 0) leaves the younger stages in flight.
//   * The barrier of a step stands before its LAST 16-deep sub-step, and guarantees the NEXT step's
//     stage: the first fragments of step c + 1 are read from LDS while the matrix cores work on the
//     last sub-step of step c, so no wave starts a step by waiting for LDS.
//   * The stream of k steps does not stop at the end of a tile: the loads of the next tile's first
//     steps are issued during the last steps of the current one.  The epilogue writes the accumulators
//     straight to memory (they hold transposed blocks, so a lane owns runs of neighbouring columns):
//     no LDS, no barrier.
//   * A tile takes up to 64 rows beyond BM (OPT & 131072) where that spares tiles: a fifth block of 32
//     rows per wave, one more operand load per stage, read and multiplied only by the tiles that have
//     such rows.  The accumulators are then 160 of a wave's 256 registers.
//   * Nothing in the steady state returns data to vector registers through the memory pipe (the
//     row map of the next tile arrives by LDS-DMA as well, group sizes and offsets are read from a copy
//     in LDS), so the compiler never inserts a wait that drains the operand loads.
//
// Requirements: those of grouped_gemm_dma.hpp, K % BK == 0 unless OPT & 65536, K / BK >= 2 * NSTAGE (fills_pipeline: with a
// row map the next tile's has arrived after NSTAGE - 1 of the steps in front of the last NSTAGE), a result of at most 0x7ffe0000
// bytes, with a row map fewer than 2^27 rows and row_div <= 32; launch with a multiple of 8 workgroups
// (persistent schedule).
#pragma once

#include "grouped_gemm_dma.hpp"

#include <type_traits>

namespace jtmoe {

// 4 bytes per lane from a raw buffer into LDS at lds_base + lane * 4 (zeros past the end)
__device__ __forceinline__ void buffer_load_lds4(i32x4_t rsrc, unsigned lds_base, int voffset) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds"
               :
               : "s"(lds_base), "v"(voffset), "s"(rsrc)
               : "memory", "m0");
}

template <typename Cfg>
struct StreamLayout {
  static constexpr int kRowBufBytes = Cfg::NT * 4;
  static constexpr int kPipeBytes = Cfg::NSTAGE * Cfg::STAGE_BYTES;
  static constexpr int kRowBufBase = kPipeBytes;
  static constexpr int kGroupBase = kRowBufBase + kRowBufBytes;  // group sizes, then first rows: 2 x JTMOE_MAX_EXPERTS ints
  static constexpr int kSmemBytes = kGroupBase + 2 * JTMOE_MAX_EXPERTS * 4;
  static_assert(kSmemBytes <= 160 * 1024, "LDS budget");
  static_assert(Cfg::BM + Cfg::XROWS <= Cfg::NT, "one row-map entry per thread");
};

// the reduction has the k steps that the kernel wants of it, in either segment or both together
template <typename Cfg>
inline bool fills_pipeline(int64_t Kdim, int segs = 1) {
  return (Kdim + Cfg::BK - 1) / Cfg::BK * segs >= 2 * Cfg::NSTAGE;
}

// A second product in the same launch: one dense group with its own matrices, width and reduction length, as the
// shared experts are beside the routed ones.
struct DenseProblem {
  const uint16_t *a0, *a1, *b0, *b1;  // a1 / b1: the up matrix or the second segment
  uint16_t *c, *save0, *save1;
  int rows, k, n, ntiles;
};

// How the workgroups of an XCD share out the tiles of two products (kJoint): the dense product's tiles first, dealt
// round, then the grouped product's, of which the workgroups without the last round of dense tiles take `lead` rounds
// more than the others -- as many grouped tiles as last as long as one dense tile.  Workgroup w of W takes in place p
// (p = 0, 1, ...) the tile with the returned index among n1 dense tiles followed by n0 grouped ones, or -1 at its end.
// Every index from 0 to n0 + n1 - 1 is returned exactly once.
__host__ __device__ inline int joint_tile(int w, int W, int p, int n1, int n0, int lead) {
  const int full = n1 / W, longer = n1 - full * W;  // `longer` workgroups have one dense tile more
  const int mine = full + (w < longer ? 1 : 0);
  if (p < mine) return p * W + w;
  const int q = p - mine, rest = W - longer;
  int i;
  if (longer == 0)
    i = q * W + w;
  else if (w < longer)
    i = lead * rest + q * W + w;
  else
    i = q < lead ? q * rest + (w - longer) : lead * rest + (q - lead) * W + w;
  return i < n0 ? n1 + i : -1;
}

// kNT = false: C = A @ B[e] with B[e] stored [K, N] (the forward products; kDual: two of them sharing the A tile).
// kNT = true:  C = sum over segs segments of A_s @ B_s[e]^T with B_s[e] stored [N, K] (the data gradients of
//              the backward pass, grouped_gemm_bwd.hpp): the B tile is then k-contiguous like the A tile,
//              lives in LDS in the same swizzled row layout and is read with ds_read_b128; the k loop
//              runs through the segments one after the other.
// kJoint: the tiles of `dp` run in the same launch (fully persistent workgroups, chunk 0).
// first_block: the launch's workgroups in front of these (a multiple of 8: a tile's XCD stays the same).
template <typename Cfg, bool kNT, bool kJoint = false>
__device__ __forceinline__ void stream_gemm_body(
    const uint16_t* __restrict__ A, const uint16_t* __restrict__ A1, const uint16_t* __restrict__ B0,
    const uint16_t* __restrict__ B1, uint16_t* __restrict__ C, const int32_t* __restrict__ group_sizes,
    const int32_t* __restrict__ offsets, int E, int dense_rows, int Kdim, int N, int ntiles_n,
    const int32_t* __restrict__ row_map, int row_div, int a_rows, uint16_t* __restrict__ save0,
    uint16_t* __restrict__ save1, int segs, int window, int chunk, const DenseProblem& dp, int first_block = 0) {
  constexpr int BM = Cfg::BM, BN = Cfg::BN, BK = Cfg::BK, NT = Cfg::NT, NS = Cfg::NSTAGE;
  constexpr int TM = Cfg::TM, TN = Cfg::TN, WN = Cfg::WN;
  constexpr int CPRA = Cfg::CPRA, KK = BK / 16, LPS = Cfg::LPS;
  constexpr int kBand = Cfg::SUBW / 64;  // 4 x 64 blocks of B side by side in a sub-tile
  constexpr bool kDual = Cfg::kDual;
  // X: rows that a tile may have beyond BM, a block of 32 more per wave.  The row blocks of a wave then lie
  // kRowStep apart, those of the waves above one another in turn; without such rows they are neighbours, so that waves
  // without rows leave the LDS to the others (two blocks of each wave are bound by its reads: down of 333 rows a group 55.8
  // us in turn, 54.3 as neighbours).
  constexpr int X = Cfg::XROWS, TMX = TM + (X ? 1 : 0), kRowStep = X ? Cfg::WAVES_M * 32 : 32, kWaveStep = X ? 32 : TM * 32;
  using L = StreamLayout<Cfg>;
  static_assert(KK % 2 == 0, "fragment double buffer wants an even number of sub-steps");
  static_assert(kNT || (Cfg::OPT & 128) != 0, "weight tiles in 4 x 64 blocks");
  static_assert(!kNT || !kDual, "the transposed-B form has one output per tile");
  // K may end inside a step (the interleaved steady part leaves no room for a branch: every load checks)
  constexpr bool kTail = (Cfg::OPT & 65536) != 0;
  static_assert(!kNT || (BN * CPRA) % NT == 0, "the B tile must divide evenly over the threads");
  static_assert(X == 0 || NS == 2, "the waits count the load of the X rows only where they drain everything");
  extern __shared__ __align__(16) unsigned char smem_raw[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / Cfg::WAVES_N, wn = wave - wm * Cfg::WAVES_N;
  // What is computed from the lane once per tile takes the lane id afresh, so that none of it stays in registers
  // through the k loops, which have none to spare.
  auto fresh_lane = [] {
    int l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return l;
  };
  const bool gather = row_map != nullptr;
  auto seg_steps = [](int k) { return kTail ? (k + BK - 1) / BK : k / BK; };  // k steps of one segment
  const int nk_segs = kNT ? segs : 1;

  // ---- schedule (as in grouped_gemm_dma_persistent_kernel) ----
  // Group sizes and first rows are copied into LDS once; every tile look-up scans them from there, so
  // that no look-up touches global memory while operand loads are in flight.
  int* const gs_l = reinterpret_cast<int*>(smem_raw + L::kGroupBase);
  int* const row0_l = gs_l + JTMOE_MAX_EXPERTS;
  if (group_sizes) {
    for (int e = tid; e < JTMOE_MAX_EXPERTS; e += NT) {
      gs_l[e] = e < E ? group_sizes[e] : 0;
      row0_l[e] = e < E ? offsets[e] : 0;
    }
    __syncthreads();
  }
  auto mtiles_with = [&](int x) {
    return group_sizes ? __builtin_amdgcn_readfirstlane(group_scan(BM, gs_l, JTMOE_MAX_EXPERTS, x, lane).total)
                       : group_mtiles(dense_rows, BM, x);
  };
  const int lead = kJoint ? max(1, (2 * dp.k + Kdim) / (2 * Kdim)) : 0;  // how many grouped tiles last as long as a dense one
  // Taller tiles where they spare a round (a tile with X rows takes up to a quarter longer: with 24 groups of 366 rows,
  // two of them below 320, and four rounds either way they cost a forward pass 2.3 %), or where there are many rounds, of
  // which they are the cheaper work.
  int extra = 0, real_mtiles = mtiles_with(0), dense_mtiles = kJoint ? group_mtiles(dp.rows, BM, 0) : 0;
  if (X != 0) {
    const int workgroups = (int)gridDim.x - first_block;  // (one for the whole launch each: chunk 0)
    auto rounds = [&](int mt, int dense_mt) {
      return (mt * ntiles_n + (kJoint ? dense_mt * dp.ntiles * lead : 0) + workgroups - 1) / workgroups;
    };
    const int tall = mtiles_with(X), dense_tall = kJoint ? group_mtiles(dp.rows, BM, X) : 0;
    const int plain_rounds = rounds(real_mtiles, dense_mtiles);
    if (plain_rounds >= (int)kManyRounds || rounds(tall, dense_tall) < plain_rounds) {
      extra = X;
      real_mtiles = tall;
      dense_mtiles = dense_tall;
    }
  }
  const int total = real_mtiles * ntiles_n;
  const int per_xcd = (total + 7) >> 3;
  const int xcd = (int)blockIdx.x & 7;
  int idx = ((int)blockIdx.x - first_block) >> 3, stride = max(1, ((int)gridDim.x - first_block) >> 3), left = 0x7fffffff;
  // kJoint: this XCD's range of either product, the odd tiles of the two at opposite ends of the XCDs
  const int total1 = kJoint ? dense_mtiles * dp.ntiles : 0;
  const int first0 = (xcd * total) >> 3, count0 = (((xcd + 1) * total) >> 3) - first0;
  const int first1 = (xcd * total1 + 7) >> 3, count1 = (((xcd + 1) * total1 + 7) >> 3) - first1;
  int place = 0;  // kJoint: how many tiles this workgroup has looked up
  if (chunk > 0) {
    idx = (idx / window) * (window * chunk) + idx % window;
    stride = window;
    left = chunk;
  }

  struct Tile {
    int expert, row0, rows, n0;  // expert < 0: a tile of `dp`
  };
  auto locate = [&](int i) -> Tile {
    Tile t;
    t.expert = 0; t.row0 = 0; t.rows = 0; t.n0 = 0;
    bool second = false;
    int logical = xcd * per_xcd + i, mts = real_mtiles, nts = ntiles_n;
    if constexpr (kJoint) {
      const int j = joint_tile(idx, stride, place++, count1, count0, lead);
      if (j < 0) return t;
      second = j < count1;
      logical = second ? first1 + j : first0 + (j - count1);
      mts = second ? dense_mtiles : real_mtiles;
      nts = second ? dp.ntiles : ntiles_n;
    } else if (i >= per_xcd || logical >= total) {
      return t;
    }
    const int group_span = Cfg::GROUP_M * nts;
    const int group = logical / group_span;
    const int in_group = logical - group * group_span;
    const int gm = min(Cfg::GROUP_M, mts - group * Cfg::GROUP_M);
    const int nt = in_group / gm;
    const int mt = group * Cfg::GROUP_M + (in_group - nt * gm);
    if (second) {
      t.expert = -1;
      const TileSpan span = group_mtile(dp.rows, mt, BM, extra);
      t.row0 = span.first;
      t.rows = span.rows;
    } else if (group_sizes) {
      const int l = fresh_lane();
      const TileRows tr = locate_tile(group_scan(BM, gs_l, JTMOE_MAX_EXPERTS, extra, l), mt, BM, row0_l, extra, l);
      t.expert = __builtin_amdgcn_readfirstlane(tr.expert);
      t.row0 = __builtin_amdgcn_readfirstlane(tr.row0);
      t.rows = __builtin_amdgcn_readfirstlane(tr.rows);
    } else {
      const TileSpan span = group_mtile(dense_rows, mt, BM, extra);
      t.row0 = span.first;
      t.rows = span.rows;
    }
    t.n0 = nt * BN;
    return t;
  };

  // ---- the load plan: descriptors and offsets of the tile whose operands are being requested.  The
  // last NS steps of a tile request the next tile's first steps, so the plan switches over to the next
  // tile NS steps before the current tile ends; nothing else of the current tile depends on it. ----
  constexpr int NSEG = kNT ? 2 : 1;                        // A descriptors (one per segment)
  constexpr int NBD = kNT ? 2 : Cfg::NSUB;                 // B descriptors (per segment / per sub-tile)
  constexpr int B_LOADS = kNT ? BN * CPRA / NT : Cfg::NSUB;  // entries of b_voff
  static_assert(!kNT || B_LOADS == Cfg::NSUB * Cfg::BSUB_LOADS, "a stage has LPS loads in either form");
  struct Plan {
    i32x4_t a_rsrc[NSEG];
    i32x4_t b_rsrc[NBD];
    int a_voff[Cfg::A_LOADS];
    int b_voff[B_LOADS];
    int x_voff;     // the chunk of the rows past BM
    bool x;         // the tile has such rows: a stage has one load more
    int k, n, nk1;  // of the tile's product (constants of the launch unless kJoint)
  };
  // the tile's product, seen from the tile
  auto second_product = [](const Tile& t) { return kJoint && t.expert < 0; };
  auto tile_k = [&](const Tile& t) { return second_product(t) ? dp.k : Kdim; };
  auto tile_n = [&](const Tile& t) { return second_product(t) ? dp.n : N; };
  // thread t fetches 16-byte chunk chunk_of(t) of row t / CPRA of the A tile (and of the rows NT / CPRA further on)
  auto chunk_of = [](int t) { return (t % CPRA) ^ ((t / CPRA / (16 / CPRA)) % CPRA); };
  const int a_c = chunk_of(tid);
  const unsigned lds0 = lds_byte_addr(smem_raw);
  const unsigned wave_lds = lds0 + wave * 1024;
  // The X rows have no more chunks than a load of the whole workgroup fetches: with fewer, several waves fetch the same.
  constexpr int kXWaves = X ? X * CPRA / 64 : 1;
  const unsigned wave_lds_x = lds0 + BM * BK * 2 + (wave % kXWaves) * 1024;
  // the rows of the tile that thread t fetches chunks of: with its A loads, and past BM
  auto load_row = [](int t, int j) { return t / CPRA + j * (NT / CPRA); };
  auto x_row = [](int t) { return BM + t / CPRA % (X ? X : 1); };
  int* const rowbuf = reinterpret_cast<int*>(smem_raw + L::kRowBufBase);

  // everything of a plan but the A row offsets
  auto plan_tile = [&](Plan& p, const Tile& t) {
    const int tid_f = wave * 64 + fresh_lane(), chunk = chunk_of(tid_f);
    const bool second = second_product(t), gathered = gather && !second;
    p.k = tile_k(t);
    p.n = tile_n(t);
    p.nk1 = seg_steps(p.k);
    const size_t wofs = second ? 0 : (size_t)t.expert * Kdim * N;
    const uint16_t *a0 = second ? dp.a0 : A, *b0 = second ? dp.b0 : B0, *b1 = second ? dp.b1 : B1;
    if constexpr (kNT) {
      const uint16_t* a1 = second ? dp.a1 : A1;
#pragma unroll
      for (int sg = 0; sg < 2; ++sg) {
        const uint16_t* a = (sg == 1 && segs > 1) ? a1 : a0;
        const uint16_t* b = (sg == 1 && segs > 1) ? b1 : b0;
        p.a_rsrc[sg] = gathered ? make_rsrc(a, a_rows * Kdim * 2) : make_rsrc(a + (size_t)t.row0 * p.k, t.rows * p.k * 2);
        p.b_rsrc[sg] = make_rsrc(b + wofs, p.n * p.k * 2);  // rows of B past N lie outside it and read as zeros
      }
      // the B tile's rows are output columns: row n0 + r of B[e], the same slots and swizzle as the A tile
#pragma unroll
      for (int j = 0; j < B_LOADS; ++j) p.b_voff[j] = ((t.n0 + tid_f / CPRA + j * (NT / CPRA)) * p.k + chunk * 8) * 2;
    } else {
#pragma unroll
      for (int u = 0; u < Cfg::NSUB; ++u) p.b_rsrc[u] = make_rsrc((kDual && u == 1 ? b1 : b0) + wofs, p.k * p.n * 2);
      p.a_rsrc[0] = gathered ? make_rsrc(a0, a_rows * Kdim * 2) : make_rsrc(a0 + (size_t)t.row0 * p.k, t.rows * p.k * 2);
      // (B in 4 x 64 blocks: row and chunk of this thread)
      const int b_blk_id = tid_f >> 5, b_k = (b_blk_id / kBand) * 4 + ((tid_f >> 3) & 3);
      const int b_c = (b_blk_id % kBand) * 8 + ((tid_f & 7) ^ (((tid_f >> 4) & 1) << 2));
#pragma unroll
      for (int u = 0; u < Cfg::NSUB; ++u) p.b_voff[u] = (b_k * p.n + t.n0 + (kDual ? 0 : u * Cfg::SUBW) + b_c * 8) * 2;
    }
#pragma unroll
    for (int j = 0; j < Cfg::A_LOADS; ++j) p.a_voff[j] = (load_row(tid_f, j) * p.k + chunk * 8) * 2;
    p.x = X != 0 && t.rows > BM;
    p.x_voff = (x_row(tid_f) * p.k + chunk * 8) * 2;
  };
  // gathered rows: the offsets come from row ids (rows past the end of the group read as zeros)
  // row_map entries are divided by row_div (the top-k of the routing) with a multiply: for
  // 0 <= n < 2^27 and 1 <= d <= 32, floor(n / d) == (n * ceil(2^32 / d)) >> 32  (the product stays
  // below 2^60, and n * (d * ceil(2^32 / d) - 2^32) < 2^27 * 32 = 2^32)
  const unsigned long long div_magic = ((1ull << 32) + (unsigned)row_div - 1) / (unsigned)row_div;
  auto plan_rows = [&](Plan& p, const Tile& t, auto row_id) {
    const int tid_f = wave * 64 + fresh_lane(), chunk = chunk_of(tid_f);
    auto offset_of = [&](int r) {
      const int src = (int)(((unsigned long long)(unsigned)row_id(r) * div_magic) >> 32);
      return r < t.rows ? (src * Kdim + chunk * 8) * 2 : 0x70000000;
    };
#pragma unroll
    for (int j = 0; j < Cfg::A_LOADS; ++j) p.a_voff[j] = offset_of(load_row(tid_f, j));
    if (p.x) p.x_voff = offset_of(x_row(tid_f));
  };
  // The steps that end the launch.  With few accumulators they have a loop of their own, without loads (128 x 256 tiles,
  // one each: 51.3 us against 53.5 for 2688 -> 1024); with many that loop would have hundreds of registers spilled, and
  // they issue loads that store zeros.
  constexpr bool kOwnEnd = X == 0 && TM * TN <= 4;
  auto plan_nothing = [](Plan& p) {
#pragma unroll
    for (int j = 0; j < Cfg::A_LOADS; ++j) p.a_voff[j] = kOutside;
#pragma unroll
    for (int j = 0; j < B_LOADS; ++j) p.b_voff[j] = kOutside;
    p.x = false;
  };
  // load i of the LPS loads of a stage (A loads first, then B) of k step kt of the planned tile
  auto issue_one = [&](const Plan& p, int kt, int stage, int i) {
    const unsigned base = wave_lds + stage * Cfg::STAGE_BYTES;
    if constexpr (kNT) {
      const bool second = kt >= p.nk1;  // uniform: the step belongs to the second segment
      const int k0 = (second ? kt - p.nk1 : kt) * BK;
      const bool outside = kTail && k0 + a_c * 8 >= p.k;  // both tiles: this lane's chunk lies past the end of the row
      if (i < Cfg::A_LOADS)
        buffer_load_lds16(second ? p.a_rsrc[1] : p.a_rsrc[0], base + i * NT * 16, outside ? kOutside : p.a_voff[i],
                          k0 * 2);
      else
        buffer_load_lds16(second ? p.b_rsrc[1] : p.b_rsrc[0], base + Cfg::A_BYTES + (i - Cfg::A_LOADS) * NT * 16,
                          outside ? kOutside : p.b_voff[i - Cfg::A_LOADS], k0 * 2);
    } else {
      const int k0 = kt * BK;
      if (i < Cfg::A_LOADS) {
        buffer_load_lds16(p.a_rsrc[0], base + i * NT * 16, kTail && k0 + a_c * 8 >= p.k ? kOutside : p.a_voff[i],
                          k0 * 2);
      } else {
        const int u = (i - Cfg::A_LOADS) / Cfg::BSUB_LOADS, jb = (i - Cfg::A_LOADS) % Cfg::BSUB_LOADS;
        buffer_load_lds16(p.b_rsrc[u], base + Cfg::A_BYTES + u * Cfg::BSUB_BYTES + jb * NT * 16,
                          p.b_voff[u] + jb * (NT * 8 / Cfg::SUBW) * p.n * 2 + (kTail ? k0 * p.n * 2 : 0), kTail ? 0 : k0 * p.n * 2);
      }
    }
  };
  // ... and the one of the X rows, if the tile has any
  auto issue_x = [&](const Plan& p, int kt, int stage) {
    if (X == 0 || !p.x) return;
    const bool second = kNT && kt >= p.nk1;
    const int k0 = (second ? kt - p.nk1 : kt) * BK;
    buffer_load_lds16(second ? p.a_rsrc[NSEG - 1] : p.a_rsrc[0], wave_lds_x + stage * Cfg::STAGE_BYTES,
                      kTail && k0 + a_c * 8 >= p.k ? kOutside : p.x_voff, k0 * 2);
  };
  auto issue = [&](const Plan& p, int kt, int stage) {
#pragma unroll
    for (int i = 0; i < LPS; ++i) issue_one(p, kt, stage, i);
    issue_x(p, kt, stage);
  };

  // ---- fragment addresses of this lane (bytes inside a stage) ----
  const int a_row = wm * kWaveStep + (lane & 31);
  const int a_sw = (a_row / (16 / CPRA)) % CPRA;
  const int a_rowoff = a_row * (BK * 2);
  const int b_laneoff = ((lane & 15) >> 2) * 128 + (lane & 3) * 8 + ((lane >> 4) & 1) * 32 + (lane >> 5) * (2 * kBand * 512);
  const int half_swap = ((lane >> 3) & 1) * 64;
  int b_blk[TN];
  // kNT: the B tile in the A tile's layout, this lane's row = its output column
  const int bt_row = wn * WN + (lane & 31);
  const int bt_sw = (bt_row / (16 / CPRA)) % CPRA;
  const int bt_rowoff = Cfg::A_BYTES + bt_row * (BK * 2);
#pragma unroll
  for (int jj = 0; jj < TN; ++jj) {
    int col;
    if (kDual)
      col = (jj < TN / 2 ? 0 : BN) + wn * (WN / 2) + (jj % (TN / 2)) * 32;
    else
      col = wn * WN + jj * 32;
    const int u = col / Cfg::SUBW;
    b_blk[jj] = Cfg::A_BYTES + u * Cfg::BSUB_BYTES + (col % Cfg::SUBW / 64) * 512 + (col & 63) * 2 +
                ((col & 32) ? -half_swap : half_swap);
  }
  auto load_frag_a = [&](int stage, int kk, int mi) -> bf16x8_t {
    const unsigned char* st = smem_raw + stage * Cfg::STAGE_BYTES;
    return *reinterpret_cast<const bf16x8_t*>(st + a_rowoff + mi * kRowStep * BK * 2 + (((kk * 2 + (lane >> 5)) ^ a_sw) << 4));
  };
  auto load_frag_b = [&](int stage, int kk, int jj) -> bf16x8_t {
    if constexpr (kNT) {
      const unsigned char* st = smem_raw + stage * Cfg::STAGE_BYTES;
      return *reinterpret_cast<const bf16x8_t*>(st + bt_rowoff + jj * 32 * BK * 2 + (((kk * 2 + (lane >> 5)) ^ bt_sw) << 4));
    }
    const unsigned char* p = smem_raw + stage * Cfg::STAGE_BYTES + b_blk[jj] + b_laneoff + kk * (4 * kBand * 512);
    const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(p));
    const s16x4_t hi =
        __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(p + kBand * 512));
    const s16x8_t both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(bf16x8_t, both);
  };
  bf16x8_t ax[2];  // of the X rows' block
  auto load_frags = [&](int stage, int kk, bf16x8_t* af, bf16x8_t* bf) {
#pragma unroll
    for (int mi = 0; mi < TM; ++mi) af[mi] = load_frag_a(stage, kk, mi);
    if (X != 0) ax[0] = load_frag_a(stage, kk, TM);
#pragma unroll
    for (int jj = 0; jj < TN; ++jj) bf[jj] = load_frag_b(stage, kk, jj);
  };

  // ---- first tile: plan, all NS stages requested, first fragments read ----
  Tile cur = locate(idx);
  if (cur.rows <= 0) return;
  Plan pl;
  plan_tile(pl, cur);
  // (a partial tile's rows past the group end are not read: the map may end with the group)
  if (gather && !second_product(cur)) plan_rows(pl, cur, [&](int r) { return r < cur.rows ? row_map[cur.row0 + r] : 0; });
  int nk = pl.nk1 * nk_segs;  // k steps of the current tile
#pragma unroll
  for (int s = 0; s < NS; ++s) issue(pl, s, s);
  bf16x8_t af[2][TM], bf[2][TN];
  wait_and_barrier<(NS - 1) * LPS>();
  load_frags(0, 0, af[0], bf[0]);
  int cs = 0;  // stage of the current k step

  while (true) {
    const int cur_n = tile_n(cur);
    // row blocks of this wave that hold rows of the tile (none either if its columns lie past N)
    const int blocks = cur.n0 + wn * Cfg::WNO < cur_n ? max(0, (cur.rows - wm * kWaveStep + kRowStep - 1) / kRowStep) : 0;
    if constexpr (!kJoint) idx += stride;
    --left;
    const Tile nxt = locate(left > 0 ? idx : 0x3fffffff);
    const bool have_next = nxt.rows > 0;
    const int nk_next = kJoint ? seg_steps(tile_k(nxt)) * nk_segs : nk;

    // row ids of the next tile: one LDS-DMA dword per thread, requested now and read NS steps before
    // this tile ends (it is older than every operand load issued from here on, so the waits below
    // cover it)
    if (gather && have_next && !second_product(nxt)) {
      const i32x4_t map_rsrc = make_rsrc(row_map + nxt.row0, nxt.rows * 4);
      buffer_load_lds4(map_rsrc, lds0 + L::kRowBufBase + wave * 256, (fresh_lane() + wave * 64) * 4);
    }

    // The tile, written out for the number NB of the wave's row blocks that take part: a tile that is not full costs the
    // matrix cores what its rows need, to two blocks of a wave.  (Accumulators that lived on from one of these forms to
    // the next would not stay in the same registers, and hundreds would be spilled: each has its own, from the zeros to
    // the epilogue.)
    const bool second = second_product(cur);
    auto run_tile = [&](auto nb) {
      constexpr int NB = decltype(nb)::value, kMfmas = NB * TN;
      f32x16_t acc[NB > 0 ? NB : 1][TN];
#pragma unroll
      for (int mi = 0; mi < NB; ++mi)
#pragma unroll
        for (int jj = 0; jj < TN; ++jj)
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[mi][jj][i] = 0.0f;
      // MFMA g of a sub-step on fragment set `set`
      auto mfma = [&](int set, int g) {
        acc[g / TN][g % TN] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bf[set][g % TN], g / TN < TM ? af[set][g / TN] : ax[set],
                                                                      acc[g / TN][g % TN], 0, 0, 0);
      };
      // fragment f of the NB + TN of a sub-step
      auto read = [&](int set, int stage, int kk, int f) {
        if (f < NB)
          (f < TM ? af[set][f] : ax[set]) = load_frag_a(stage, kk, f);
        else
          bf[set][f - NB] = load_frag_b(stage, kk, f - NB);
      };
      // a step: with the loads of step `ahead` of the planned tile, or (kLoads = false) as the one before `left` others that end
      // the launch
      auto step = [&](auto loads_tag, int ahead, int left) {
        constexpr bool kLoads = decltype(loads_tag)::value;
        // sub-steps 0 .. KK-2: the fragments of the following sub-step are requested, then this one's MFMAs, which the
        // scheduler interleaves with the LDS reads (two per MFMA)
#pragma unroll
        for (int kk = 0; kk < KK - 1; ++kk) {
          if (NB > 0)
#pragma unroll
            for (int f = 0; f < NB + TN; ++f) read((kk + 1) & 1, cs, kk + 1, f);
#pragma unroll
          for (int g = 0; g < kMfmas; ++g) mfma(kk & 1, g);
#pragma unroll
          for (int g = 0; g < kMfmas; ++g) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        // the next step's stage has arrived (own loads: the wait; everyone's: the barrier), and every
        // wave holds its last fragments of the current stage, which is therefore free
        if (kLoads || left == NS - 1)
          wait_and_barrier<(NS - 2) * LPS>();
        else if (NS > 3 && left == NS - 2)
          wait_and_barrier<(NS > 3 ? NS - 3 : 0) * LPS>();
        else
          wait_and_barrier<0>();
        __builtin_amdgcn_sched_barrier(0);
        // last sub-step, in a fixed order: after each of its MFMAs operand loads of step `ahead` (into the stage just
        // released) and fragment reads of the next step are issued
        const int ns = (NS & (NS - 1)) == 0 ? (cs + 1) & (NS - 1) : cs + 1 == NS ? 0 : cs + 1;
        constexpr int kSlots = kMfmas > 0 ? kMfmas : 1;
        constexpr int kLoadsPer = (LPS + kSlots - 1) / kSlots, kFragsPer = (NB + TN + kSlots - 1) / kSlots;
#pragma unroll
        for (int g = 0; g < kSlots; ++g) {
          if (NB > 0) mfma((KK - 1) & 1, g);
          __builtin_amdgcn_sched_barrier(0);
          if (kLoads) {
#pragma unroll
            for (int q = 0; q < kLoadsPer; ++q)
              if (g * kLoadsPer + q < LPS) issue_one(pl, ahead, cs, g * kLoadsPer + q);
          }
          if (NB > 0)
#pragma unroll
            for (int q = 0; q < kFragsPer; ++q)
              if (g * kFragsPer + q < NB + TN) read(0, ns, 0, g * kFragsPer + q);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (kLoads) issue_x(pl, ahead, cs);
        cs = ns;
      };
      // all steps but the last NS, then, with the next tile's plan, those: their loads are its first steps'
#pragma unroll 1
      for (int part = 0; part < 2; ++part) {
        const int j0 = part ? nk - NS : 0, j1 = part ? nk : nk - NS, ahead = part ? NS - nk : NS;
        if (part) {
          if (have_next) {
            plan_tile(pl, nxt);
            if (gather && !second_product(nxt)) plan_rows(pl, nxt, [&](int r) { return rowbuf[r]; });
          } else if constexpr (kOwnEnd) {
            break;
          } else {
            plan_nothing(pl);
          }
        }
        for (int j = j0; j < j1; ++j) step(std::true_type{}, j + ahead, 0);
      }
      if constexpr (kOwnEnd) {
        if (!have_next) {
#pragma unroll 1
          for (int left = NS - 1; left >= 0; --left) step(std::false_type{}, 0, left);
        }
      }
      // epilogue: straight from the accumulators to memory (no LDS, no barrier)
      if constexpr (NB > 0)
        store_transposed_accumulators<Cfg, NB>(acc, wm * kWaveStep, kRowStep, wn, cur.row0, cur.rows, cur.n0, cur_n,
                                               second ? dp.rows : dense_rows, second ? dp.c : C,
                                               second ? dp.save0 : save0, second ? dp.save1 : save1);
    };
    if (X != 0 && blocks > TM)
      run_tile(std::integral_constant<int, TMX>{});
    else if (TM > 2 && blocks > 2)
      run_tile(std::integral_constant<int, TM>{});
    else if (blocks > 0)
      run_tile(std::integral_constant<int, TM < 2 ? TM : 2>{});
    else
      run_tile(std::integral_constant<int, 0>{});
    static_assert(TM == 1 || TM == 2 || TM == 4, "row blocks per wave");
    if (!have_next) break;
    // (with X rows no fragment stays in registers through the epilogue; without, a wave whose tile is full has read them)
    if (X != 0 || blocks <= (TM > 2 ? 2 : 0)) load_frags(cs, 0, af[0], bf[0]);
    cur = nxt;
    nk = nk_next;
  }
  wait_vmcnt<0>();  // (the loads of plan_nothing still write to LDS)
}

template <typename Cfg>
__global__ __launch_bounds__(Cfg::NT) void grouped_gemm_stream_kernel(
    const uint16_t* __restrict__ A, const uint16_t* __restrict__ B0, const uint16_t* __restrict__ B1,
    uint16_t* __restrict__ C, const int32_t* __restrict__ group_sizes, const int32_t* __restrict__ offsets, int E,
    int dense_rows, int Kdim, int N, int ntiles_n, const int32_t* __restrict__ row_map, int row_div,
    int a_rows, uint16_t* __restrict__ save0, uint16_t* __restrict__ save1, int window, int chunk) {
  stream_gemm_body<Cfg, false>(A, nullptr, B0, B1, C, group_sizes, offsets, E, dense_rows, Kdim, N, ntiles_n,
                               row_map, row_div, a_rows, save0, save1, 1, window, chunk, DenseProblem{});
}

// A grouped and a dense product in one launch of persistent workgroups (a multiple of 8, chunk 0).  The requirements
// above hold for both.
template <typename Cfg>
__global__ __launch_bounds__(Cfg::NT) void grouped_gemm_joint_kernel(
    const uint16_t* __restrict__ A, const uint16_t* __restrict__ B0, const uint16_t* __restrict__ B1,
    uint16_t* __restrict__ C, const int32_t* __restrict__ group_sizes, const int32_t* __restrict__ offsets, int E,
    int dense_rows, int Kdim, int N, int ntiles_n, const int32_t* __restrict__ row_map, int row_div,
    int a_rows, uint16_t* __restrict__ save0, uint16_t* __restrict__ save1, DenseProblem dp) {
  stream_gemm_body<Cfg, false, true>(A, nullptr, B0, B1, C, group_sizes, offsets, E, dense_rows, Kdim, N,
                                     ntiles_n, row_map, row_div, a_rows, save0, save1, 1, 0, 0, dp);
}

// The transposed-B form: the arguments of grouped_gemm_nt_kernel (grouped_gemm_bwd.hpp) plus the schedule.
// Requirements: (Kdim / BK, rounded up with OPT & 65536) * segs >= 2 * NSTAGE, and those of the kernel above.
template <typename Cfg>
__global__ __launch_bounds__(Cfg::NT) void grouped_gemm_stream_nt_kernel(
    const uint16_t* __restrict__ A0, const uint16_t* __restrict__ A1, const uint16_t* __restrict__ B0,
    const uint16_t* __restrict__ B1, uint16_t* __restrict__ C, const int32_t* __restrict__ group_sizes,
    const int32_t* __restrict__ offsets, int E, int dense_rows, int Kdim, int N, int ntiles_n, int segs,
    int window, int chunk) {
  stream_gemm_body<Cfg, true>(A0, A1, B0, B1, C, group_sizes, offsets, E, dense_rows, Kdim, N, ntiles_n,
                              nullptr, 1, 0, nullptr, nullptr, segs, window, chunk, DenseProblem{});
}

template <typename Cfg>
__global__ __launch_bounds__(Cfg::NT) void grouped_gemm_joint_nt_kernel(
    const uint16_t* __restrict__ A0, const uint16_t* __restrict__ A1, const uint16_t* __restrict__ B0,
    const uint16_t* __restrict__ B1, uint16_t* __restrict__ C, const int32_t* __restrict__ group_sizes,
    const int32_t* __restrict__ offsets, int E, int dense_rows, int Kdim, int N, int ntiles_n, int segs,
    DenseProblem dp) {
  stream_gemm_body<Cfg, true, true>(A0, A1, B0, B1, C, group_sizes, offsets, E, dense_rows, Kdim, N, ntiles_n,
                                    nullptr, 1, 0, nullptr, nullptr, segs, 0, 0, dp);
}

// The 256-row tiles of the library, of up to 320 rows: gate/up, down and data gradients, each also for a reduction that is
// no multiple of 64.  64-deep steps in two stages; with 32-deep ones in four, us (64-deep / 32-deep): 131072 rows in 64
// groups, 2048 x 1408: gate/up 1313 / 1332, down 730 / 741, dZ 743 / 774, dX 1347 / 1406; 8192 rows in 8 groups, 1024 x
// 2048: gate/up 71.6 / 72.9.  Eight waves of 128 x 64: with 64 x 128 there is no room for a block more per wave.
//
// Against 256 rows and a tile of its own for what is left of each group (uneven groups by random routing; us, before /
// now; both products of a layer call alone, matrices not in the caches; gradients in a training pass):
//   16384 rows in 64 groups, 2048 x 1408    gate/up 271 / 213, down 134 / 117, dZ 151 (half tiles) / 137, dX 312 / 209
//   16384 rows in 16 groups, 1024 x 2816    gate/up 195 / 196, down 131 (half tiles 110) / 87, dZ 113 / 104, dX 280 / 169
//   8192 rows in 8 groups, 1024 x 2048      gate/up 80 / 72
//   131072 rows in 64 groups, 2048 x 1408   gate/up 1343 / 1313, down 757 / 730, dZ 728 / 697, dX 1335 / 1261
// (Bound by the matrix cores at the power limit at 131072 rows, by rounds over the CUs at the others.)
using GateUpStreamCfg = DmaGemmCfg<256, 128, 64, 2, 4, true, 2, 16 + 128 + 131072>;
using GateUpStreamTailCfg = DmaGemmCfg<256, 128, 64, 2, 4, true, 2, 16 + 128 + 65536 + 131072>;
using DownStreamCfg = DmaGemmCfg<256, 256, 64, 2, 4, false, 2, 16 + 128 + 32768 + 131072>;
using DownStreamTailCfg = DmaGemmCfg<256, 256, 64, 2, 4, false, 2, 16 + 128 + 32768 + 65536 + 131072>;
using DgradStreamCfg = DmaGemmCfg<256, 256, 64, 2, 4, false, 2, 16 + 128 + 131072>;
using DgradStreamTailCfg = DmaGemmCfg<256, 256, 64, 2, 4, false, 2, 16 + 128 + 65536 + 131072>;
// ... without the rows beyond 256, for launches in which no round is to be spared: gate/up in 32-deep steps and four
// stages (figures at tile_shape).  Alone, the others then run in the kernels of grouped_gemm_dma.hpp and
// grouped_gemm_bwd.hpp (64 groups of 180 rows, us: down 90 against 97 here, dZ 119 against 128); these are for joint
// launches (down 60 against 63 us with them, 4096 tokens of 1024, 8 experts top-2 and one shared of 2048).
template <bool kTail, bool kJoint>
using GateUpPlainCfg = DmaGemmCfg<256, 128, 32, kJoint ? 4 : 2, kJoint ? 2 : 4, true, 4, 16 + 128 + (kTail ? 65536 : 0)>;
template <bool kTail>
using DownPlainCfg = DmaGemmCfg<256, 256, 32, 2, 4, false, 4, 16 + 128 + 32768 + (kTail ? 65536 : 0)>;
template <bool kTail>
using DgradPlainCfg = DmaGemmCfg<256, 256, 64, 2, 4, false, 2, 16 + 128 + (kTail ? 65536 : 0)>;
// Smaller tiles (tile_shape).  128 x 128 ones in eight waves: gate/up of 1024 rows, 2048 x 2816, 33.8 us against 40.5 in
// four waves and 32-deep steps, down 29.2 against 37.6; the
// data gradients are up to 5 % faster in four.  (The check for a ragged last step costs nothing: one variant
// serves every width where there is no SwiGLU.)
template <bool kTail>
using GateUpQuarterCfg = DmaGemmCfg<64, 64, 64, 2, 2, true, 4, 16 + 128 + (kTail ? 65536 : 0)>;
template <bool kTail>
using GateUpNarrowCfg = DmaGemmCfg<128, 64, 64, 2, 2, true, 4, 16 + 128 + (kTail ? 65536 : 0)>;
template <bool kTail>
using GateUpHalfCfg = DmaGemmCfg<128, 128, 64, 2, 4, true, 3, 16 + 128 + (kTail ? 65536 : 0)>;
template <bool kTail>
using GateUpHalfShortCfg = DmaGemmCfg<128, 128, 32, 2, 2, true, 4, 16 + 128 + (kTail ? 65536 : 0)>;
using QuarterCfg = DmaGemmCfg<64, 64, 64, 2, 2, false, 4, 16 + 128 + 65536>;  // down and data gradients
using NarrowCfg = DmaGemmCfg<128, 64, 64, 2, 2, false, 4, 16 + 128 + 65536>;
using DownHalfCfg = DmaGemmCfg<128, 128, 64, 2, 4, false, 4, 16 + 128 + 65536>;
using DgradHalfDeepCfg = DmaGemmCfg<128, 128, 64, 2, 2, false, 4, 16 + 128 + 65536>;
using HalfShortCfg = DmaGemmCfg<128, 128, 32, 2, 2, false, 4, 16 + 128 + 65536>;
using Rows256Cfg = DmaGemmCfg<256, 128, 64, 4, 2, false, 3, 16 + 128 + 65536>;
using Rows128Cfg = DmaGemmCfg<128, 256, 64, 2, 4, false, 3, 16 + 128 + 65536>;
// two workgroups per CU
using DownHalfDeepCfg = DmaGemmCfg<128, 128, 64, 2, 2, false, 2, 16 + 128 + 65536>;

// launch(Cfg{}) with the configuration of a shape
template <bool kTail, bool kJoint, typename Launch>
int with_gate_up_tiles(TileShape s, Launch launch) {
  switch (s) {
    case TileShape::k64x64: return launch(GateUpQuarterCfg<kTail>{});
    case TileShape::k128x64: return launch(GateUpNarrowCfg<kTail>{});
    case TileShape::k128x128: return launch(GateUpHalfCfg<kTail>{});
    case TileShape::k128x128Short: return launch(GateUpHalfShortCfg<kTail>{});
    case TileShape::kPlain: return launch(GateUpPlainCfg<kTail, kJoint>{});
    default: return launch(std::conditional_t<kTail, GateUpStreamTailCfg, GateUpStreamCfg>{});
  }
}
// ... for down products and data gradients, all but the largest (no data gradient asks for the short ones: the deep kernel
// would be refused)
template <bool kDown, typename Launch>
int with_smaller_tiles(TileShape s, Launch launch) {
  switch (s) {
    case TileShape::k64x64: return launch(QuarterCfg{});
    case TileShape::k128x64: return launch(NarrowCfg{});
    case TileShape::k128x128: return launch(std::conditional_t<kDown, DownHalfCfg, DgradHalfDeepCfg>{});
    case TileShape::k256x128: return launch(Rows256Cfg{});
    case TileShape::k128x128Short: return launch(std::conditional_t<kDown, HalfShortCfg, DgradHalfDeepCfg>{});
    default: return launch(Rows128Cfg{});
  }
}
// A product of the shared experts beside the workgroups of a small launch in front of the routed products, each tile on
// a CU of its own: behind `front` workgroups (a multiple of 8).  grid = 0: not at these sizes and pointers, or not where
// the product is a part of the routed one's launch.  (grouped_gemm.hip; the tiles are 64 x 64 or 128 x 64.)
struct SharedTiles {
  TileShape tiles;
  DenseProblem p;
  int grid;
};
constexpr int kDispatchFront = 8;  // the workgroups of the dispatch in front of such tiles
TileShape tiles_beside(Product product, int64_t T, int64_t H, int64_t Is, int64_t I, int64_t E, int64_t K, int front,
                       double cus);  // by the sizes alone; kPlain: none
SharedTiles shared_gate_up_beside(const void* x, const SharedExperts& s, int64_t T, int64_t H, int64_t E, int64_t K, int front);
SharedTiles shared_down_beside(const SharedExperts& s, int64_t T, int64_t H, int64_t E, int64_t K, int front);

// (Also in router.hip, whose flags round divisions correctly and contract nothing.  A gate/up product of a whole reduction
// has the same bits there: silu_rcp neither divides nor adds to a product.  One that divides would not.)
template <typename Cfg>
__device__ __forceinline__ void dense_stream_tiles(const DenseProblem& p, int front) {
  static_assert(!Cfg::kDual || (Cfg::OPT & 65536) == 0, "gate/up of whole reductions only");
  stream_gemm_body<Cfg, false>(p.a0, nullptr, p.b0, p.b1, p.c, nullptr, nullptr, 1, p.rows, p.k, p.n, p.ntiles, nullptr, 1,
                               0, p.save0, p.save1, 1, 0, 0, DenseProblem{}, front);
}

}  // namespace jtmoe
