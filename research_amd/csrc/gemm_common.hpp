// Pieces shared by the grouped GEMM kernels: vector types, the m-tile -> expert
// lookup and the workgroup -> tile order.
#pragma once

#include "common.hpp"

#include <cmath>

namespace jtmoe {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(8))) short s16x8_t;
typedef __attribute__((ext_vector_type(4))) short s16x4_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;

// word 3 of a raw buffer descriptor on gfx9: 32-bit data format, untyped
constexpr int kBufferFlags = 0x00020000;

struct TileRows {
  int expert;
  int row0;  // first row of the tile
  int rows;  // valid rows in the tile (0 = no such tile)
};

// m-tiles of a group of n rows.  With extra == 0: BM rows each, the last one what is left.  With extra rows to a tile
// (beyond BM) the rows that whole tiles leave over are spread over these, `extra` to each from the first one on, and
// only rows that do not fit in there start a tile of their own.
__host__ __device__ __forceinline__ int group_mtiles(int n, int BM, int extra) {
  if (n <= 0) return 0;
  const int whole = n < BM ? 1 : n / BM;
  return whole + (n - whole * BM > extra * whole ? 1 : 0);
}
// rows [first, first + rows) of the group: its m-tile i
struct TileSpan {
  int first, rows;
};
__host__ __device__ __forceinline__ TileSpan group_mtile(int n, int i, int BM, int extra) {
  const int whole = n < BM ? 1 : n / BM, left = n - whole * BM;
  const bool fits = left <= extra * whole;
  const int spread = fits && left > 0 ? left : 0, tiles = whole + (fits ? 0 : 1);
  auto start = [&](int t) { return t * BM + (t * extra < spread ? t * extra : spread); };
  const int first = start(i);
  return {first, (i + 1 < tiles ? start(i + 1) : n) - first};
}

// Tiles are counted expert by expert, group_mtiles each.  group_scan computes, in
// every lane of the calling wave, the tile counts of the lane's own experts, their exclusive
// prefix and the total; locate_tile then finds the expert and row range of m-tile `mt`.
// E <= JTMOE_MAX_EXPERTS.
struct GroupScan {
  static constexpr int kPer = JTMOE_MAX_EXPERTS / 64;  // experts per lane, contiguous
  int n[kPer], tiles[kPer];
  int first;  // tiles before this lane's experts
  int total;  // tiles of all experts
};

__device__ __forceinline__ GroupScan group_scan(int BM, const int32_t* __restrict__ group_sizes, int E, int extra, int lane) {
  GroupScan g;
  int local = 0;
#pragma unroll
  for (int j = 0; j < GroupScan::kPer; ++j) {
    const int e = lane * GroupScan::kPer + j;
    g.n[j] = e < E ? group_sizes[e] : 0;
    g.tiles[j] = group_mtiles(g.n[j], BM, extra);
    local += g.tiles[j];
  }
  int incl = local;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int v = __shfl_up(incl, d);
    if (lane >= d) incl += v;
  }
  g.first = incl - local;
  g.total = __shfl(incl, 63);
  return g;
}

__device__ __forceinline__ GroupScan group_scan(int BM, const int32_t* __restrict__ group_sizes, int E) {
  return group_scan(BM, group_sizes, E, 0, threadIdx.x & 63);
}

__device__ __forceinline__ TileRows locate_tile(const GroupScan& g, int mt, int BM,
                                                const int32_t* __restrict__ offsets, int extra, int lane) {
  TileRows r;
  r.expert = 0;
  r.row0 = 0;
  r.rows = 0;
  int first = g.first;
  int last = first;
#pragma unroll
  for (int j = 0; j < GroupScan::kPer; ++j) last += g.tiles[j];
  const bool mine = mt >= first && mt < last;
  const unsigned long long owners = __ballot(mine);
  if (owners == 0ull) return r;
  const int owner = __ffsll((long long)owners) - 1;
  int expert = 0, local_tile = 0, rows_e = 0;
#pragma unroll
  for (int j = 0; j < GroupScan::kPer; ++j) {
    if (mine && mt >= first && mt < first + g.tiles[j]) {
      expert = lane * GroupScan::kPer + j;
      local_tile = mt - first;
      rows_e = g.n[j];
    }
    first += g.tiles[j];
  }
  expert = __shfl(expert, owner);
  local_tile = __shfl(local_tile, owner);
  rows_e = __shfl(rows_e, owner);
  r.expert = expert;
  const TileSpan span = group_mtile(rows_e, local_tile, BM, extra);
  r.row0 = offsets[expert] + span.first;
  r.rows = span.rows;
  return r;
}

__device__ __forceinline__ TileRows locate_tile(const GroupScan& g, int mt, int BM, const int32_t* __restrict__ offsets) {
  return locate_tile(g, mt, BM, offsets, 0, threadIdx.x & 63);
}

// m-tile `mt` of a grouped (or, with group_sizes == nullptr, dense) row range.  Every lane of the
// calling wave gets the same answer.
__device__ __forceinline__ TileRows find_tile_wave(int mt, int BM, const int32_t* __restrict__ group_sizes,
                                                   const int32_t* __restrict__ offsets, int E, int dense_rows) {
  if (group_sizes == nullptr) {
    TileRows r;
    r.expert = 0;
    r.row0 = 0;
    r.rows = 0;
    const int row0 = mt * BM;
    if (row0 < dense_rows) {
      r.row0 = row0;
      r.rows = min(BM, dense_rows - row0);
    }
    return r;
  }
  return locate_tile(group_scan(BM, group_sizes, E), mt, BM, offsets);
}

__device__ __forceinline__ float silu_fast(float g) { return g / (1.0f + __expf(-g)); }

struct TileCoord {
  int mt, nt;  // mt < 0: this workgroup has no tile
};

// Workgroup id -> (m-tile, n-tile).  Consecutive workgroup ids go round-robin to the 8 XCDs, so
// each XCD gets a contiguous range of the logical order, and that order is walked in groups of
// group_m m-tiles x all n-tiles so that neighbours share operand panels in their L2.
// (block / blocks: this workgroup's index among the workgroups that share out the tiles, and their number --
// the launch's own unless other workgroups of the launch do something else)
__device__ __forceinline__ TileCoord xcd_tile_order(int mtiles, int ntiles_n, int group_m, int block, int blocks) {
  TileCoord t;
  const int total = mtiles * ntiles_n;
  const int per_xcd = blocks >> 3;
  const int logical = (block & 7) * per_xcd + (block >> 3);
  if (logical >= total) {
    t.mt = -1;
    t.nt = 0;
    return t;
  }
  const int group_span = group_m * ntiles_n;
  const int group = logical / group_span;
  const int in_group = logical - group * group_span;
  const int gm = min(group_m, mtiles - group * group_m);
  t.nt = in_group / gm;
  t.mt = group * group_m + (in_group - t.nt * gm);
  return t;
}

// The tile of this workgroup when the launch was sized for an upper bound of `mtiles_bound` m-tiles
// and only `mtiles` of them exist (group sizes live on the device): the XCD ranges are cut from the
// real count, so that the surplus workgroups are spread over all XCDs instead of idling one of them.
// Requires gridDim.x / 8 >= ceil(mtiles * ntiles_n / 8), which the bound guarantees.
__device__ __forceinline__ TileCoord xcd_tile_order_balanced(int mtiles, int ntiles_n, int group_m, int block) {
  TileCoord t;
  t.mt = -1;
  t.nt = 0;
  const int total = mtiles * ntiles_n;
  const int per_xcd = (total + 7) >> 3;
  const int idx = block >> 3;
  const int logical = (block & 7) * per_xcd + idx;
  if (idx >= per_xcd || logical >= total) return t;
  const int group_span = group_m * ntiles_n;
  const int group = logical / group_span;
  const int in_group = logical - group * group_span;
  const int gm = min(group_m, mtiles - group * group_m);
  t.nt = in_group / gm;
  t.mt = group * group_m + (in_group - t.nt * gm);
  return t;
}

__device__ __forceinline__ TileCoord xcd_tile_order(int mtiles, int ntiles_n, int group_m) {
  return xcd_tile_order(mtiles, ntiles_n, group_m, (int)blockIdx.x, (int)gridDim.x);
}
__device__ __forceinline__ TileCoord xcd_tile_order_balanced(int mtiles, int ntiles_n, int group_m) {
  return xcd_tile_order_balanced(mtiles, ntiles_n, group_m, (int)blockIdx.x);
}

// Second half of every epilogue: a wave has parked its WM x WNO block of bf16 results in its own
// LDS slice `cw` (row stride CS elements) and streams it out row by row with 16-byte stores.
// Row r of the block is output row out_row0 + r; rows at or past rows_end and columns at or past
// N are dropped.
template <int WM, int WNO, int CS, bool kStream = false>
__device__ __forceinline__ void store_wave_block(const uint16_t* __restrict__ cw, int lane, uint16_t* __restrict__ out,
                                                 int N, size_t out_row0, int rows_end, int col0) {
  constexpr int CPR_OUT = WNO / 8;
  constexpr int OUT_CHUNKS = WM * CPR_OUT;
#pragma unroll
  for (int j = 0; j < OUT_CHUNKS / 64; ++j) {
    const int c = lane + j * 64;
    const int r = c / CPR_OUT, ch = c - r * CPR_OUT;
    const u32x4_t v = *reinterpret_cast<const u32x4_t*>(cw + r * CS + ch * 8);
    const int col = col0 + ch * 8;
    if (r < rows_end && col < N) {
      u32x4_t* const dst = reinterpret_cast<u32x4_t*>(out + (out_row0 + r) * N + col);
      if (kStream)
        __builtin_nontemporal_store(v, dst);  // the result is not read again by this kernel
      else
        *dst = v;
    }
  }
}

// number of workgroups for `mtiles x ntiles_n` tiles: a multiple of 8 (one slice per XCD)
inline int64_t gemm_grid(int64_t mtiles, int64_t ntiles_n) { return (mtiles * ntiles_n + 7) / 8 * 8; }

// number of workgroups of a persistent launch: one per CU of the current device, a whole number per
// XCD (the 256-row configurations fit one workgroup per CU); looked up once per process
inline int persistent_grid_size() {
  static const int size = [] {
    int device = 0, cus = 0;
    if (hipGetDevice(&device) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus < 8)
      return 8;
    return cus / 8 * 8;
  }();
  return size;
}

// m-tiles of BM rows to be expected: exact for one dense group; otherwise the groups that a balanced choice
// leaves with a row, and half a tile of padding in each once groups outgrow half a tile
inline double expected_mtiles(int64_t rows, int64_t E, bool dense, int BM) {
  if (dense) return (double)((rows + BM - 1) / BM);
  const double groups = (double)E * (1.0 - std::exp(-(double)rows / (double)E)), mean = (double)rows / groups;
  return groups * (mean > BM / 2 ? mean / BM + 0.5 : 1.0);
}

// The same where the tiles are as tall as a group is: rows per group spread evenly over mean +- 3 sqrt(mean) (top-k
// groups of random rows lie within that), so that groups of 162 rows count as one 256-row tile and two of 128, and
// not as 1.13 and 1.77.  From the latter the half tiles looked like 15 % less than three rounds where the whole
// ones need two: 1300 tokens top-8, 64 experts of 1408, 2048 wide 332 us a layer call against 311 without them.
// How far the groups really spread is not known on the host, so half tiles have to pay by either estimate.
inline double spread_mtiles(int64_t rows, int64_t E, bool dense, int BM) {
  if (dense) return (double)((rows + BM - 1) / BM);
  const double groups = (double)E * (1.0 - std::exp(-(double)rows / (double)E)), mean = (double)rows / groups;
  const double hi = mean + 3.0 * std::sqrt(mean), lo = std::fmax(0.0, mean - 3.0 * std::sqrt(mean));
  auto tiles_upto = [BM](double x) {  // integral of ceil(n / BM) over n from 0 to x
    const double q = std::floor(x / BM);
    return BM * q * (q + 1.0) / 2.0 + (x - q * BM) * (q + 1.0);
  };
  return groups * (tiles_upto(hi) - tiles_upto(lo)) / (hi - lo);
}

// m-tiles of 256 rows, each of up to 64 more where that spares tiles (group_mtiles; the stream kernel takes them only
// where they spare a round), by the two estimates: what a group's
// whole tiles leave over spread evenly over 256 rows, and groups spread evenly over mean +- 3 sqrt(mean).
inline double tall_mtiles(int64_t rows, int64_t E, bool dense, bool spread) {
  if (dense) return (double)group_mtiles((int)rows, 256, 64);
  const double groups = (double)E * (1.0 - std::exp(-(double)rows / (double)E)), mean = (double)rows / groups;
  const double reach = spread ? 3.0 * std::sqrt(mean) : 128.0;
  double tiles = 0.0;
  for (int i = 0; i < 32; ++i) {
    const int n = (int)(mean + reach * ((i + 0.5) / 16.0 - 1.0));
    tiles += n > 0 ? group_mtiles(n, 256, 64) : 1;
  }
  return groups * tiles / 32.0;
}
// what a launch of 256-row tiles of N columns counts, by either estimate
inline double whole_tiles(int64_t rows, int64_t E, bool dense, double ntiles, double cus, bool spread, bool tall) {
  const double plain = (spread ? spread_mtiles(rows, E, dense, 256) : expected_mtiles(rows, E, dense, 256)) * ntiles;
  return plain <= cus || !tall ? plain : std::fmin(plain, tall_mtiles(rows, E, dense, spread) * ntiles);
}

// 128 x 128 tiles against 256 x 256 ones, by rounds over the CUs: a round of 512 half tiles takes 0.57 of a round of
// 256 whole ones, a last round of at most 256 of them 0.42, the launch 0.12 more; half tiles read their operands
// twice as often, so beyond one per CU they are taken only where that is 15 % less.  Down products: one half tile
// per CU 40 us against 63 (2048 tokens, shared 2816; 64-deep steps 41), two per CU with 64-deep steps 55 against 64
// (4096 tokens; 32-deep 69); 8192 rows x 2048 -> 1024 in 8 groups: 57 against 56 (576 tiles, whole ones kept);
// 16384 rows in 16 groups x 2816 -> 1024 (1088 against 256 tiles of up to 320 rows): 109 against 87.  The data
// gradients follow the same line (figures at DgradHalfCfg); on the wrong side of it 32768
// rows in 64 groups x 2048 -> 1408 would take 262 us against 228.
enum class HalfTiles { kNone, kOnePerCu, kRounds };
// what `half` half tiles take, in rounds of whole ones
inline double half_tile_rounds(double half, double cus) {
  const double rounds = std::floor(half / (2 * cus)), rest = half - rounds * 2 * cus;
  return 0.12 + 0.57 * rounds + (rest <= 0.0 ? 0.0 : (rest <= cus ? 0.42 : 0.57));
}
// (tall: with the 256-row tiles counted as the stream kernel takes them, of up to 320 rows)
inline HalfTiles half_tiles(int64_t rows, int64_t E, bool dense, int64_t N, double cus, bool tall = true) {
  const double half_n = (double)((N + 127) / 128), full_n = (double)((N + 255) / 256);
  if (expected_mtiles(rows, E, dense, 128) * half_n <= cus) return HalfTiles::kOnePerCu;
  auto pays = [cus](double half, double full) { return 1.15 * half_tile_rounds(half, cus) < std::ceil(full / cus); };
  return pays(expected_mtiles(rows, E, dense, 128) * half_n, whole_tiles(rows, E, dense, full_n, cus, false, tall)) &&
                 pays(spread_mtiles(rows, E, dense, 128) * half_n, whole_tiles(rows, E, dense, full_n, cus, true, tall))
             ? HalfTiles::kRounds
             : HalfTiles::kNone;
}

// Tile of a product that has no streaming or 64-row tiles, for `rows` rows in E groups times N columns and, in the same
// launch, dense_rows x dense_N.
//
// Where every tile finds a CU of its own nothing hides a step's latency but the loads in flight (operands arrive some
// 1.3 us after their request, whatever the tile), so the smallest tiles that still do are the fastest.  Rows that may
// end up in more tiles than the estimates say cost a second round: both have to fit.  us for 128 x 128 / 128 x 64 / 64 x
// 64, matrices cold:
//   one group, 2048 x 2816: 387 rows gate/up 30.3 / 21.7 (176 tiles) / 30.8 (308), down 23.7 / 19.1 / 16.6 (224); 700 rows
//   32.5 / 38.7 (264) / 37.0, down 27.5 / 22.0 (192) / 29.0
//   8 groups, 1024 x 2048: 400 rows gate/up 25.2 / 20.4 / 20.9, down 17.8 / 14.6 / 12.1
// One output a tile: 256 x 128 and 128 x 256 ones in three stages take 0.6 of a round of 256 x 256 ones, whose two stages
// drain once a step (us, 256 x 256 / 128 x 256 / 256 x 128): 2048 rows 2816 -> 2048 down 62 / 41 / 40, dX 127 / 83 / 77; 6000
// rows in 16 groups, 2816 -> 1024, down 66 / 47 / 44, dX 129 / 91 / 87; two rounds of them are no less than one (8192 rows:
// 73 / 75 / 81, 139 / 155 / 153).
// Groups that fit one tile of 128 rows (kFewGroupRows): bound by the expert matrices, read once, and so by the bytes of them
// in flight: half as many rows, and more stages or workgroups for it.  us, 256-row tiles / 128-row ones; 64 groups, 2048 x
// 1408: 77 rows gate/up 146 / 140, dZ 105 / 94, dX 152 / 138, down 77.2 / 78.6; 128 groups, 2048 x 768: 93 rows 168 / 157 and 97
// / 96, skewed by Zipf's law 198 / 180 and 111 / 106; at 137 rows gate/up 172 / 206, down 87 / 111.  Nearer to 128 rows a few
// groups more than fit are likely: not where 5 % more tiles are a round more (96 groups of 100, 1304 x 904, four rounds for
// three: gate/up 118 / 131).
// Beyond, 128-row tiles (128 x 256 with one output) where they take no more rounds: 12 groups of 333 rows, 1280 x 1792,
// two rounds either way: gate/up 62 / 50, three for two 53 / 55 (8192 rows, 1024 x 2048).
// kTall: 256-row tiles of up to 320 rows (a kernel of their own, which without such rows is slower than the others' by up to
// 5 %); else plain ones.  By the spread of the groups, where they spare rounds enough for the time a taller tile takes: 1.2 of a
// plain one, 1.25 for one data gradient alone, which has to spare a tenth of the tiles as well, and for products of one output
// beside dense tiles, which fill the last round of either, unless the tiles themselves are fewer by as much.  us, plain /
// taller (rounds), of passes without a pause: 64 groups of 256 rows, 2048 x 1408, gate/up 267 / 209, down 158 / 116, dX 305 /
// 208 (5, 3 and 3, 2); of 328 gate/up 310 / 303 (6, 5), beside shared tiles down 188 / 202 and dX 352 / 373 (5, 4; by tiles
// 4.3, 3.4); of 256, gate/up beside shared tiles 289 / 253 (5, 4; 4.8, 3.4); of 512 down 227 / 208 and dX 429 / 357 (5, 4), dZ
// 235 / 203 (4, 3), but gate/up, which the line leaves out, 408 / 377 (7, 6); dZ of 64 groups of 600 271 / 271, of 40 of 1638,
// 1304 x 904, 234 / 230 (5, 4), of 24 of 698, 1000 x 2664, 129 / 134 (4, 3, with 94 % of the tiles).
// With eight rounds and more the tiles that are left count, and the kernel decides from the real sizes: 64 groups of 698 rows
// (94 % of the tiles) gate/up 509 / 542, of 1024 (85 %) 746 / 693, down 438 / 411 and dX 783 / 740, of 2048 (88 %) 1369 / 1314,
// 792 / 755 and 1382 / 1343; 128 skewed groups of 750 (88 %), 2048 x 768, down 392 / 379, dX 625 / 635, of 1024 (85 %) dX 827 /
// 829.  Beside shared tiles, where the plain kernel is slower too, always: 64 groups of 698 623 / 603.
// k128x128Pair: two workgroups to a CU.
enum class TileShape { k64x64, k128x64, k128x128, k128x128Short, k128x128Pair, k256x128, k128x256, kTall, kPlain };
enum class Product { kGateUp, kDown, kGradient, kGradientPair };  // the last: of two segments
inline bool large_tiles(TileShape s) { return s == TileShape::kTall || s == TileShape::kPlain; }
constexpr int64_t kFewGroupRows = 108, kFewGroupRowsSure = 94;  // mean + 3.5 standard deviations within 128
constexpr double kManyRounds = 8.0;
inline TileShape tile_shape(Product product, int64_t rows, int64_t E, bool dense, int64_t N, double cus,
                            int64_t dense_rows = 0, int64_t dense_N = 0) {
  const bool dual = product == Product::kGateUp, alone = dense_rows == 0;
  auto one_each = [&](int BM, int BN) {
    const double mtiles = std::fmax(expected_mtiles(rows, E, dense, BM), spread_mtiles(rows, E, dense, BM));
    return mtiles * (double)((N + BN - 1) / BN) + (double)((dense_rows + BM - 1) / BM * ((dense_N + BN - 1) / BN)) <= cus;
  };
  if (one_each(64, 64)) return TileShape::k64x64;
  if (one_each(128, 64)) return TileShape::k128x64;
  if (one_each(128, 128)) return TileShape::k128x128;
  if (!dual && one_each(256, 128)) return TileShape::k256x128;
  if (!dual && one_each(128, 256)) return TileShape::k128x256;
  const int BN = dual ? 128 : 256;
  const double nt = (double)((N + BN - 1) / BN), dense_nt = (double)((dense_N + BN - 1) / BN);
  auto rounds = [cus](double tiles) { return std::ceil(tiles / cus); };
  const double plain = spread_mtiles(rows, E, dense, 256) * nt + (double)((dense_rows + 255) / 256) * dense_nt;
  if (!dense && alone && rows <= kFewGroupRows * E && (rows <= kFewGroupRowsSure * E || rounds(1.05 * plain) == rounds(plain)))
    return dual ? TileShape::k128x128 : product == Product::kDown ? TileShape::k128x256 : TileShape::k128x128Pair;
  const double tall = tall_mtiles(rows, E, dense, true) * nt + (double)group_mtiles((int)dense_rows, 256, 64) * dense_nt;
  const bool fewer = tall <= 0.9 * plain;
  if (rounds(plain) >= kManyRounds) return !alone || fewer ? TileShape::kTall : TileShape::kPlain;
  const double low = std::fmax(expected_mtiles(rows, E, dense, 128), spread_mtiles(rows, E, dense, 128)) * nt +
                     (double)((dense_rows + 127) / 128) * dense_nt;
  if (rounds(low) <= rounds(plain) && 0.72 * rounds(low) < 1.2 * rounds(tall)) return dual ? TileShape::k128x128 : TileShape::k128x256;
  const bool one_gradient = alone && product == Product::kGradient;
  const double longer = one_gradient || (!alone && !dual && 1.3 * tall >= plain) ? 1.25 : 1.2;
  return longer * rounds(tall) < rounds(plain) && (fewer || !one_gradient) ? TileShape::kTall : TileShape::kPlain;
}
// ... with a reduction of `steps` 64-deep steps at least, of which a kernel wants twice as many as it has stages, and, for
// launches of one half tile per CU, nothing larger than that.  k128x128Short: in 32-deep steps.
inline TileShape tile_shape_for(TileShape s, bool half, int64_t steps, bool dual) {
  const bool small = s == TileShape::k64x64 || s == TileShape::k128x64 || s == TileShape::k128x128;
  if (half && !small) s = TileShape::k128x128;
  const bool four = s == TileShape::k64x64 || s == TileShape::k128x64 || (s == TileShape::k128x128 && !dual);  // stages, or three
  const bool fits = s == TileShape::kTall || s == TileShape::kPlain || steps >= 2 * (four ? 4 : 3);
  return fits ? s : half ? TileShape::k128x128Short : TileShape::kTall;
}

// ---- routed and shared experts in one launch ----
// Alone, the shared experts' products are a part of a round behind the routed ones; as more tiles of the routed
// launch they fill its last round.  `rows` routed rows in E groups times N columns, T shared rows times N1 columns with
// a reduction `longer` times as long (dual: gate/up, tiles 128 columns wide whatever their height).  kOnePerCu: half
// tiles hold both products at once; kRounds: 256-row tiles; kNone: launches of their own.
// Estimates in full rounds of routed 256-row tiles; a launch of half tiles with a CU each is one_per_cu of them times
// its reduction (measured beside full rounds, at the power limit: shared down of 2816 at 2048 tokens 40 us, a round of
// routed tiles of 1408 53; gate/up at 1024 tokens 41 and 57; dx of 2048 at 4096 tokens 41 and 99).  At equal
// rounds a call gains or loses up to 3 % with few of them (less of a last round idle against a higher clock in two part-filled
// ones) and gains up to 1 % from six on.  As for half tiles it has to pay by two estimates of how the groups spread (1300
// tokens, 64 experts top-8: two rounds of routed tiles by one, 2.3 by the other; down jointly 3 % more a call), and with
// three standard deviations more groups than are to be expected: with a few rows per group each is a tile, and a round more
// streams the experts' matrices a second time (backward of 24 tokens, 64 experts top-8, 2048 x 1408, shared 2816: dX jointly
// 194 us where 63 groups had a row, 121 + 39 apart; of 27 tokens 595 the pass against 555).  The 256-row tiles are counted
// without rows beyond these, with which the lines were drawn.
inline HalfTiles joint_tiles(int64_t rows, int64_t E, int64_t N, int64_t T, int64_t N1, double longer, double cus,
                             double one_per_cu, bool dual = false) {
  auto across = [dual](int64_t n, int bn) { return (double)(dual ? (n + 127) / 128 : (n + bn - 1) / bn); };
  auto dense_tiles = [&](int bm) { return (double)((T + bm - 1) / bm) * across(N1, bm); };
  auto alone = [&](HalfTiles h, double half, double full) {
    if (h == HalfTiles::kOnePerCu) return one_per_cu;
    return h == HalfTiles::kRounds && !dual ? half_tile_rounds(half, cus) : std::ceil(full / cus);
  };
  if (expected_mtiles(rows, E, false, 128) * across(N, 128) + dense_tiles(128) <= cus) return HalfTiles::kOnePerCu;
  const HalfTiles routed = half_tiles(rows, E, false, N, cus, /*tall=*/false);
  const double shared = longer * alone(half_tiles(T, 1, true, N1, cus, /*tall=*/false), dense_tiles(128), dense_tiles(256));
  const double mean = (double)rows / (double)E, empty = std::exp(-mean);
  const double more_groups =
      std::fmin((double)E * empty, 3.0 * std::sqrt((double)E * empty * (1.0 - (1.0 + mean) * empty)));
  auto pays = [&](auto mtiles) {
    const double full = mtiles(rows, E, false, 256) * across(N, 256), half = mtiles(rows, E, false, 128) * across(N, 128);
    const double both =
        std::fmax(longer, std::ceil((full + more_groups * across(N, 256) + longer * dense_tiles(256)) / cus));
    const double apart = alone(routed, half, full) + shared;
    return both < apart || (both == apart && both > 6.0);
  };
  return pays(expected_mtiles) && pays(spread_mtiles) ? HalfTiles::kRounds : HalfTiles::kNone;
}

}  // namespace jtmoe
