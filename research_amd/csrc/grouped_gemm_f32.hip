// Launchers of the single-precision grouped GEMMs (grouped_gemm_f32.hpp).
#include "gemm_launch.hpp"
#include "grouped_gemm_f32.hpp"

#include <algorithm>

namespace jtmoe {
namespace {

constexpr int64_t kF32Limit = (int64_t)1 << 29;  // elements: byte offsets stay below 2^31

// m-tiles of a launch: exact for one dense group, an upper bound (group sizes live on the device) otherwise
inline int64_t f32_mtiles(bool dense, int64_t rows, int64_t E, int BM) {
  return (rows + BM - 1) / BM + (dense ? 0 : std::min(E, rows));
}

// Rounds over the CUs times the work of a tile, in units of a 64 x 64 tile.  With unequal groups about half a
// tile per group is padding.  At 8 groups, 512 x 1024 the rule takes the small tiles, us against the large ones: 2048 rows
// gate/up 57 and 73, down 38 and 72; 4096 rows 106 and 118, 61 (544 tiles, three units) and 77 (144 tiles, four units);
// 8192 rows 170 and 179, 94 and 129.
inline int64_t f32_cost(bool dense, int64_t rows, int64_t E, int64_t N, int BM, int BN, int units,
                        int64_t cus = persistent_grid_size()) {
  const int64_t mt = (rows + BM - 1) / BM + (dense ? 0 : std::min(E, rows) / 2);
  const int64_t tiles = mt * ((N + BN - 1) / BN);
  return (tiles + cus - 1) / cus * units;
}

template <typename Cfg>
int launch_f32(const void* a0, const void* a1, const void* b0, const void* b1, void* c, const int32_t* group_sizes,
               const int32_t* offsets, int64_t rows, int64_t Kdim, int64_t N, int64_t E, const int32_t* row_map,
               int row_div, int64_t a_rows, int segs, void* save0, void* save1, hipStream_t stream) {
  const int64_t mtiles = f32_mtiles(group_sizes == nullptr, rows, E, Cfg::BM), nt = (N + Cfg::BN - 1) / Cfg::BN;
  const int64_t grid = gemm_grid(mtiles, nt);
  if (grid >= ((int64_t)1 << 31)) return fail(JTMOE_EUNSUPPORTED, "grouped gemm (f32): grid too large");
  grouped_gemm_f32_kernel<Cfg><<<(unsigned)grid, Cfg::NT, Cfg::SMEM_BYTES, stream>>>(
      static_cast<const float*>(a0), static_cast<const float*>(a1), static_cast<const float*>(b0),
      static_cast<const float*>(b1), static_cast<float*>(c), group_sizes, offsets, (int)E, (int)rows, (int)Kdim, (int)N,
      (int)mtiles, (int)nt, row_map, row_div, (int)a_rows, segs, static_cast<float*>(save0),
      static_cast<float*>(save1));
  return JTMOE_OK;
}

__global__ __launch_bounds__(256) void reduce_partials_f32_kernel(const float4* __restrict__ partial, int splits,
                                                                  size_t nvec, float4* __restrict__ out) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= nvec) return;
  float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  for (int s = 0; s < splits; ++s) {
    const float4 v = partial[(size_t)s * nvec + i];
    acc.x += v.x;
    acc.y += v.y;
    acc.z += v.z;
    acc.w += v.w;
  }
  out[i] = acc;
}

// Runs of rows of a one-group weight gradient (the router's [H, E], the shared experts'): enough of them
// for two workgroups per CU, none shorter than 128 rows.
inline int f32_tn_splits(int64_t rows, int64_t KA, int64_t N) {
  const int64_t tiles = ((KA + 63) / 64) * ((N + 63) / 64);
  const int64_t want = 2 * persistent_grid_size() / std::max<int64_t>(tiles, 1);
  return (int)std::max<int64_t>(1, std::min({want, rows / 128, (int64_t)64}));
}

template <int BMO, int BNO>
int launch_f32_tn(const float* p, const float* d0, const float* d1, float* c0, float* c1, const int32_t* group_sizes,
                  const int32_t* offsets, int64_t rows, int64_t KA, int64_t N, int64_t E, int split_chunk,
                  hipStream_t stream) {
  constexpr size_t smem = 2 * 32 * (BMO + BNO) * 4;
  const int64_t mt = (KA + BMO - 1) / BMO, nt = (N + BNO - 1) / BNO, grid = E * mt * nt * (d1 ? 2 : 1);
  if (grid >= ((int64_t)1 << 31)) return fail(JTMOE_EUNSUPPORTED, "grouped gemm (f32): grid too large");
  grouped_gemm_f32_tn_kernel<BMO, BNO><<<(unsigned)grid, 256, smem, stream>>>(
      p, d0, d1, c0, c1, group_sizes, offsets, (int)E, (int)rows, (int)KA, (int)N, (int)mt, (int)nt, split_chunk);
  return JTMOE_OK;
}

}  // namespace

bool f32_gemm_supported(const void* a0, const void* a1, const void* b0, const void* b1, const void* c, int64_t a_rows,
                        int64_t Kdim, int64_t N) {
  return Kdim % 4 == 0 && N % 4 == 0 && Kdim * N < kF32Limit && a_rows * Kdim < kF32Limit && aligned16(a0) &&
         aligned16(a1) && aligned16(b0) && aligned16(b1) && aligned16(c);
}

int launch_f32_nn(const void* a, const void* b0, const void* b1, void* c, const int32_t* group_sizes,
                  const int32_t* offsets, int64_t rows, int64_t Kdim, int64_t N, int64_t E, const int32_t* row_map,
                  int row_div, int64_t a_rows, void* save0, void* save1, hipStream_t stream) {
  const bool dense = group_sizes == nullptr;
#define JT_F32(BM, BN, DUAL)                                                                                    \
  launch_f32<F32Cfg<BM, BN, DUAL, false>>(a, nullptr, b0, b1, c, group_sizes, offsets, rows, Kdim, N, E, row_map,   \
                                          row_div, a_rows, 1, save0, save1, stream)
  if (b1)
    return f32_cost(dense, rows, E, N, 128, 64, 4) <= f32_cost(dense, rows, E, N, 64, 64, 2) ? JT_F32(128, 64, true)
                                                                                             : JT_F32(64, 64, true);
  return f32_cost(dense, rows, E, N, 128, 128, 4) <= f32_cost(dense, rows, E, N, 64, 64, 1) ? JT_F32(128, 128, false)
                                                                                            : JT_F32(64, 64, false);
#undef JT_F32
}

int launch_f32_nt(const void* a0, const void* a1, const void* b0, const void* b1, void* c, const int32_t* group_sizes,
                  const int32_t* offsets, int64_t rows, int64_t Kdim, int64_t N, int64_t E, int segs, hipStream_t stream) {
  const bool dense = group_sizes == nullptr;
#define JT_F32(BM, BN)                                                                                       \
  launch_f32<F32Cfg<BM, BN, false, true>>(a0, a1, b0, b1, c, group_sizes, offsets, rows, Kdim, N, E, nullptr, 1,  \
                                          rows, segs, nullptr, nullptr, stream)
  return f32_cost(dense, rows, E, N, 128, 128, 4) <= f32_cost(dense, rows, E, N, 64, 64, 1) ? JT_F32(128, 128)
                                                                                            : JT_F32(64, 64);
#undef JT_F32
}

size_t f32_tn_split_bytes(int64_t rows, int64_t KA, int64_t N, bool dual) {
  const int splits = f32_tn_splits(rows, KA, N);
  if (splits < 2 || KA % 4 != 0 || N % 4 != 0) return 0;
  return align_up((size_t)splits * KA * N * sizeof(float) * (dual ? 2 : 1), 256);
}

int launch_f32_tn(const void* p_, const void* d0_, const void* d1_, void* c0_, void* c1_, const int32_t* group_sizes,
                  const int32_t* offsets, int64_t rows, int64_t KA, int64_t N, int64_t E, void* split_ws,
                  hipStream_t stream) {
  const float *p = static_cast<const float*>(p_), *d0 = static_cast<const float*>(d0_), *d1 = static_cast<const float*>(d1_);
  float *c0 = static_cast<float*>(c0_), *c1 = static_cast<float*>(c1_);
  const int splits = split_ws && group_sizes == nullptr ? f32_tn_splits(rows, KA, N) : 1;
  if (splits > 1) {
    const int chunk = (int)((rows + splits - 1) / splits);
    float* part0 = static_cast<float*>(split_ws);
    float* part1 = part0 + (size_t)splits * KA * N;
    const int rc = launch_f32_tn<64, 64>(p, d0, d1, part0, part1, nullptr, nullptr, rows, KA, N, splits, chunk, stream);
    if (rc) return rc;
    const size_t nvec = (size_t)KA * N / 4;
    for (int i = 0; i < (d1 ? 2 : 1); ++i)
      reduce_partials_f32_kernel<<<(unsigned)((nvec + 255) / 256), 256, 0, stream>>>(
          reinterpret_cast<const float4*>(i ? part1 : part0), splits, nvec, reinterpret_cast<float4*>(i ? c1 : c0));
    return JTMOE_OK;
  }
  // a tile's reduction is as long as its group, so the number of tiles alone decides
  const int64_t matrices = d1 ? 2 : 1, cus = persistent_grid_size();
  const int64_t big = matrices * E * ((KA + 127) / 128) * ((N + 127) / 128);
  const int64_t small = matrices * E * ((KA + 63) / 64) * ((N + 63) / 64);
  if ((big + cus - 1) / cus * 4 <= (small + cus - 1) / cus)
    return launch_f32_tn<128, 128>(p, d0, d1, c0, c1, group_sizes, offsets, rows, KA, N, E, 0, stream);
  return launch_f32_tn<64, 64>(p, d0, d1, c0, c1, group_sizes, offsets, rows, KA, N, E, 0, stream);
}

// One launch where it saves work in the last rounds of three.  Cost in k steps of a 64 x 64 tile per CU: the launches of
// their own in whole rounds of the tiles they take, the joint one spread evenly, but no shorter than its longest tile.
// The weight gradients' large tiles are the faster ones as long as rounds are full (131 against 114 TFLOP/s), so a tenth
// has to be saved.  4096 rows in 8 groups, 512 x 1024 (10496 against 12288 steps): 192 us against 238 for the three;
// twice the rows (20736 against 22528) keep launches of their own.
bool f32_backward_joint(int64_t rows, int64_t H, int64_t I, int64_t E, int64_t cus) {
  const int64_t depth = std::max<int64_t>(rows / std::max<int64_t>(E, 1), 1);
  const auto tn = [&](int64_t matrices) {
    const int64_t big = matrices * E * ((H + 127) / 128) * ((I + 127) / 128);
    const int64_t small = matrices * E * ((H + 63) / 64) * ((I + 63) / 64);
    return std::min((big + cus - 1) / cus * 4, (small + cus - 1) / cus) * depth;
  };
  const int64_t apart =
      std::min(f32_cost(false, rows, E, H, 128, 128, 4, cus), f32_cost(false, rows, E, H, 64, 64, 1, cus)) * 2 * I +
      tn(2) + tn(1);
  const int64_t mt = (rows + 63) / 64 + std::min(E, rows) / 2, th = (H + 63) / 64, ti = (I + 63) / 64;
  const int64_t joint = std::max((mt * th * 2 * I + 3 * E * th * ti * depth + cus - 1) / cus, 2 * I);
  return joint * 10 <= apart * 9;
}

bool f32_backward_products_supported(const F32Backward& b, int64_t rows, int64_t H, int64_t I, int64_t E,
                                     int compute_units) {
  const int64_t grid = gemm_grid(f32_mtiles(false, rows, E, 64), (H + 63) / 64) + 3 * E * ((H + 63) / 64) * ((I + 63) / 64);
  return rows > 0 && rows * H < kF32Limit && grid < ((int64_t)1 << 31) && aligned16(b.hw) && aligned16(b.dyp) &&
         f32_gemm_supported(b.dg, b.du, b.gate, b.up, b.dxp, rows, I, H) &&
         f32_gemm_supported(b.xp, b.d_gate, b.d_up, b.d_down, nullptr, rows, H, I) &&
         f32_backward_joint(rows, H, I, E, compute_units > 0 ? compute_units : persistent_grid_size());
}

int launch_f32_backward_products(const F32Backward& b, const int32_t* group_sizes, const int32_t* offsets, int64_t rows,
                                 int64_t H, int64_t I, int64_t E, hipStream_t stream) {
  const int64_t th = (H + 63) / 64, ti = (I + 63) / 64, mtiles = f32_mtiles(false, rows, E, 64);
  const int64_t dx_blocks = gemm_grid(mtiles, th), grid = dx_blocks + 3 * E * th * ti;
  const auto in = [](const void* p) { return static_cast<const float*>(p); };
  const auto out = [](void* p) { return static_cast<float*>(p); };
  const F32BackwardProducts p{in(b.dg),   in(b.du),      in(b.hw),    in(b.xp),     in(b.dyp),   in(b.gate), in(b.up),
                              out(b.dxp), out(b.d_gate), out(b.d_up), out(b.d_down), group_sizes, offsets,    (int)rows,
                              (int)H,     (int)I,        (int)E,      (int)mtiles,  (int)dx_blocks};
  grouped_gemm_f32_backward_kernel<<<(unsigned)grid, 256, F32Cfg<64, 64, false, true>::SMEM_BYTES, stream>>>(p);
  return check_launch("experts backward (f32 products)");
}

}  // namespace jtmoe

// what the rule above says of these sizes
extern "C" const char* jtmoe_f32_backward_kernel(int64_t rows, int64_t H, int64_t I, int64_t E, int compute_units) {
  using namespace jtmoe;
  const int64_t limit = (int64_t)1 << 24;
  if (rows <= 0 || rows >= ((int64_t)1 << 31) || H <= 0 || H >= limit || I <= 0 || I >= limit || E <= 0 ||
      E > JTMOE_MAX_EXPERTS || compute_units < 0)
    return "";
  return f32_backward_products_supported({}, rows, H, I, E, compute_units) ? "joint" : "separate";
}
