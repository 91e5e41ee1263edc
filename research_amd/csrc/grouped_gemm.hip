// Grouped SwiGLU expert FFN: two grouped GEMM launches over variable-size,
// expert-contiguous row groups.
//
// Follows the three jax.lax.ragged_dot calls of the reference and the SwiGLU
// between them (moe.py:638-641), and SharedSwiGLU.__call__ (moe.py:361-364) as
// the one-group dense case:
//   launch 1 (dual):  act = round(silu(round(X Wg[e])) * round(X Wu[e]))   [rows, I]
//   launch 2:         Y   = round(act Wd[e])                                [rows, H]
// `round` is the rounding to the compute dtype (identity for fp32); products
// are accumulated in fp32 on the matrix cores (v_mfma_f32_32x32x16_bf16 for
// bf16, v_mfma_f32_32x32x2_f32 for fp32).
#include "common.hpp"
#include "dispatch_small.hpp"
#include "gemm_launch.hpp"
#include "grouped_gemm_dma.hpp"
#include "grouped_gemm_skinny.hpp"
#include "grouped_gemm_stream.hpp"

#include <algorithm>
#include <mutex>

namespace jtmoe {
namespace {

// ---------------------------------------------------------------------------
// Generic kernel: any shape, any alignment, both dtypes.  64x64x32 tiles, four
// waves (2x2), each owning one 32x32 accumulator tile (two when kDual).
// Operands are staged element by element through LDS with bounds checks; B is
// transposed on the way in so that both MFMA operands are k-contiguous.
// ---------------------------------------------------------------------------
constexpr int GBM = 64, GBN = 64, GBK = 32;
constexpr int GPAD = 8;  // elements; keeps 16-byte alignment of bf16 rows

template <typename T>
__device__ __forceinline__ void mfma_tile(const T* __restrict__ a_row, const T* __restrict__ b_row, int khalf,
                                          f32x16_t& acc);

// a_row / b_row point at the k = 0 element of this lane's A row / B column in LDS
template <>
__device__ __forceinline__ void mfma_tile<bf16_raw>(const bf16_raw* __restrict__ a_row,
                                                    const bf16_raw* __restrict__ b_row, int khalf, f32x16_t& acc) {
#pragma unroll
  for (int kk = 0; kk < GBK / 16; ++kk) {
    const bf16x8_t a = *reinterpret_cast<const bf16x8_t*>(a_row + kk * 16 + khalf * 8);
    const bf16x8_t b = *reinterpret_cast<const bf16x8_t*>(b_row + kk * 16 + khalf * 8);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
  }
}

template <>
__device__ __forceinline__ void mfma_tile<float>(const float* __restrict__ a_row, const float* __restrict__ b_row,
                                                 int khalf, f32x16_t& acc) {
#pragma unroll
  for (int kk = 0; kk < GBK / 2; ++kk) {
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a_row[kk * 2 + khalf], b_row[kk * 2 + khalf], acc, 0, 0, 0);
  }
}

template <typename T, bool kDual>
__global__ __launch_bounds__(256) void grouped_gemm_generic_kernel(
    const T* __restrict__ A, const T* __restrict__ B0, const T* __restrict__ B1, T* __restrict__ C,
    const int32_t* __restrict__ group_sizes, const int32_t* __restrict__ offsets, int E, int dense_rows, int Kdim,
    int N, int ntiles_n, const int32_t* __restrict__ row_map, int row_div, T* __restrict__ save0,
    T* __restrict__ save1) {
  __shared__ __align__(16) T As[GBM][GBK + GPAD];
  __shared__ int a_row_of[GBM];  // row of A behind tile row r (through the row map, if there is one)
  __shared__ __align__(16) T Bs0[GBN][GBK + GPAD];
  __shared__ __align__(16) T Bs1[kDual ? GBN : 1][GBK + GPAD];

  const int mt = blockIdx.x / ntiles_n;
  const int nt = blockIdx.x - mt * ntiles_n;
  const TileRows tr = find_tile_wave(mt, GBM, group_sizes, offsets, E, dense_rows);
  if (tr.rows <= 0) return;
  const int n0 = nt * GBN;
  const size_t wofs = (size_t)tr.expert * Kdim * N;
  const T* Bg0 = B0 + wofs;
  const T* Bg1 = kDual ? B1 + wofs : nullptr;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int frag_row = lane & 31, khalf = lane >> 5;

  f32x16_t acc0, acc1;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    acc0[i] = 0.0f;
    acc1[i] = 0.0f;
  }

  T zero;
  __builtin_memset(&zero, 0, sizeof(T));
  if (tid < GBM && tid < tr.rows) a_row_of[tid] = row_map ? row_map[tr.row0 + tid] / row_div : tr.row0 + tid;
  __syncthreads();

  for (int k0 = 0; k0 < Kdim; k0 += GBK) {
    for (int idx = tid; idx < GBM * GBK; idx += 256) {
      const int r = idx / GBK, c = idx - r * GBK;
      const int gk = k0 + c;
      T v = zero;
      if (r < tr.rows && gk < Kdim) v = A[(size_t)a_row_of[r] * Kdim + gk];
      As[r][c] = v;
    }
    for (int idx = tid; idx < GBK * GBN; idx += 256) {
      const int k = idx / GBN, n = idx - k * GBN;
      const int gk = k0 + k, gn = n0 + n;
      const bool ok = gk < Kdim && gn < N;
      Bs0[n][k] = ok ? Bg0[(size_t)gk * N + gn] : zero;
      if (kDual) Bs1[n][k] = ok ? Bg1[(size_t)gk * N + gn] : zero;
    }
    __syncthreads();
    const T* a_row = &As[wm * 32 + frag_row][0];
    mfma_tile<T>(a_row, &Bs0[wn * 32 + frag_row][0], khalf, acc0);
    if (kDual) mfma_tile<T>(a_row, &Bs1[wn * 32 + frag_row][0], khalf, acc1);
    __syncthreads();
  }

  // 32x32 accumulator layout: value i of lane l is row 8*(i/4) + 4*(l/32) + i%4, column l%32
  const int col = n0 + wn * 32 + (lane & 31);
  if (col < N) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = wm * 32 + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
      if (r < tr.rows) {
        float v;
        if (kDual) {
          const float g = Elem<T>::round(acc0[i]);
          const float u = Elem<T>::round(acc1[i]);
          v = silu_fast(g) * u;
          if (save0) {
            Elem<T>::store(save0 + (size_t)(tr.row0 + r) * N + col, g);
            Elem<T>::store(save1 + (size_t)(tr.row0 + r) * N + col, u);
          }
        } else {
          v = acc0[i];
        }
        Elem<T>::store(C + (size_t)(tr.row0 + r) * N + col, v);
      }
    }
  }
}

// upper bound on the number of m-tiles when the group sizes live on the device
inline int64_t max_m_tiles(int64_t rows, int64_t groups, int BM) {
  return (rows + BM - 1) / BM + (groups < rows ? groups : rows);
}

template <typename T, bool kDual>
int launch_generic(const void* a, const void* b0, const void* b1, void* c, const int32_t* group_sizes,
                   const int32_t* offsets, int64_t rows, int64_t Kdim, int64_t N, int64_t E, hipStream_t stream,
                   const int32_t* row_map = nullptr, int row_div = 1, void* save0 = nullptr, void* save1 = nullptr) {
  const bool dense = group_sizes == nullptr;
  const int64_t mtiles = dense ? (rows + GBM - 1) / GBM : max_m_tiles(rows, E, GBM);
  const int64_t nt = (N + GBN - 1) / GBN;
  if (mtiles * nt >= ((int64_t)1 << 31)) return fail(JTMOE_EUNSUPPORTED, "grouped gemm: grid too large");
  grouped_gemm_generic_kernel<T, kDual><<<(unsigned)(mtiles * nt), 256, 0, stream>>>(
      static_cast<const T*>(a), static_cast<const T*>(b0), static_cast<const T*>(b1), static_cast<T*>(c), group_sizes,
      offsets, (int)E, (int)rows, (int)Kdim, (int)N, (int)nt, row_map, row_div, static_cast<T*>(save0),
      static_cast<T*>(save1));
  return JTMOE_OK;
}

template <typename Cfg>
int launch_fast(const void* a, const void* b0, const void* b1, void* c, const int32_t* group_sizes,
                const int32_t* offsets, int64_t rows, int64_t Kdim, int64_t N, int64_t E, hipStream_t stream,
                const int32_t* row_map = nullptr, int row_div = 1, int64_t a_rows = 0, void* save0 = nullptr,
                void* save1 = nullptr, int64_t uniform_rows = 0, int64_t a_group_rows = 0,
                const Beside* beside = nullptr) {
  // the 256-row configurations run as persistent workgroups (see persistent_schedule), the others one
  // tile per workgroup
  constexpr bool kPersistent = Cfg::BM == 256 && Cfg::NSTAGE == 2 && Cfg::BK == 64;
  static std::once_flag once;
  static hipError_t attr_err = hipSuccess;
  auto kernel = [] {
    if constexpr (kPersistent)
      return &grouped_gemm_dma_persistent_kernel<Cfg>;
    else
      return &grouped_gemm_dma_kernel<Cfg>;
  }();
  std::call_once(once, [&] {
    attr_err = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)Cfg::SMEM_BYTES);
  });
  if (attr_err != hipSuccess)
    return fail(JTMOE_ELAUNCH, "grouped gemm: kernel set-up: %s", hipGetErrorString(attr_err));
  const bool dense = group_sizes == nullptr;
  const int64_t mtiles = uniform_rows > 0 ? E * ((uniform_rows + Cfg::BM - 1) / Cfg::BM)
                         : dense          ? (rows + Cfg::BM - 1) / Cfg::BM
                                          : max_m_tiles(rows, E, Cfg::BM);
  const int64_t nt = (N + Cfg::BN - 1) / Cfg::BN;
  const int64_t tiles_grid = gemm_grid(mtiles, nt);
  if (tiles_grid >= ((int64_t)1 << 31)) return fail(JTMOE_EUNSUPPORTED, "grouped gemm: grid too large");
  if constexpr (kPersistent) {
    if (uniform_rows > 0 || a_group_rows > 0)
      return fail(JTMOE_EUNSUPPORTED, "grouped gemm: the decode forms run one tile per workgroup");
    const PersistentSchedule ps = persistent_schedule(tiles_grid, persistent_grid_size(), kTilesPerWorkgroup<Cfg>);
    kernel<<<(unsigned)ps.grid, Cfg::NT, Cfg::SMEM_BYTES, stream>>>(
        static_cast<const uint16_t*>(a), static_cast<const uint16_t*>(b0), static_cast<const uint16_t*>(b1),
        static_cast<uint16_t*>(c), group_sizes, offsets, (int)E, (int)rows, (int)Kdim, (int)N, (int)mtiles, (int)nt,
        row_map, row_div, (int)a_rows, static_cast<uint16_t*>(save0), static_cast<uint16_t*>(save1), ps.window,
        ps.chunk);
  } else {
    // (the shared experts come beside a router of whole 128-row chunks: never with a ragged reduction here)
    constexpr bool kBeside = (Cfg::OPT & 65536) == 0;
    if constexpr (kBeside) if (beside) {
      grouped_gemm_dma_beside_kernel<Cfg><<<(unsigned)(tiles_grid + beside->blocks), Cfg::NT, Cfg::SMEM_BYTES, stream>>>(
          static_cast<const uint16_t*>(a), static_cast<const uint16_t*>(b0), static_cast<const uint16_t*>(b1),
          static_cast<uint16_t*>(c), group_sizes, offsets, (int)E, (int)rows, (int)Kdim, (int)N, (int)mtiles, (int)nt,
          row_map, row_div, (int)a_rows, static_cast<uint16_t*>(save0), static_cast<uint16_t*>(save1),
          (int)a_group_rows, *beside);
      return JTMOE_OK;
    }
    kernel<<<(unsigned)tiles_grid, Cfg::NT, Cfg::SMEM_BYTES, stream>>>(
        static_cast<const uint16_t*>(a), static_cast<const uint16_t*>(b0), static_cast<const uint16_t*>(b1),
        static_cast<uint16_t*>(c), group_sizes, offsets, (int)E, (int)rows, (int)Kdim, (int)N, (int)mtiles, (int)nt,
        row_map, row_div, (int)a_rows, static_cast<uint16_t*>(save0), static_cast<uint16_t*>(save1), (int)uniform_rows,
        (int)a_group_rows);
  }
  return JTMOE_OK;
}


// The stream kernel (grouped_gemm_stream.hpp): one software pipeline through all tiles of a workgroup, results written
// straight from the accumulators.  Its envelope is narrower than launch_fast's (see stream_ok).  Tiles of up to
// 320 rows run in one workgroup per CU for the whole launch (0.5 to 2 % faster than in workgroups of four tiles each), the
// others in workgroups of four (skewed groups: 275 us for gate/up of 24000 rows in 128 groups, 2048 x 768, against 265).
template <typename Cfg>
int launch_stream(const void* a, const void* b0, const void* b1, void* c, const int32_t* group_sizes,
                  const int32_t* offsets, int64_t rows, int64_t Kdim, int64_t N, int64_t E, hipStream_t stream,
                  const int32_t* row_map, int row_div, int64_t a_rows, void* save0, void* save1,
                  int workgroups_per_cu = 1) {
  using L = StreamLayout<Cfg>;
  static std::once_flag once;
  static hipError_t attr_err = hipSuccess;
  auto kernel = &grouped_gemm_stream_kernel<Cfg>;
  std::call_once(once, [&] {
    attr_err = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)L::kSmemBytes);
  });
  if (attr_err != hipSuccess)
    return fail(JTMOE_ELAUNCH, "grouped gemm: kernel set-up: %s", hipGetErrorString(attr_err));
  const bool dense = group_sizes == nullptr;
  if (!fills_pipeline<Cfg>(Kdim)) return fail(JTMOE_EUNSUPPORTED, "grouped gemm: reduction of %lld too short", (long long)Kdim);
  const int64_t mtiles = dense ? (rows + Cfg::BM - 1) / Cfg::BM : max_m_tiles(rows, E, Cfg::BM);
  const int64_t nt = (N + Cfg::BN - 1) / Cfg::BN;
  const int64_t tiles_grid = gemm_grid(mtiles, nt);
  if (tiles_grid >= ((int64_t)1 << 31)) return fail(JTMOE_EUNSUPPORTED, "grouped gemm: grid too large");
  const PersistentSchedule ps =
      persistent_schedule(tiles_grid, workgroups_per_cu * persistent_grid_size(), Cfg::XROWS ? 0 : 4);
  kernel<<<(unsigned)ps.grid, Cfg::NT, L::kSmemBytes, stream>>>(
      static_cast<const uint16_t*>(a), static_cast<const uint16_t*>(b0), static_cast<const uint16_t*>(b1),
      static_cast<uint16_t*>(c), group_sizes, offsets, (int)E, (int)rows, (int)Kdim, (int)N, (int)nt, row_map, row_div, (int)a_rows, static_cast<uint16_t*>(save0), static_cast<uint16_t*>(save1), ps.window, ps.chunk);
  return JTMOE_OK;
}

// A routed product and the shared experts' one in the same launch.  Routed operands as in launch_fast; `dp` without its
// tile counts.
struct RoutedProblem {
  const void *a, *b0, *b1;
  void *c, *save0, *save1;
  const int32_t *group_sizes, *offsets, *row_map;
  int64_t rows, K, N, E, a_rows;
  int row_div;
};

DenseProblem dense_problem(const RoutedProblem& s) {
  return {static_cast<const uint16_t*>(s.a), nullptr, static_cast<const uint16_t*>(s.b0), static_cast<const uint16_t*>(s.b1),
          static_cast<uint16_t*>(s.c), static_cast<uint16_t*>(s.save0), static_cast<uint16_t*>(s.save1), (int)s.rows,
          (int)s.K, (int)s.N, 0};
}

template <typename Cfg>
int launch_joint(const RoutedProblem& r, DenseProblem dp, hipStream_t stream) {
  constexpr int kSmem = (int)StreamLayout<Cfg>::kSmemBytes;
  static std::once_flag once;
  static hipError_t attr_err = hipSuccess;
  auto kernel = &grouped_gemm_joint_kernel<Cfg>;
  std::call_once(once, [&] {
    attr_err = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kSmem);
  });
  if (attr_err != hipSuccess)
    return fail(JTMOE_ELAUNCH, "grouped gemm: kernel set-up: %s", hipGetErrorString(attr_err));
  const int64_t least = std::min<int64_t>(r.K, dp.k);
  if (!fills_pipeline<Cfg>(least)) return fail(JTMOE_EUNSUPPORTED, "grouped gemm: reduction of %lld too short", (long long)least);
  const int64_t mtiles = max_m_tiles(r.rows, r.E, Cfg::BM), nt = (r.N + Cfg::BN - 1) / Cfg::BN;
  dp.ntiles = (dp.n + Cfg::BN - 1) / Cfg::BN;
  const int64_t tiles_grid = gemm_grid(mtiles, nt) + gemm_grid((dp.rows + Cfg::BM - 1) / Cfg::BM, dp.ntiles);
  if (tiles_grid >= ((int64_t)1 << 28)) return fail(JTMOE_EUNSUPPORTED, "grouped gemm: grid too large");
  const int64_t grid = std::min<int64_t>(tiles_grid, persistent_grid_size());
  kernel<<<(unsigned)grid, Cfg::NT, kSmem, stream>>>(
      static_cast<const uint16_t*>(r.a), static_cast<const uint16_t*>(r.b0), static_cast<const uint16_t*>(r.b1),
      static_cast<uint16_t*>(r.c), r.group_sizes, r.offsets, (int)r.E, (int)r.rows, (int)r.K, (int)r.N, (int)nt,
      r.row_map, r.row_div, (int)r.a_rows, static_cast<uint16_t*>(r.save0), static_cast<uint16_t*>(r.save1), dp);
  return JTMOE_OK;
}

// what the stream kernel needs beyond fast_ok: enough k steps to fill its pipeline, a result of at most
// 0x7ffe0000 bytes (32-bit store offsets; the kernel drops a store by giving it the offset 0x7fff0000,
// which must lie past the end of every admitted result) and, with a row map, fewer than 2^27 rows and a
// divisor of at most 32
template <typename Cfg>
inline bool stream_ok(int64_t rows, int64_t Kdim, int64_t N, const int32_t* row_map, int row_div) {
  return ((Cfg::OPT & 65536) != 0 || Kdim % Cfg::BK == 0) && fills_pipeline<Cfg>(Kdim) && rows * N * 2 <= (int64_t)0x7ffe0000 &&
         (row_map == nullptr || (rows < ((int64_t)1 << 27) && row_div >= 1 && row_div <= 32));
}

template <typename Cfg>
int launch_skinny(const void* a, const void* b0, const void* b1, void* c, const int32_t* group_sizes,
                  const int32_t* offsets, int64_t rows, int64_t Kdim, int64_t N, int64_t E, hipStream_t stream,
                  const int32_t* row_map = nullptr, int row_div = 1, int64_t a_rows = 0, void* save0 = nullptr,
                  void* save1 = nullptr, int64_t a_group_rows = 0, const Beside* beside = nullptr) {
  static_assert(Cfg::SMEM_BYTES <= 64 * 1024, "launched without a raised limit");
  const int64_t mtiles = group_sizes == nullptr ? (rows + Cfg::BM - 1) / Cfg::BM : max_m_tiles(rows, E, Cfg::BM);
  const int64_t nt = (N + Cfg::BN - 1) / Cfg::BN;
  const int64_t grid = gemm_grid(mtiles, nt);
  if (grid >= ((int64_t)1 << 31)) return fail(JTMOE_EUNSUPPORTED, "grouped gemm: grid too large");
  const SkinnyProblem p{static_cast<const uint16_t*>(a), static_cast<const uint16_t*>(b0), static_cast<const uint16_t*>(b1),
                        static_cast<uint16_t*>(c), static_cast<uint16_t*>(save0), static_cast<uint16_t*>(save1),
                        group_sizes, offsets, row_map, (int)E, (int)rows, (int)Kdim, (int)N, (int)mtiles, (int)nt, row_div,
                        (int)a_rows, (int)a_group_rows};
  if (beside)
    grouped_gemm_skinny_beside_kernel<Cfg><<<(unsigned)(grid + beside->blocks), Cfg::NT,
                                             std::max<int>(Cfg::SMEM_BYTES, BesideCfg::SMEM_BYTES), stream>>>(p, *beside);
  else
    grouped_gemm_skinny_kernel<Cfg><<<(unsigned)grid, Cfg::NT, Cfg::SMEM_BYTES, stream>>>(p);
  return JTMOE_OK;
}

// ---- which kernel takes a product ------------------------------------------------------------------------
// All times below: rows of T tokens in E groups by a balanced top-k, matrices cold, launch overhead included.
// Streaming tiles (grouped_gemm_skinny.hpp) while they find a CU each: of the shapes with at most one tile per CU
// the one with the most tiles, so that the matrices are drawn through as many CUs as possible.  us for gate/up and
// down together, 2048 -> 1408, 64 experts top-8, 1 token: 35 against 87 in 64-row LDS tiles; shared experts of 2816:
// 34 at 1 token, 36 at 64 (148 in 64-row LDS tiles), 43 at 130 with 32-row tiles (58 without them).  Tiles of 128
// columns and 32 or 64 rows do not pay where half tiles can be had: 68 against 53 at 387 tokens, 91 against 63 at 700.
// With more tiles than CUs, and up to four rows per group reached (a group's second tile reads its matrix again),
// they compete with the 64-row LDS tiles over the number that is resident at once.  Kernel times, us, LDS tiles, four to
// a CU, / streaming; 64 experts of 2048 -> 1408 and 128 of 2048 -> 768, top-8:
//   gate/up, LDS tiles as wide; streaming up to two tiles per CU.  64 experts: 8 tokens 76.1 / 74.0, 10 92.2 / 101.4, 15
//   102.3 / 105.3; 128: 8 tokens 65.4 / 66.0, 12 75.2 / 75.0, 20 96.5 / 101.1, 64 123.9 / 121.7.
//   down, LDS tiles 256 wide; streaming while all of its tiles are resident, three to a CU, and from more than two LDS tiles
//   per CU on, but not in between.  64 experts: 8 tokens 49.0 / 46.8, 10 48.4 / 50.3, 15 50.8 / 61.6, 64 57.8 / 75.5; 128: 8
//   tokens 28.8 / 33.8, 12 40.5 / 42.4, 20 45.9 / 47.3, 24 61.5 / 54.0, 37 66.2 / 63.2, 56 67.8 / 66.0.
// (The lines were drawn with three and two LDS tiles on a CU, which took longer; where they stand now they cost 4 to 10 % of
// a product at 10 tokens of 64 experts and 2 to 5 % of the down product at 12 to 20 tokens of 128.)
inline bool pick_skinny(int64_t rows, int64_t E, bool dense, int64_t N, bool dual, double cus, ProductKernel* out) {
  struct Shape {
    ProductKernel id;
    int RB, BN;
  };
  constexpr Shape shapes[] = {{ProductKernel::kStream16x64, 1, 64}, {ProductKernel::kStream32x64, 2, 64},
                              {ProductKernel::kStream16x128, 1, 128}};
  double most = 0.0;
  for (const Shape& s : shapes) {
    const double tiles = expected_mtiles(rows, E, dense, 16 * s.RB) * (double)((N + s.BN - 1) / s.BN);
    if (tiles <= cus && tiles > most) {
      most = tiles;
      *out = s.id;
    }
  }
  if (most == 0.0 && !dense && (double)rows <= 4.0 * expected_mtiles(rows, E, false, 16)) {
    const double tiles = expected_mtiles(rows, E, false, 16) * (double)((N + 127) / 128);
    const double lds_tiles = expected_mtiles(rows, E, false, 64) * (double)((N + 255) / 256);
    *out = ProductKernel::kStream16x128;
    return dual ? tiles <= 2.0 * cus : tiles <= 3.0 * cus || lds_tiles > 2.0 * cus;
  }
  return most > 0.0;
}

inline bool streaming_or_rows64(ProductKernel k) {
  return k == ProductKernel::kStream16x128 || k == ProductKernel::kStream16x64 || k == ProductKernel::kStream32x64 ||
         k == ProductKernel::kRows64 || k == ProductKernel::kRows64Tail;
}

// Rows per group up to which 64-row LDS tiles hold nearly every group in one tile: each expert matrix is then
// read by one row of workgroups, with non-temporal loads.  us for gate/up and down, 64 experts: mean 48 rows 121
// and 61 (256-row tiles 141 and 77), mean 64 rows, where half of the groups need a second tile, 203 and 103 (148
// and 78).
constexpr int64_t kTinyGroupRows = 52;  // four or fewer in a hundred groups above 64

// Then half tiles where they pay (half_tiles); gate/up only with at most one per CU: 1024 tokens, shared 2816: 41 us
// against 50 in 256-row tiles; with more, two rounds of half tiles: 2048 tokens 77 against 52.
ProductKernel gate_up_kernel(int64_t rows, int64_t H, int64_t I, int64_t E, bool dense, double cus,
                             const int32_t* row_map = nullptr, int row_div = 1) {
  const bool tail = H % 64 != 0;
  ProductKernel k;
  if (pick_skinny(rows, E, dense, I, true, cus, &k)) return k;
  if (!dense && rows <= kTinyGroupRows * E) return tail ? ProductKernel::kRows64Tail : ProductKernel::kRows64;
  if (half_tiles(rows, E, dense, I, cus) == HalfTiles::kOnePerCu &&
      stream_ok<GateUpHalfShortCfg<true>>(rows, H, I, row_map, row_div))
    return tail ? ProductKernel::kHalfTail : ProductKernel::kHalf;
  if (stream_ok<GateUpStreamTailCfg>(rows, H, I, row_map, row_div))
    return tail ? ProductKernel::kRows256Tail : ProductKernel::kRows256;
  return tail ? ProductKernel::kRows256ShortTail : ProductKernel::kRows256Short;
}

ProductKernel down_kernel(int64_t rows, int64_t H, int64_t I, int64_t E, bool dense, double cus) {
  ProductKernel k;
  if (pick_skinny(rows, E, dense, H, false, cus, &k)) return k;
  if (!dense && rows <= kTinyGroupRows * E) return ProductKernel::kRows64;
  const HalfTiles half = half_tiles(rows, E, dense, H, cus);
  if (half == HalfTiles::kOnePerCu && stream_ok<HalfShortCfg>(rows, I, H, nullptr, 1)) return ProductKernel::kHalf;
  if (half != HalfTiles::kNone && stream_ok<DownHalfDeepCfg>(rows, I, H, nullptr, 1)) return ProductKernel::kHalfDeep;
  return I % 64 == 0 ? ProductKernel::kRows256 : ProductKernel::kRows256Tail;
}

// Routed and shared experts in one launch (joint_tiles): the kernel of both, or kGeneral for launches of their own.
// Not with routed rows in streaming tiles, which a few rows per group are too few to give up.
// Not with the routed rows in 64-row tiles: those are resident all at once and share the memory's rate, and the shared
// tiles, whose matrices every 64 rows read again, take their share of it (387 tokens, 64 experts top-8 of 1408, shared
// 2816, 2048 wide: 158 us for gate/up together, 119 + 28 apart, 111 against 66 + 25 for down).
// Measured (us, gate/up and down, routed + shared apart against joint): 2048 tokens of that model 293 + 58 and
// 173 + 40 against 306 and 182; 2931 tokens, 1000 wide, 24 experts top-3 of 2664 and one shared, down 81 + 45
// against 94; 4096 tokens, 1024 wide, 8 experts top-2 of 2048 and one shared, down 55 + 29 against 62.
ProductKernel joint_gate_up(int64_t rows, int64_t H, int64_t I, int64_t E, int64_t T, int64_t Is, double cus,
                            const int32_t* row_map = nullptr, int row_div = 1) {
  const ProductKernel routed = gate_up_kernel(rows, H, I, E, false, cus, row_map, row_div);
  if (streaming_or_rows64(routed) || !stream_ok<GateUpStreamTailCfg>(rows, H, I, row_map, row_div) ||
      !stream_ok<GateUpStreamTailCfg>(T, H, Is, nullptr, 1))
    return ProductKernel::kGeneral;
  const bool tail = H % 64 != 0;
  switch (joint_tiles(rows, E, I, T, Is, 1.0, cus, 0.72, /*dual=*/true)) {
    case HalfTiles::kOnePerCu:
      // (H too short for the half tiles' deeper stages takes four 32-deep ones)
      if (!stream_ok<GateUpHalfShortCfg<true>>(rows, H, I, row_map, row_div)) return ProductKernel::kGeneral;
      return tail ? ProductKernel::kHalfTail : ProductKernel::kHalf;
    case HalfTiles::kRounds: return tail ? ProductKernel::kRows256Tail : ProductKernel::kRows256;
    default: return ProductKernel::kGeneral;
  }
}

ProductKernel joint_down(int64_t rows, int64_t H, int64_t I, int64_t E, int64_t T, int64_t Is, double cus) {
  if (streaming_or_rows64(down_kernel(rows, H, I, E, false, cus)) ||
      !stream_ok<DownStreamTailCfg>(rows, I, H, nullptr, 1) || !stream_ok<DownStreamTailCfg>(T, Is, H, nullptr, 1))
    return ProductKernel::kGeneral;
  switch (joint_tiles(rows, E, H, T, H, (double)Is / (double)I, cus, 0.4)) {
    case HalfTiles::kOnePerCu:
      return stream_ok<HalfShortCfg>(rows, std::min(I, Is), H, nullptr, 1) ? ProductKernel::kHalf : ProductKernel::kGeneral;
    case HalfTiles::kRounds: return I % 64 == 0 && Is % 64 == 0 ? ProductKernel::kRows256 : ProductKernel::kRows256Tail;
    default: return ProductKernel::kGeneral;
  }
}

inline bool fast_ok(const void* a, const void* b0, const void* b1, const void* c, int64_t Kdim, int64_t N) {
  return Kdim % 8 == 0 && N % 8 == 0 && Kdim * N < ((int64_t)1 << 30) && aligned16(a) && aligned16(b0) && (b1 == nullptr || aligned16(b1)) &&
         aligned16(c);
}

// ---- the tiles of a launch whose kernel the rules above have chosen -----------------------------------------
// (T rows times N1 columns with a reduction of K1 in the same launch, T = 0: none)
inline TileShape stream_tiles(Product product, ProductKernel k, int64_t rows, int64_t K, int64_t N, int64_t E, bool dense,
                              double cus, int64_t T = 0, int64_t K1 = 0, int64_t N1 = 0) {
  const bool half = k == ProductKernel::kHalf || k == ProductKernel::kHalfTail;
  const int64_t least = T ? std::min(K, K1) : K;
  TileShape s = tile_shape(product, rows, E, dense, N, cus, T, N1);
  if (s == TileShape::kPlain && (least + 31) / 32 < 8) s = TileShape::kTall;  // (plain tiles have four 32-deep stages here)
  return tile_shape_for(s, half, (least + 63) / 64, product == Product::kGateUp);
}

// kHalf to kRows256Tail, with the activations as they are; kTall, kPlain: 256-row tiles of the stream kernel and of the other
TileShape down_tiles(ProductKernel k, int64_t rows, int64_t H, int64_t I, int64_t E, bool dense, double cus) {
  const TileShape tiles = stream_tiles(Product::kDown, k, rows, I, H, E, dense, cus);
  const bool streams = stream_ok<DownStreamTailCfg>(rows, I, H, nullptr, 1);
  if (k == ProductKernel::kHalfDeep) {
    // Two half tiles per CU only where few CUs get a second one (4252 rows 2616 -> 1080, 306 of them: 50 us, 153 tiles of 256 x
    // 128 57; groups of 250 rows, 296 of them, 55 and 46), or for want of steps (128 groups of 56 rows, skewed, 768 -> 2048: 92
    // us against 97 in half tiles).
    if (dense && 4 * ((rows + 127) / 128) * ((H + 127) / 128) <= 5 * (int64_t)cus) return TileShape::k128x128Pair;
    const TileShape smaller = large_tiles(tiles) ? tile_shape_for(TileShape::k128x256, false, (I + 63) / 64, false) : tiles;
    return streams && !large_tiles(smaller) ? smaller : TileShape::k128x128Pair;
  }
  if (streams && (!large_tiles(tiles) || tiles == TileShape::kTall)) return tiles;
  return TileShape::kPlain;  // also for a reduction too short for the stream kernel, or a result past its limit
}

// y = act Wd[e] on the matrix cores (fast_ok holds); with a map, packed row j reads row row_map[j] / row_div of
// its group's block of a_group_rows rows (the decode path), and the tiles of `beside` run in the same launch
int launch_down_fast(const void* act, const void* down, const int32_t* group_sizes, const int32_t* offsets,
                     int64_t rows, int64_t H, int64_t I, int64_t E, void* y, hipStream_t stream,
                     const int32_t* row_map = nullptr, int row_div = 1, int64_t a_group_rows = 0,
                     const Beside* beside = nullptr) {
#define JT_DOWN(LAUNCH, CFG) LAUNCH<CFG>(act, down, nullptr, y, group_sizes, offsets, rows, I, H, E, stream, row_map, row_div, a_group_rows, nullptr, nullptr
  using S11 = SkinnyCfg<1, 1, false>;
  using S12 = SkinnyCfg<1, 2, false>;
  using S22 = SkinnyCfg<2, 2, false>;
  const ProductKernel k = down_kernel(rows, H, I, E, group_sizes == nullptr, persistent_grid_size());
  switch (k) {
    case ProductKernel::kStream16x128: return JT_DOWN(launch_skinny, S11), a_group_rows, beside);
    case ProductKernel::kStream16x64: return JT_DOWN(launch_skinny, S12), a_group_rows, beside);
    case ProductKernel::kStream32x64: return JT_DOWN(launch_skinny, S22), a_group_rows, beside);
    case ProductKernel::kRows64: return JT_DOWN(launch_fast, DownTinyCfg), 0, a_group_rows, beside);
    default: break;
  }
  // (at most half a tile of rows per group on the decode path: the rules above take all of it)
  if (row_map || beside) return fail(JTMOE_EUNSUPPORTED, "grouped gemm: no down kernel reads blocks of rows per group at this size");
  const bool tail = k == ProductKernel::kRows256Tail;
  switch (const TileShape tiles = down_tiles(k, rows, H, I, E, group_sizes == nullptr, persistent_grid_size())) {
    case TileShape::k128x128Pair: return JT_DOWN(launch_stream, DownHalfDeepCfg), 2);
    case TileShape::kTall:
      if (tail) return JT_DOWN(launch_stream, DownStreamTailCfg));
      return JT_DOWN(launch_stream, DownStreamCfg));
    case TileShape::kPlain:
      if (tail) return JT_DOWN(launch_fast, DownTailCfg));
      return JT_DOWN(launch_fast, DownCfg));
    default: return with_smaller_tiles<true>(tiles, [&](auto cfg) { return JT_DOWN(launch_stream, decltype(cfg))); });
  }
#undef JT_DOWN
}

// (`beside`: streaming and 64-row tiles take these tiles along, and say so)
template <typename T>
int launch_gate_up(const RoutedProblem& p, hipStream_t stream, const Beside* beside = nullptr,
                   bool* beside_taken = nullptr) {
  const bool dense = p.group_sizes == nullptr;
  const bool gather_ok = p.row_map == nullptr || p.a_rows * p.K < ((int64_t)1 << 30);
  const bool saves_ok = aligned16(p.save0) && aligned16(p.save1);
#define JT_GATE_UP(LAUNCH, CFG, ...)                                                                             \
  LAUNCH<CFG>(p.a, p.b0, p.b1, p.c, p.group_sizes, p.offsets, p.rows, p.K, p.N, p.E, stream, p.row_map, p.row_div, \
              p.a_rows, p.save0, p.save1 __VA_ARGS__)
#define JT_BESIDE , 0, beside
#define JT_BESIDE64 , 0, 0, beside
  if (Elem<T>::is_bf16 && fast_ok(p.a, p.b0, p.b1, p.c, p.K, p.N) && gather_ok && saves_ok) {
    using S11 = SkinnyCfg<1, 1, true>;
    using S12 = SkinnyCfg<1, 2, true>;
    using S22 = SkinnyCfg<2, 2, true>;
    const ProductKernel k = gate_up_kernel(p.rows, p.K, p.N, p.E, dense, persistent_grid_size(), p.row_map, p.row_div);
    if (beside) *beside_taken = streaming_or_rows64(k) && k != ProductKernel::kRows64Tail;
    auto tiles = [&](ProductKernel k) { return stream_tiles(Product::kGateUp, k, p.rows, p.K, p.N, p.E, dense, persistent_grid_size()); };
    switch (k) {
      case ProductKernel::kStream16x128: return JT_GATE_UP(launch_skinny, S11, JT_BESIDE);
      case ProductKernel::kStream16x64: return JT_GATE_UP(launch_skinny, S12, JT_BESIDE);
      case ProductKernel::kStream32x64: return JT_GATE_UP(launch_skinny, S22, JT_BESIDE);
      case ProductKernel::kRows64: return JT_GATE_UP(launch_fast, GateUpTinyCfg, JT_BESIDE64);
      case ProductKernel::kRows64Tail: return JT_GATE_UP(launch_fast, GateUpTinyTailCfg);
      case ProductKernel::kHalf:
      case ProductKernel::kRows256:
        return with_gate_up_tiles<false, false>(tiles(k), [&](auto cfg) { return JT_GATE_UP(launch_stream, decltype(cfg)); });
      case ProductKernel::kHalfTail:
      case ProductKernel::kRows256Tail:
        return with_gate_up_tiles<true, false>(tiles(k), [&](auto cfg) { return JT_GATE_UP(launch_stream, decltype(cfg)); });
      case ProductKernel::kRows256Short: return JT_GATE_UP(launch_fast, GateUpCfg);
      default: return JT_GATE_UP(launch_fast, GateUpTailCfg);
    }
  }
#undef JT_BESIDE64
#undef JT_BESIDE
#undef JT_GATE_UP
  if (!Elem<T>::is_bf16 && f32_gemm_supported(p.a, p.save0, p.b0, p.b1, p.c, p.row_map ? p.a_rows : p.rows, p.K, p.N) &&
      aligned16(p.save1))
    return launch_f32_nn(p.a, p.b0, p.b1, p.c, p.group_sizes, p.offsets, p.rows, p.K, p.N, p.E, p.row_map, p.row_div,
                         p.a_rows, p.save0, p.save1, stream);
  return launch_generic<T, true>(p.a, p.b0, p.b1, p.c, p.group_sizes, p.offsets, p.rows, p.K, p.N, p.E, stream,
                                 p.row_map, p.row_div, p.save0, p.save1);
}

template <typename T>
int launch_down(const RoutedProblem& p, hipStream_t stream) {
  if (Elem<T>::is_bf16 && fast_ok(p.a, p.b0, nullptr, p.c, p.K, p.N))
    return launch_down_fast(p.a, p.b0, p.group_sizes, p.offsets, p.rows, p.N, p.K, p.E, p.c, stream);
  if (!Elem<T>::is_bf16 && f32_gemm_supported(p.a, nullptr, p.b0, nullptr, p.c, p.rows, p.K, p.N))
    return launch_f32_nn(p.a, p.b0, nullptr, p.c, p.group_sizes, p.offsets, p.rows, p.K, p.N, p.E, nullptr, 1, 0,
                         nullptr, nullptr, stream);
  return launch_generic<T, false>(p.a, p.b0, nullptr, p.c, p.group_sizes, p.offsets, p.rows, p.K, p.N, p.E, stream);
}

// A product of the routed experts and of the shared ones in one launch: the kernel that the rules above choose, or
// kGeneral where they or the operands ask for launches of their own.
ProductKernel joint_gate_up_of(const RoutedProblem& p, const RoutedProblem& s) {
  const bool ok = (p.row_map == nullptr || p.a_rows * p.K < ((int64_t)1 << 30)) && fast_ok(p.a, p.b0, p.b1, p.c, p.K, p.N) &&
                  fast_ok(s.a, s.b0, s.b1, s.c, s.K, s.N) && aligned16(p.save0) && aligned16(p.save1) &&
                  aligned16(s.save0) && aligned16(s.save1);
  return ok ? joint_gate_up(p.rows, p.K, p.N, p.E, s.rows, s.N, persistent_grid_size(), p.row_map, p.row_div)
            : ProductKernel::kGeneral;
}

ProductKernel joint_down_of(const RoutedProblem& p, const RoutedProblem& s) {
  const bool ok = fast_ok(p.a, p.b0, nullptr, p.c, p.K, p.N) && fast_ok(s.a, s.b0, nullptr, s.c, s.K, s.N);
  return ok ? joint_down(p.rows, p.N, p.K, p.E, s.rows, s.K, persistent_grid_size()) : ProductKernel::kGeneral;
}

// Gate/up and down of both kinds of experts.  In launches of their own the shared pair follows the routed one, whose
// activations are then read while the caches hold them (800 and 1300 tokens, 64 experts top-8: 1.5 % of a call).
template <typename T>
int launch_with_shared(const RoutedProblem& gu, const RoutedProblem& dn, const RoutedProblem& sgu,
                       const RoutedProblem& sdn, hipStream_t stream, bool gate_up_done, bool down_done) {
  const ProductKernel jg = Elem<T>::is_bf16 && !gate_up_done ? joint_gate_up_of(gu, sgu) : ProductKernel::kGeneral;
  const ProductKernel jd = Elem<T>::is_bf16 && !down_done ? joint_down_of(dn, sdn) : ProductKernel::kGeneral;
  const bool joint_gu = jg != ProductKernel::kGeneral, joint_dn = jd != ProductKernel::kGeneral;
  const DenseProblem dgu = dense_problem(sgu), ddn = dense_problem(sdn);
  auto gate_up = [&](auto cfg) { return launch_joint<decltype(cfg)>(gu, dgu, stream); };
  auto down = [&](auto cfg) { return launch_joint<decltype(cfg)>(dn, ddn, stream); };
  int rc;
  auto tiles_with = [](Product product, ProductKernel k, const RoutedProblem& p, const RoutedProblem& s) {
    return stream_tiles(product, k, p.rows, p.K, p.N, p.E, false, persistent_grid_size(), s.rows, s.K, s.N);
  };
  if (!joint_gu) {
    rc = launch_gate_up<T>(gu, stream);
  } else {
    const TileShape tiles = tiles_with(Product::kGateUp, jg, gu, sgu);
    const bool tail = jg == ProductKernel::kHalfTail || jg == ProductKernel::kRows256Tail;
    rc = tail ? with_gate_up_tiles<true, true>(tiles, gate_up) : with_gate_up_tiles<false, true>(tiles, gate_up);
  }
  if (!rc && !gate_up_done && !joint_gu && joint_dn) rc = launch_gate_up<T>(sgu, stream);
  if (rc) return rc;
  if (!joint_dn) {
    rc = launch_down<T>(dn, stream);
  } else {
    const TileShape tiles = tiles_with(Product::kDown, jd, dn, sdn);
    const bool tail = jd == ProductKernel::kRows256Tail;
    if (tiles == TileShape::kPlain)
      rc = tail ? down(DownPlainCfg<true>{}) : down(DownPlainCfg<false>{});
    else if (tiles == TileShape::kTall)
      rc = tail ? down(DownStreamTailCfg{}) : down(DownStreamCfg{});
    else
      rc = with_smaller_tiles<true>(tiles, down);
  }
  if (!rc && !gate_up_done && !joint_gu && !joint_dn) rc = launch_gate_up<T>(sgu, stream);
  if (!rc && !down_done && !joint_dn) rc = launch_down<T>(sdn, stream);
  return rc;
}

template <typename T>
int launch_pair(const void* x, const void* gate, const void* up, const void* down, const int32_t* group_sizes,
                const int32_t* offsets, int64_t rows, int64_t H, int64_t I, int64_t E, void* act, void* y,
                hipStream_t stream, int first_stage, const int32_t* row_map = nullptr, int row_div = 1,
                int64_t x_rows = 0, void* save_gate = nullptr, void* save_up = nullptr,
                const SharedExperts* shared = nullptr) {
  if (rows == 0) return JTMOE_OK;
  const RoutedProblem gu{x, gate, up, act, save_gate, save_up, group_sizes, offsets, row_map, rows, H, I, E, x_rows, row_div};
  const RoutedProblem dn{act, down, nullptr, y, nullptr, nullptr, group_sizes, offsets, nullptr, rows, I, H, E, 0, 1};
  int rc = JTMOE_OK;
  if (shared != nullptr) {
    const RoutedProblem sgu{x, shared->gate, shared->up, shared->act, shared->gate_pre, shared->up_pre, nullptr, nullptr,
                            nullptr, x_rows, H, shared->Is, 1, 0, 1};
    const RoutedProblem sdn{shared->act, shared->down, nullptr, shared->y, nullptr, nullptr, nullptr, nullptr, nullptr,
                            x_rows, shared->Is, H, 1, 0, 1};
    if (shared->few_rows) {
      // (a few tokens: the router has run the shared gate/up product, its down product goes beside the routed gate/up)
      const SkinnyProblem down_p = dense_skinny(shared->act, shared->down, nullptr, shared->y, nullptr, nullptr, x_rows,
                                                shared->Is, H, BesideCfg::BM, BesideCfg::BN);
      const Beside beside{down_p, (int)gemm_grid(down_p.mtiles, down_p.ntiles_n)};
      bool taken = false;
      rc = launch_gate_up<T>(gu, stream, &beside, &taken);
      if (!rc) rc = launch_down<T>(dn, stream);
      if (!rc && !taken) rc = launch_down<T>(sdn, stream);
      return rc ? rc : check_launch("grouped gemm");
    }
    rc = launch_with_shared<T>(gu, dn, sgu, sdn, stream, shared->gate_up_done, shared->down_done);
    return rc ? rc : check_launch("grouped gemm");
  }
  rc = launch_gate_up<T>(gu, stream);
  if (rc) return rc;
  stage_mark(first_stage, stream);
  rc = launch_down<T>(dn, stream);
  if (rc) return rc;
  stage_mark(first_stage + 1, stream);
  return check_launch("grouped gemm");
}

int validate_gemm(const char* what, int64_t rows, int64_t H, int64_t I, int64_t E, int dtype) {
  JT_REQUIRE(dtype_ok(dtype), "%s: unknown dtype %d", what, dtype);
  JT_REQUIRE(rows >= 0 && rows < ((int64_t)1 << 31), "%s: row count %lld out of range", what, (long long)rows);
  JT_REQUIRE(H > 0 && I > 0 && E > 0, "%s: H=%lld I=%lld E=%lld out of range", what, (long long)H, (long long)I,
             (long long)E);
  JT_REQUIRE(H < ((int64_t)1 << 24) && I < ((int64_t)1 << 24), "%s: H or I too large", what);
  return JTMOE_OK;
}

}  // namespace

// ---- the down launch of the layer's decode path (declared in common.hpp) ----
int launch_down_from_all_tokens(const void* act_full, const void* down, const int32_t* group_sizes,
                                const int32_t* offsets, const int32_t* source_order, int64_t T, int64_t K, int64_t H,
                                int64_t I, int64_t E, void* packed_y, hipStream_t stream, const SharedExperts* shared) {
  if (!fast_ok(act_full, down, nullptr, packed_y, I, H))
    return fail(JTMOE_EINVAL, "moe_forward: operands must be 16-byte aligned");
  if (!shared)
    return launch_down_fast(act_full, down, group_sizes, offsets, T * K, H, I, E, packed_y, stream, source_order, (int)K,
                            /*a_group_rows=*/T);
  const SkinnyProblem p = dense_skinny(shared->act, shared->down, nullptr, shared->y, nullptr, nullptr, T, shared->Is, H,
                                       BesideCfg::BM, BesideCfg::BN);
  const Beside beside{p, (int)gemm_grid(p.mtiles, p.ntiles_n)};
  return launch_down_fast(act_full, down, group_sizes, offsets, T * K, H, I, E, packed_y, stream, source_order, (int)K,
                          /*a_group_rows=*/T, &beside);
}

bool shared_in_skinny_tiles(const void* x, const SharedExperts& s, int64_t T, int64_t H) {
  return fast_ok(x, s.gate, s.up, s.act, H, s.Is) && fast_ok(s.act, s.down, nullptr, s.y, s.Is, H) &&
         aligned16(s.gate_pre) && aligned16(s.up_pre) &&
         gate_up_kernel(T, H, s.Is, 1, true, persistent_grid_size()) == ProductKernel::kStream16x64 &&
         down_kernel(T, H, s.Is, 1, true, persistent_grid_size()) == ProductKernel::kStream16x64;
}

// ---- products of the shared experts beside the small launches in front of the routed ones ----
// Both take tiles that find a CU each; they run on as they would alone, and the launch beside them, a few workgroups and
// 7 to 12 us, costs nothing.  Sizes whose products are parts of the routed launches (joint_gate_up, joint_down) stay there.
// (kPlain: none)
TileShape tiles_beside(Product product, int64_t T, int64_t H, int64_t Is, int64_t I, int64_t E, int64_t K, int front,
                       double cus) {
  const bool dual = product == Product::kGateUp;
  const ProductKernel k = dual ? gate_up_kernel(T, H, Is, 1, true, cus) : down_kernel(T, H, Is, 1, true, cus);
  const bool joint = (dual ? joint_gate_up(T * K, H, I, E, T, Is, cus) : joint_down(T * K, H, I, E, T, Is, cus)) != ProductKernel::kGeneral;
  // (gate/up of whole reductions only: see dense_stream_tiles)
  const bool streams = k == ProductKernel::kHalf || (dual ? k == ProductKernel::kRows256
                                                          : (k == ProductKernel::kRows256 || k == ProductKernel::kRows256Tail) &&
                                                                stream_ok<DownStreamTailCfg>(T, Is, H, nullptr, 1));
  if (joint || !streams) return TileShape::kPlain;
  const int64_t N = dual ? Is : H;
  const TileShape tiles = stream_tiles(product, k, T, dual ? H : Is, N, 1, true, cus);
  if (tiles != TileShape::k64x64 && tiles != TileShape::k128x64) return TileShape::kPlain;
  const int BM = tiles == TileShape::k64x64 ? 64 : 128;
  return front + gemm_grid((T + BM - 1) / BM, (N + 63) / 64) <= (int64_t)cus ? tiles : TileShape::kPlain;
}

namespace {

SharedTiles beside_front(const RoutedProblem& s, TileShape tiles) {
  if (tiles == TileShape::kPlain) return SharedTiles{};
  SharedTiles t{tiles, dense_problem(s), 0};
  t.p.ntiles = (int)((s.N + 63) / 64);
  const int BM = tiles == TileShape::k64x64 ? 64 : 128;
  t.grid = (int)gemm_grid((s.rows + BM - 1) / BM, t.p.ntiles);
  return t;
}

struct DispatchPlan {
  const int32_t* ids;
  const bf16_raw* weights;
  int A, E;
  int32_t *group_sizes, *offsets, *source_order, *inverse;
  float *counts, *importance;
};

template <typename Cfg>
__global__ __launch_bounds__(Cfg::NT) void dispatch_beside_kernel(DispatchPlan d, DenseProblem shared) {
  static_assert(JTMOE_MAX_EXPERTS <= Cfg::NT, "an expert per thread of the dispatch");
  extern __shared__ __align__(16) unsigned char smem_raw[];
  if ((int)blockIdx.x >= kDispatchFront)
    dense_stream_tiles<Cfg>(shared, kDispatchFront);
  else if (blockIdx.x == 0)
    dispatch_small_body<Cfg::NT, true, bf16_raw>(d.ids, d.weights, d.A, d.E, d.group_sizes, d.offsets, d.source_order,
                                                 d.inverse, d.counts, d.importance, smem_raw);
}

}  // namespace

SharedTiles shared_gate_up_beside(const void* x, const SharedExperts& s, int64_t T, int64_t H, int64_t E, int64_t K, int front) {
  if (!fast_ok(x, s.gate, s.up, s.act, H, s.Is) || !aligned16(s.gate_pre) || !aligned16(s.up_pre)) return SharedTiles{};
  return beside_front({x, s.gate, s.up, s.act, s.gate_pre, s.up_pre, nullptr, nullptr, nullptr, T, H, s.Is, 1, 0, 1},
                      tiles_beside(Product::kGateUp, T, H, s.Is, s.routed_I, E, K, front, persistent_grid_size()));
}

SharedTiles shared_down_beside(const SharedExperts& s, int64_t T, int64_t H, int64_t E, int64_t K, int front) {
  if (!fast_ok(s.act, s.down, nullptr, s.y, s.Is, H)) return SharedTiles{};
  return beside_front({s.act, s.down, nullptr, s.y, nullptr, nullptr, nullptr, nullptr, nullptr, T, s.Is, H, 1, 0, 1},
                      tiles_beside(Product::kDown, T, H, s.Is, s.routed_I, E, K, front, persistent_grid_size()));
}

int launch_dispatch_beside_shared(const int32_t* ids, const void* weights, const void* x, int64_t T, int64_t H, int64_t E,
                                  int64_t K, int32_t* group_sizes, int32_t* offsets, int32_t* source_order,
                                  int32_t* inverse, float* counts, float* importance, SharedExperts& shared, bool* taken,
                                  hipStream_t stream) {
  const bool down = shared.gate_up_done;
  const SharedTiles t = down ? shared_down_beside(shared, T, H, E, K, kDispatchFront)
                             : shared_gate_up_beside(x, shared, T, H, E, K, kDispatchFront);
  if (t.grid == 0) return JTMOE_OK;
  const DispatchPlan plan{ids, static_cast<const bf16_raw*>(weights), (int)(T * K), (int)E, group_sizes, offsets,
                          source_order, inverse, counts, importance};
  auto launch = [&](auto cfg) {
    using Cfg = decltype(cfg);
    const size_t smem = std::max<size_t>(StreamLayout<Cfg>::kSmemBytes, dispatch_small_smem_bytes((int)E, Cfg::NT, true));
    static std::once_flag once;
    static hipError_t attr_err = hipSuccess;
    auto kernel = &dispatch_beside_kernel<Cfg>;
    std::call_once(once, [&] {
      attr_err = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     160 * 1024);
    });
    if (attr_err != hipSuccess) return fail(JTMOE_ELAUNCH, "dispatch: kernel set-up: %s", hipGetErrorString(attr_err));
    kernel<<<kDispatchFront + t.grid, Cfg::NT, smem, stream>>>(plan, t.p);
    *taken = true;
    (down ? shared.down_done : shared.gate_up_done) = true;
    return check_launch("dispatch and shared experts");
  };
  const bool quarter = t.tiles == TileShape::k64x64;
  if (down) return quarter ? launch(QuarterCfg{}) : launch(NarrowCfg{});
  return quarter ? launch(GateUpQuarterCfg<false>{}) : launch(GateUpNarrowCfg<false>{});
}

// ---- the gathering launch pair as the layer uses it (declared in common.hpp) ----
int launch_swiglu_gather(const void* x, const int32_t* source_order, const void* gate, const void* up,
                         const void* down, const int32_t* group_sizes, const int32_t* offsets, int64_t T, int64_t K,
                         int64_t H, int64_t I, int64_t E, int dtype, void* act, void* packed_y, hipStream_t stream,
                         const SharedExperts* shared, void* gate_pre, void* up_pre) {
  int rc = validate_gemm("grouped_swiglu_gather", T * K, H, I, E, dtype);
  if (rc) return rc;
  if (T > 0)
    JT_REQUIRE(x && source_order && gate && up && down && group_sizes && offsets && act && packed_y,
               "grouped_swiglu_gather: null pointer argument");
  if (shared != nullptr) {
    rc = validate_gemm("shared_swiglu", T, H, shared->Is, 1, dtype);
    if (rc) return rc;
    JT_REQUIRE(shared->gate && shared->up && shared->down && shared->act && shared->y, "shared_swiglu: null pointer argument");
  }
  if (dtype == JTMOE_BF16)
    return launch_pair<bf16_raw>(x, gate, up, down, group_sizes, offsets, T * K, H, I, E, act, packed_y, stream,
                                 kStageGateUp, source_order, (int)K, T, gate_pre, up_pre, shared);
  return launch_pair<float>(x, gate, up, down, group_sizes, offsets, T * K, H, I, E, act, packed_y, stream,
                            kStageGateUp, source_order, (int)K, T, gate_pre, up_pre, shared);
}

}  // namespace jtmoe

using namespace jtmoe;

extern "C" int jtmoe_grouped_swiglu(const void* packed_x, const void* gate, const void* up, const void* down,
                                    const int32_t* group_sizes, const int32_t* offsets, int64_t A, int64_t H,
                                    int64_t I, int64_t E, int dtype, void* act, void* packed_y, void* stream) {
  clear_error();
  int rc = validate_gemm("grouped_swiglu", A, H, I, E, dtype);
  if (rc) return rc;
  if (E > JTMOE_MAX_EXPERTS) return fail(JTMOE_EUNSUPPORTED, "grouped_swiglu: E=%lld exceeds %d", (long long)E, JTMOE_MAX_EXPERTS);
  if (A == 0) return JTMOE_OK;
  JT_REQUIRE(packed_x && gate && up && down && group_sizes && offsets && act && packed_y,
             "grouped_swiglu: null pointer argument");
  hipStream_t s = as_stream(stream);
  if (dtype == JTMOE_BF16)
    return launch_pair<bf16_raw>(packed_x, gate, up, down, group_sizes, offsets, A, H, I, E, act, packed_y, s, kStageGateUp);
  return launch_pair<float>(packed_x, gate, up, down, group_sizes, offsets, A, H, I, E, act, packed_y, s, kStageGateUp);
}

extern "C" int jtmoe_shared_swiglu(const void* x, const void* gate, const void* up, const void* down, int64_t T,
                                   int64_t H, int64_t Is, int dtype, void* act, void* shared_y, void* stream) {
  clear_error();
  int rc = validate_gemm("shared_swiglu", T, H, Is, 1, dtype);
  if (rc) return rc;
  if (T == 0) return JTMOE_OK;
  JT_REQUIRE(x && gate && up && down && act && shared_y, "shared_swiglu: null pointer argument");
  hipStream_t s = as_stream(stream);
  if (dtype == JTMOE_BF16)
    return launch_pair<bf16_raw>(x, gate, up, down, nullptr, nullptr, T, H, Is, 1, act, shared_y, s, kStageSharedGateUp);
  return launch_pair<float>(x, gate, up, down, nullptr, nullptr, T, H, Is, 1, act, shared_y, s, kStageSharedGateUp);
}

// the kernels that the rules above choose, by name
static const char* const kProductKernelNames[] = {"general", "stream_16x128", "stream_16x64", "stream_32x64", "rows64",
                                                  "rows64_tail", "half", "half_tail", "half_deep", "rows256",
                                                  "rows256_tail", "rows256_short", "rows256_short_tail"};

static bool product_sizes_ok(int product, int64_t rows, int64_t K, int64_t N, int64_t E, int compute_units) {
  return product >= 0 && product <= 3 && rows > 0 && K > 0 && N > 0 && E >= 0 && K < ((int64_t)1 << 24) &&
         N < ((int64_t)1 << 24) && rows < ((int64_t)1 << 31) && compute_units >= 0;
}

static ProductKernel product_kernel(int product, int64_t rows, int64_t K, int64_t N, int64_t groups, bool dense, double cus) {
  if (product >= 2) return data_gradient_kernel(rows, K, N, groups, dense, product - 1, cus);
  if (!fast_ok(nullptr, nullptr, nullptr, nullptr, K, N)) return ProductKernel::kGeneral;
  return product == 0 ? gate_up_kernel(rows, K, N, groups, dense, cus) : down_kernel(rows, N, K, groups, dense, cus);
}

extern "C" const char* jtmoe_product_kernel(int product, int64_t rows, int64_t K, int64_t N, int64_t E, int compute_units) {
  if (!product_sizes_ok(product, rows, K, N, E, compute_units)) return "";
  const double cus = compute_units > 0 ? compute_units : persistent_grid_size();
  return kProductKernelNames[(int)product_kernel(product, rows, K, N, E == 0 ? 1 : E, E == 0, cus)];
}

// ... and their tiles; "_tail" where a ragged reduction has a variant of its own
static const char* tile_name(TileShape s, bool tail) {
  static const char* const names[][2] = {{"64x64", "64x64_tail"}, {"128x64", "128x64_tail"}, {"128x128", "128x128_tail"},
                                         {"128x128_short", "128x128_short_tail"}, {"128x128_pair", "128x128_pair"},
                                         {"256x128", "256x128"}, {"128x256", "128x256"}, {"tall", "tall_tail"},
                                         {"plain", "plain_tail"}};
  return names[(int)s][tail];
}

extern "C" const char* jtmoe_product_tiles(int product, int64_t rows, int64_t K, int64_t N, int64_t E, int compute_units) {
  if (!product_sizes_ok(product, rows, K, N, E, compute_units)) return "";
  const bool dense = E == 0;
  const double cus = compute_units > 0 ? compute_units : persistent_grid_size();
  const int64_t groups = dense ? 1 : E;
  const ProductKernel k = product_kernel(product, rows, K, N, groups, dense, cus);
  if (k == ProductKernel::kGeneral || streaming_or_rows64(k) || k == ProductKernel::kRows256Short || k == ProductKernel::kRows256ShortTail)
    return kProductKernelNames[(int)k];
  if (product == 0)
    return tile_name(stream_tiles(Product::kGateUp, k, rows, K, N, groups, dense, cus),
                     k == ProductKernel::kHalfTail || k == ProductKernel::kRows256Tail);
  const TileShape s = product == 1 ? down_tiles(k, rows, N, K, groups, dense, cus)
                                   : data_gradient_tiles(k, rows, K, N, groups, dense, product - 1, cus);
  return tile_name(s, k == ProductKernel::kRows256Tail && large_tiles(s));
}

static bool joint_sizes_ok(int product, int64_t T, int64_t top_k, int64_t H, int64_t I, int64_t Is, int64_t E,
                           int compute_units) {
  const int64_t limit = (int64_t)1 << 24;
  return product >= 0 && product <= 3 && T > 0 && top_k > 0 && H > 0 && I > 0 && Is > 0 && E > 0 && H < limit &&
         I < limit && Is < limit && T * top_k < ((int64_t)1 << 31) && compute_units >= 0;
}

static ProductKernel joint_kernel(int product, int64_t T, int64_t top_k, int64_t H, int64_t I, int64_t Is, int64_t E, double cus) {
  if (product >= 2) return joint_data_gradient_kernel(T * top_k, H, I, E, T, Is, product - 1, cus);
  if (!fast_ok(nullptr, nullptr, nullptr, nullptr, H, I) || !fast_ok(nullptr, nullptr, nullptr, nullptr, H, Is))
    return ProductKernel::kGeneral;
  return product == 0 ? joint_gate_up(T * top_k, H, I, E, T, Is, cus) : joint_down(T * top_k, H, I, E, T, Is, cus);
}

extern "C" const char* jtmoe_joint_kernel(int product, int64_t T, int64_t top_k, int64_t H, int64_t I, int64_t Is,
                                          int64_t E, int compute_units) {
  if (!joint_sizes_ok(product, T, top_k, H, I, Is, E, compute_units)) return "";
  const double cus = compute_units > 0 ? compute_units : persistent_grid_size();
  const ProductKernel k = joint_kernel(product, T, top_k, H, I, Is, E, cus);
  return k == ProductKernel::kGeneral ? "separate" : kProductKernelNames[(int)k];
}

extern "C" const char* jtmoe_joint_tiles(int product, int64_t T, int64_t top_k, int64_t H, int64_t I, int64_t Is,
                                         int64_t E, int compute_units) {
  if (!joint_sizes_ok(product, T, top_k, H, I, Is, E, compute_units)) return "";
  const double cus = compute_units > 0 ? compute_units : persistent_grid_size();
  const int64_t rows = T * top_k;
  const ProductKernel k = joint_kernel(product, T, top_k, H, I, Is, E, cus);
  if (k == ProductKernel::kGeneral) return "separate";
  const bool tail = k == ProductKernel::kHalfTail || k == ProductKernel::kRows256Tail;
  if (product == 0) return tile_name(stream_tiles(Product::kGateUp, k, rows, H, I, E, false, cus, T, H, Is), tail);
  const TileShape s = product == 1   ? stream_tiles(Product::kDown, k, rows, I, H, E, false, cus, T, Is, H)
                      : product == 2 ? joint_data_gradient_tiles(k, rows, H, I, E, T, H, Is, 1, cus)
                                     : joint_data_gradient_tiles(k, rows, I, H, E, T, Is, H, 2, cus);
  return tile_name(s, tail && large_tiles(s));
}

extern "C" int jtmoe_grouped_swiglu_gather_supported(int64_t T, int64_t H, int64_t I, int dtype) {
  return dtype == JTMOE_BF16 && H % 64 == 0 && I % 64 == 0 && H * I < ((int64_t)1 << 30) &&
         T * H < ((int64_t)1 << 29);
}

extern "C" int jtmoe_grouped_swiglu_gather(const void* x, const int32_t* source_order, const void* gate,
                                           const void* up, const void* down, const int32_t* group_sizes,
                                           const int32_t* offsets, int64_t T, int64_t K, int64_t H, int64_t I,
                                           int64_t E, int dtype, void* act, void* packed_y, void* stream) {
  clear_error();
  JT_REQUIRE(T >= 0 && K > 0 && T * K < ((int64_t)1 << 31), "grouped_swiglu_gather: T=%lld K=%lld out of range",
             (long long)T, (long long)K);
  const int64_t A = T * K;
  int rc = validate_gemm("grouped_swiglu_gather", A, H, I, E, dtype);
  if (rc) return rc;
  if (E > JTMOE_MAX_EXPERTS)
    return fail(JTMOE_EUNSUPPORTED, "grouped_swiglu_gather: E=%lld exceeds %d", (long long)E, JTMOE_MAX_EXPERTS);
  if (A == 0) return JTMOE_OK;
  JT_REQUIRE(x && source_order && gate && up && down && group_sizes && offsets && act && packed_y,
             "grouped_swiglu_gather: null pointer argument");
  if (!jtmoe_grouped_swiglu_gather_supported(T, H, I, dtype) || !aligned16(x))
    return fail(JTMOE_EUNSUPPORTED,
                "grouped_swiglu_gather: needs bf16, H and I multiples of 64 and 16-byte aligned rows "
                "(use jtmoe_dispatch + jtmoe_grouped_swiglu otherwise)");
  return launch_swiglu_gather(x, source_order, gate, up, down, group_sizes, offsets, T, K, H, I, E, dtype, act,
                              packed_y, as_stream(stream));
}

// Forward pass that keeps what the backward pass needs: the two rounded products
// gate_pre = round(X Wg[e]) and up_pre = round(X Wu[e]) are stored next to act and packed_y.
// With source_order the rows of x are fetched through the permutation (packed row j is token
// source_order[j] / K); without it x is already packed and has T rows.
extern "C" int jtmoe_grouped_swiglu_train(const void* x, const int32_t* source_order, const void* gate, const void* up,
                                          const void* down, const int32_t* group_sizes, const int32_t* offsets,
                                          int64_t T, int64_t K, int64_t H, int64_t I, int64_t E, int dtype,
                                          void* gate_pre, void* up_pre, void* act, void* packed_y, void* stream) {
  clear_error();
  JT_REQUIRE(T >= 0 && K > 0 && T * K < ((int64_t)1 << 31), "grouped_swiglu_train: T=%lld K=%lld out of range",
             (long long)T, (long long)K);
  const int64_t A = source_order ? T * K : T;
  int rc = validate_gemm("grouped_swiglu_train", A, H, I, E, dtype);
  if (rc) return rc;
  if (E > JTMOE_MAX_EXPERTS)
    return fail(JTMOE_EUNSUPPORTED, "grouped_swiglu_train: E=%lld exceeds %d", (long long)E, JTMOE_MAX_EXPERTS);
  if (A == 0) return JTMOE_OK;
  JT_REQUIRE(x && gate && up && down && group_sizes && offsets && gate_pre && up_pre && act && packed_y,
             "grouped_swiglu_train: null pointer argument");
  hipStream_t s = as_stream(stream);
  if (dtype == JTMOE_BF16)
    return launch_pair<bf16_raw>(x, gate, up, down, group_sizes, offsets, A, H, I, E, act, packed_y, s, kStageGateUp,
                                 source_order, (int)K, T, gate_pre, up_pre);
  return launch_pair<float>(x, gate, up, down, group_sizes, offsets, A, H, I, E, act, packed_y, s, kStageGateUp,
                            source_order, (int)K, T, gate_pre, up_pre);
}

extern "C" int jtmoe_shared_swiglu_train(const void* x, const void* gate, const void* up, const void* down, int64_t T,
                                         int64_t H, int64_t Is, int dtype, void* gate_pre, void* up_pre, void* act,
                                         void* shared_y, void* stream) {
  clear_error();
  int rc = validate_gemm("shared_swiglu_train", T, H, Is, 1, dtype);
  if (rc) return rc;
  if (T == 0) return JTMOE_OK;
  JT_REQUIRE(x && gate && up && down && gate_pre && up_pre && act && shared_y,
             "shared_swiglu_train: null pointer argument");
  hipStream_t s = as_stream(stream);
  if (dtype == JTMOE_BF16)
    return launch_pair<bf16_raw>(x, gate, up, down, nullptr, nullptr, T, H, Is, 1, act, shared_y, s,
                                 kStageSharedGateUp, nullptr, 1, 0, gate_pre, up_pre);
  return launch_pair<float>(x, gate, up, down, nullptr, nullptr, T, H, Is, 1, act, shared_y, s, kStageSharedGateUp,
                            nullptr, 1, 0, gate_pre, up_pre);
}
