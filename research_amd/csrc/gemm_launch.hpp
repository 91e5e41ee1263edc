// Launchers of the two grouped GEMM forms of the backward pass (grouped_gemm_bwd.hip),
// callable from the entry points in backward.hip.  Both pick the LDS-DMA bf16 kernels when
// shape and alignment allow and an element-wise staged kernel (any dtype, any shape) otherwise.
#pragma once

#include "common.hpp"

namespace jtmoe {

// The bf16 kernel of a product, as the dispatch rules choose it (jtmoe_product_kernel names them), or a family of tiles of
// which tile_shape then picks one (jtmoe_product_tiles).  "Tail": K ends inside a step, or a gate/up product that divides
// (silu_gate).
enum class ProductKernel {
  kGeneral,
  kStream16x128,  // grouped_gemm_skinny.hpp: tiles of 16 or 32 rows
  kStream16x64,
  kStream32x64,
  kRows64,        // 64-row LDS tiles, non-temporal loads of the matrix
  kRows64Tail,
  kHalf,          // where 128 x 128 tiles have a CU each; down and gradients in short steps, or two tiles to a CU
  kHalfTail,
  kHalfDeep,      // down: two 128 x 128 tiles to a CU pay; gradients: they have a CU each
  kRows256,       // beyond
  kRows256Tail,
  kRows256Short,  // gate/up whose reduction is too short for the stream kernel
  kRows256ShortTail,
};

// C[rows of group e, :] = sum over s < segs of A_s[rows of e, :] @ B_s[e]^T
//   A_s: [rows, Kdim]      B_s: [E, N, Kdim]      C: [rows, N]      group_sizes == nullptr: one group holding every row
int launch_gemm_nt(int dtype, const void* a0, const void* a1, const void* b0, const void* b1, void* c,
                   const int32_t* group_sizes, const int32_t* offsets, int64_t rows, int64_t Kdim, int64_t N,
                   int64_t E, int segs, hipStream_t stream);
// ... and the kernel it takes for bf16 operands (16-byte aligned, below 2 GiB) on `cus` compute units
ProductKernel data_gradient_kernel(int64_t rows, int64_t Kdim, int64_t N, int64_t E, bool dense, int segs, double cus);
// ... in which tiles
enum class TileShape;
TileShape data_gradient_tiles(ProductKernel k, int64_t rows, int64_t Kdim, int64_t N, int64_t E, bool dense, int segs, double cus);

// The routed product above and the shared experts' one (one dense group of s.rows rows) in one launch.  Operands as in
// launch_gemm_nt; gemm_nt_joint: the kernel, or kGeneral where launches of their own are faster or
// the operands ask for them.
struct NtProblem {
  const void *a0, *a1, *b0, *b1;
  void* c;
  int64_t rows, Kdim, N;
};
ProductKernel gemm_nt_joint(int dtype, const NtProblem& p, int64_t E, const NtProblem& s, int segs);
int launch_gemm_nt_joint(int dtype, const NtProblem& p, const int32_t* group_sizes, const int32_t* offsets, int64_t E,
                         const NtProblem& s, int segs, hipStream_t stream);
// ... by the sizes alone, for segs = 1 (dZ: reduction H, width I or Is) and 2 (dX: reduction I or Is, width H); kGeneral:
// launches of their own
ProductKernel joint_data_gradient_kernel(int64_t rows, int64_t H, int64_t I, int64_t E, int64_t T, int64_t Is, int segs,
                                         double cus);
// ... and its tiles: rows x N with a reduction of Kdim beside T x N1 with one of K1
TileShape joint_data_gradient_tiles(ProductKernel k, int64_t rows, int64_t Kdim, int64_t N, int64_t E, int64_t T, int64_t K1,
                                    int64_t N1, int segs, double cus);

// C_i[e] = P[rows of group e, :]^T @ D_i[rows of group e, :]     (i = 0, and 1 if d1 is given)
//   P: [rows, KA], D_i: [rows, N]; either may instead be [gathered_rows, .] read through row_map
//   C_i: [E, KA, N]; an empty group yields zeros
//   split_ws: scratch of gemm_tn_split_bytes(...) bytes, or nullptr.  With it, a one-group call whose
//   output has too few tiles to fill the chip is run as partial sums over runs of rows (float32, in
//   split_ws) that a second kernel adds up in a fixed order.
int launch_gemm_tn(int dtype, const void* p, const void* d0, const void* d1, void* c0, void* c1,
                   const int32_t* group_sizes, const int32_t* offsets, int64_t rows, int64_t KA, int64_t N, int64_t E,
                   const int32_t* row_map, int row_div, bool p_gather, bool d_gather, int64_t gathered_rows,
                   hipStream_t stream, void* split_ws = nullptr);
size_t gemm_tn_split_bytes(int dtype, int64_t rows, int64_t KA, int64_t N, bool dual);

// Single precision on the matrix cores (grouped_gemm_f32.hip): K and N multiples of 4, 16-byte aligned
// operands (null ones count as aligned), operands below 2 GiB.  a_rows: rows of the gathered matrix with a row
// map, else `rows`.  NN with b1: gate and up with the SwiGLU (and the two products in save0 / save1).
bool f32_gemm_supported(const void* a0, const void* a1, const void* b0, const void* b1, const void* c, int64_t a_rows,
                        int64_t Kdim, int64_t N);
int launch_f32_nn(const void* a, const void* b0, const void* b1, void* c, const int32_t* group_sizes,
                  const int32_t* offsets, int64_t rows, int64_t Kdim, int64_t N, int64_t E, const int32_t* row_map,
                  int row_div, int64_t a_rows, void* save0, void* save1, hipStream_t stream);
int launch_f32_nt(const void* a0, const void* a1, const void* b0, const void* b1, void* c, const int32_t* group_sizes,
                  const int32_t* offsets, int64_t rows, int64_t Kdim, int64_t N, int64_t E, int segs, hipStream_t stream);
int launch_f32_tn(const void* p, const void* d0, const void* d1, void* c0, void* c1, const int32_t* group_sizes,
                  const int32_t* offsets, int64_t rows, int64_t KA, int64_t N, int64_t E, void* split_ws,
                  hipStream_t stream);
size_t f32_tn_split_bytes(int64_t rows, int64_t KA, int64_t N, bool dual);

// dXp and the three weight gradients of the routed experts in one launch, where that is supported and faster
// (compute_units: of the device to answer for, 0: the current one)
struct F32Backward {
  const void *dg, *du, *hw, *xp, *dyp, *gate, *up;
  void *dxp, *d_gate, *d_up, *d_down;
};
bool f32_backward_products_supported(const F32Backward& b, int64_t rows, int64_t H, int64_t I, int64_t E,
                                     int compute_units = 0);
int launch_f32_backward_products(const F32Backward& b, const int32_t* group_sizes, const int32_t* offsets, int64_t rows,
                                 int64_t H, int64_t I, int64_t E, hipStream_t stream);

}  // namespace jtmoe
