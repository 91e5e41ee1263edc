// RMSNorm over the last axis, the normalisation the decoder block puts in front of the MoE
// layer (ffn_pre_norm) and behind it (ffn_post_norm): blocks.py:224-230 of the reference,
// modules built by build_rms_norm (models/components/norm.py:12-31) = flax nnx.RMSNorm with
// a float32 scale, and the reference's own forward-only kernel boundary
// (kernels/rmsnorm.py:14-21, kernels/cuda/rmsnorm/rmsnorm_ffi.cu).
//
//   var = mean(f32(x)^2)        (fp32)
//   mul = rsqrt(var + eps) * scale                      (fp32, one factor per column)
//   y   = round_dtype(f32(x) * mul)
//
// 1/sqrt is computed as a correctly rounded square root followed by a correctly rounded
// division, so that a NumPy float32 restatement agrees bit for bit given the same sum.
#include "common.hpp"

namespace jtmoe {
namespace {

__device__ __forceinline__ float wave_sum_f32(float v) {
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d);
  return v;
}

// bf16 rows of a multiple of 8 elements, at most 4096, with 16-byte alignment: a workgroup per row, a wave per 64
// vectors of it, which stay in registers.  Every wave adds up the squares of the whole row, in the order of the kernel
// below, from LDS.  Latency bounds it: one load, one exchange, one store.  Up to one round of the 8192 waves the chip
// holds; us, wave per row / workgroup per row, 2048 columns: 387 rows 7.5 / 4.3, 2048 rows 10.8 / 7.4, both in a layer
// call, 4096 rows 9.2 / 10.0, 16384 30.6 / 27.6; 8192 rows of 4096 columns 31.0 / 34.8, 16384 of 768 14.1 / 15.0.
constexpr int kMaxRowWaves = 8, kMaxWaves = 8192;
__global__ __launch_bounds__(64 * kMaxRowWaves) void rmsnorm_row_kernel(const uint4* __restrict__ x,
                                                                        const float4* __restrict__ scale, int row_vecs,
                                                                        float eps, uint4* __restrict__ y) {
#pragma clang fp contract(off)
  __shared__ uint4 row[kMaxRowWaves][64];
  const int lane = threadIdx.x, v = threadIdx.y * 64 + lane;
  const bool in = v < row_vecs;
  uint4 q = make_uint4(0, 0, 0, 0);
  float4 s0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), s1 = s0;
  if (in) {
    q = x[(size_t)blockIdx.x * row_vecs + v];
    s0 = scale[v * 2];
    s1 = scale[v * 2 + 1];
  }
  row[threadIdx.y][lane] = q;
  __syncthreads();
  float ss = 0.0f;
  for (int p = 0; p < (int)blockDim.y; ++p) {
    const uint4 r = row[p][lane];
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float lo = bf16_bits_to_f32(w[i] & 0xffffu), hi = bf16_bits_to_f32(w[i] >> 16);
      ss += lo * lo;
      ss += hi * hi;
    }
  }
  ss = wave_sum_f32(ss);
  const float inv = 1.0f / sqrtf(ss / (float)(row_vecs * 8) + eps);
  if (!in) return;
  const uint32_t w[4] = {q.x, q.y, q.z, q.w};
  const float sc[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float lo = bf16_bits_to_f32(w[i] & 0xffffu) * (inv * sc[2 * i]);
    const float hi = bf16_bits_to_f32(w[i] >> 16) * (inv * sc[2 * i + 1]);
    o[i] = f32_to_bf16_bits(lo) | (f32_to_bf16_bits(hi) << 16);
  }
  y[(size_t)blockIdx.x * row_vecs + v] = make_uint4(o[0], o[1], o[2], o[3]);
}

// One wave per row; any row length.  bf16 rows of a multiple of 8 elements with 16-byte
// alignment take the vector path (kVec).
template <typename T, bool kVec>
__global__ __launch_bounds__(256) void rmsnorm_kernel(const T* __restrict__ x, const float* __restrict__ scale,
                                                      int rows, int H, float eps, T* __restrict__ y) {
#pragma clang fp contract(off)
  const int r = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= rows) return;
  const int lane = threadIdx.x & 63;
  const T* xr = x + (size_t)r * H;
  T* yr = y + (size_t)r * H;
  float ss = 0.0f;
  if (kVec) {
    const uint4* xv = reinterpret_cast<const uint4*>(xr);
    for (int v = lane; v < H / 8; v += 64) {
      const uint4 q = xv[v];
      const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float lo = bf16_bits_to_f32(w[i] & 0xffffu), hi = bf16_bits_to_f32(w[i] >> 16);
        ss += lo * lo;
        ss += hi * hi;
      }
    }
  } else {
    for (int i = lane; i < H; i += 64) {
      const float v = Elem<T>::load(xr + i);
      ss += v * v;
    }
  }
  ss = wave_sum_f32(ss);
  const float inv = 1.0f / sqrtf(ss / (float)H + eps);
  if (kVec) {
    const uint4* xv = reinterpret_cast<const uint4*>(xr);
    uint4* yv = reinterpret_cast<uint4*>(yr);
    for (int v = lane; v < H / 8; v += 64) {
      const uint4 q = xv[v];
      const uint32_t w[4] = {q.x, q.y, q.z, q.w};
      uint32_t o[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float lo = bf16_bits_to_f32(w[i] & 0xffffu) * (inv * scale[v * 8 + 2 * i]);
        const float hi = bf16_bits_to_f32(w[i] >> 16) * (inv * scale[v * 8 + 2 * i + 1]);
        o[i] = f32_to_bf16_bits(lo) | (f32_to_bf16_bits(hi) << 16);
      }
      yv[v] = make_uint4(o[0], o[1], o[2], o[3]);
    }
  } else {
    for (int i = lane; i < H; i += 64) Elem<T>::store(yr + i, Elem<T>::load(xr + i) * (inv * scale[i]));
  }
}

}  // namespace
}  // namespace jtmoe

using namespace jtmoe;

extern "C" int jtmoe_rmsnorm(const void* x, const float* scale, int64_t T, int64_t H, double eps, int dtype, void* y,
                             void* stream) {
  clear_error();
  JT_REQUIRE(dtype_ok(dtype), "rmsnorm: unknown dtype %d", dtype);
  JT_REQUIRE(T >= 0 && H > 0 && H < ((int64_t)1 << 24) && T < ((int64_t)1 << 31), "rmsnorm: T=%lld H=%lld out of range",
             (long long)T, (long long)H);
  JT_REQUIRE(eps >= 0.0, "rmsnorm: eps must not be negative");
  if (T == 0) return JTMOE_OK;
  JT_REQUIRE(x && scale && y, "rmsnorm: null pointer argument");
  hipStream_t s = as_stream(stream);
  const unsigned grid = (unsigned)((T + 3) / 4);
  if (dtype == JTMOE_BF16) {
    const int64_t waves = (H + 511) / 512;
    if (H % 8 == 0 && waves > 1 && waves <= kMaxRowWaves && T * waves <= kMaxWaves && aligned16(x) && aligned16(y) && aligned16(scale))
      rmsnorm_row_kernel<<<(unsigned)T, dim3(64, (unsigned)waves), 0, s>>>(
          static_cast<const uint4*>(x), reinterpret_cast<const float4*>(scale), (int)(H / 8), (float)eps,
          static_cast<uint4*>(y));
    else if (H % 8 == 0 && aligned16(x) && aligned16(y))
      rmsnorm_kernel<bf16_raw, true><<<grid, 256, 0, s>>>(static_cast<const bf16_raw*>(x), scale, (int)T, (int)H,
                                                          (float)eps, static_cast<bf16_raw*>(y));
    else
      rmsnorm_kernel<bf16_raw, false><<<grid, 256, 0, s>>>(static_cast<const bf16_raw*>(x), scale, (int)T, (int)H,
                                                           (float)eps, static_cast<bf16_raw*>(y));
  } else {
    rmsnorm_kernel<float, false><<<grid, 256, 0, s>>>(static_cast<const float*>(x), scale, (int)T, (int)H, (float)eps,
                                                      static_cast<float*>(y));
  }
  return check_launch("rmsnorm");
}
