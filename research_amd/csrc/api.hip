// Library-level pieces of libjtmoe: error state, the sequence balance loss and
// the whole-layer launcher that chains the stage launchers on one stream.
#include "common.hpp"

#include <cstdarg>
#include <cstdio>

namespace jtmoe {

namespace {
thread_local char g_error[512] = "";
}

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof(g_error), fmt, ap);
  va_end(ap);
  return code;
}

void clear_error() { g_error[0] = '\0'; }

thread_local StageTimer* g_stage_timer = nullptr;

int check_launch(const char* what) {
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return fail(JTMOE_ELAUNCH, "%s: %s", what, hipGetErrorString(err));
  return JTMOE_OK;
}

namespace {

// ---- sequence balance loss (reference moe.py:828-840) --------------------------
// loss = 1/B sum_b sum_e f[b,e] P[b,e],  f = E / (K S) * count,  P = mean over s of scores / sum_e scores.
//
// Bound by latency, not by bytes (4 MB of scores at 8 x 2048 x 64): one workgroup per sequence walked
// S / 4 dependent steps and took 406 us forward and 274 us backward there.  A sequence is therefore cut
// into chunks of tokens, enough workgroups to fill the chip, and a wave takes 64 / W tokens at a time,
// W = the lanes that E experts need (8 experts: eight tokens per step instead of one in an eighth of the
// wave).  Forward: partial sums per chunk, then one workgroup adds them in chunk order.  Backward: each
// workgroup counts its whole sequence's ids itself (they are a fraction of the scores and come from the
// L2), which needs neither scratch nor a second launch.  Every sum has a fixed order.
// Measured there: forward 406 + 5 -> 14 + 8 us, backward 274 -> 15 us.  Many short sequences (16384 of 8 tokens, 256
// experts): forward 785 -> 37 us, of which one launch adds up the sequences' shares; backward 49 -> 48.
constexpr int kBalThreads = 256;
constexpr int kBalWaves = kBalThreads / kWave;
constexpr int kBalFinalThreads = 1024;
constexpr int kBalMinTokens = 16;  // tokens of a chunk: at least a few steps of every wave

inline int bal_clamp(int64_t v, int64_t lo, int64_t hi) { return (int)(v < lo ? lo : (v > hi ? hi : v)); }
// chunks per sequence of the forward pass: one workgroup per CU, and at most 64 partial sums for the
// finishing workgroup to add up
inline int bal_max_chunks(int64_t B) { return bal_clamp((256 + B - 1) / B, 1, 64); }
// A step of a workgroup's tokens takes 0.45 us, 1024 partial sums 0.4 us of the
// finishing one: where the latter is more a sequence stays whole and its workgroup writes one number (us at 64 and
// 200 sequences of 64 tokens, 256 experts: 16 and 16 whole, 28 and 49 in chunks; 32 of 512: 67 and 33).
inline int bal_chunks(int64_t B, int64_t S, int64_t E) {
  const int chunks = bal_clamp((S + kBalMinTokens - 1) / kBalMinTokens, 1, bal_max_chunks(B));
  const int64_t tokens_per_step = kBalWaves * (E <= 8 ? 8 : E <= 16 ? 4 : E <= 32 ? 2 : 1);
  return S * 1024 <= B * E * chunks * tokens_per_step ? 1 : chunks;
}
// ... of the backward pass: two workgroups per CU (no finishing step), but no more than 8 E / K, beyond
// which counting the sequence's S K ids in every chunk would move more bytes than half of the chunk's own
// scores
inline int bal_backward_chunks(int64_t B, int64_t S, int64_t E, int64_t K) {
  const int most = bal_clamp(8 * E / K, 8, 64);
  return bal_clamp((S + kBalMinTokens - 1) / kBalMinTokens, 1, bal_clamp((512 + B - 1) / B, 1, most));
}

// Sum over the W lanes that share a token.
template <int W>
__device__ __forceinline__ float bal_row_sum(float v) {
#pragma unroll
  for (int m = W / 2; m >= 1; m >>= 1) v += __shfl_xor(v, m);
  return v;
}

// psum[chunk][b][e] = sum over the chunk's tokens of scores / max(row sum, 1e-20), pcnt = the ids' histogram.
// W lanes per token, PL experts per lane (W * PL >= E).  kWhole: the chunk is the whole sequence, and psum[b] is its
// share of the loss, sum over e of f[b,e] P[b,e]; nothing else is written.
template <int W, int PL, bool kWhole>
__global__ __launch_bounds__(kBalThreads) void balance_partial_kernel(const int32_t* __restrict__ ids,
                                                                      const float* __restrict__ scores, int B, int S,
                                                                      int E, int K, int chunk_tokens,
                                                                      float* __restrict__ psum, int* __restrict__ pcnt) {
  extern __shared__ float smem[];
  constexpr int kRows = kBalWaves * (kWave / W);             // tokens per step of the workgroup
  float* part = smem;                                        // [kRows][E]
  int* cnt = reinterpret_cast<int*>(smem + kRows * E);       // [E]
  const int chunk = blockIdx.x, b = blockIdx.y, tid = threadIdx.x;
  const int row = tid / W, e0 = tid % W;
  const int s_lo = chunk * chunk_tokens, s_hi = min(S, s_lo + chunk_tokens);
  for (int e = tid; e < E; e += kBalThreads) cnt[e] = 0;
  __syncthreads();
  const int32_t* ids_b = ids + (size_t)b * S * K;
  for (int i = s_lo * K + tid; i < s_hi * K; i += kBalThreads) {
    const int id = ids_b[i];
    if (id >= 0 && id < E) atomicAdd(&cnt[id], 1);
  }
  float acc[PL];
#pragma unroll
  for (int j = 0; j < PL; ++j) acc[j] = 0.0f;
#pragma unroll 4
  for (int s = s_lo + row; s < s_hi; s += kRows) {
    const float* p = scores + ((size_t)b * S + s) * E;
    float v[PL];
    float sum = 0.0f;
#pragma unroll
    for (int j = 0; j < PL; ++j) {
      const int e = e0 + j * W;
      v[j] = e < E ? p[e] : 0.0f;
      sum += v[j];
    }
    const float d = fmaxf(bal_row_sum<W>(sum), 1e-20f);
#pragma unroll
    for (int j = 0; j < PL; ++j) acc[j] += v[j] / d;
  }
#pragma unroll
  for (int j = 0; j < PL; ++j) {
    const int e = e0 + j * W;
    if (e < E) part[row * E + e] = acc[j];
  }
  __syncthreads();
  const float fscale = (float)E / ((float)K * (float)S);
  float local = 0.0f;
  for (int e = tid; e < E; e += kBalThreads) {
    float t = 0.0f;
    for (int r = 0; r < kRows; ++r) t += part[r * E + e];
    if constexpr (kWhole) {
      local += fscale * (float)cnt[e] * (t / (float)S);
    } else {
      psum[((size_t)chunk * B + b) * E + e] = t;
      pcnt[((size_t)chunk * B + b) * E + e] = cnt[e];
    }
  }
  if constexpr (kWhole) {
    __shared__ float red[kBalWaves];
    local = bal_row_sum<kWave>(local);
    if ((tid & (kWave - 1)) == 0) red[tid / kWave] = local;
    __syncthreads();
    if (tid == 0) psum[b] = (red[0] + red[1]) + (red[2] + red[3]);
  }
}

// loss = mean of the sequences' shares.  A thread keeps eight loads in flight and adds them in order.
__global__ __launch_bounds__(kBalFinalThreads) void balance_mean_kernel(const float* __restrict__ share, int B,
                                                                        float* __restrict__ loss) {
  __shared__ float red[kBalFinalThreads / kWave];
  const int tid = threadIdx.x;
  float local = 0.0f;
#pragma unroll 8
  for (int b = tid; b < B; b += kBalFinalThreads) local += share[b];
  local = bal_row_sum<kWave>(local);
  if ((tid & (kWave - 1)) == 0) red[tid / kWave] = local;
  __syncthreads();
  if (tid == 0) {
    float t = 0.0f;
#pragma unroll
    for (int w = 0; w < kBalFinalThreads / kWave; ++w) t += red[w];
    loss[0] = t / (float)B;
  }
}

// loss from the chunks' sums.  With fewer (sequence, expert) pairs than threads, R = 1024 / pairs threads
// share a pair (thread i: pair i % pairs, chunks i / pairs, + R, ...), so that the finishing workgroup is
// not a chain of 64 loads per pair: 25 -> 5 us at 4 x 1024 x 8.
__global__ __launch_bounds__(kBalFinalThreads) void balance_final_kernel(const float* __restrict__ psum,
                                                                         const int* __restrict__ pcnt, int chunks,
                                                                         int B, int S, int E, int K,
                                                                         float* __restrict__ loss) {
  __shared__ float s_p[kBalFinalThreads];
  __shared__ int s_c[kBalFinalThreads];
  __shared__ float red[kBalFinalThreads / kWave];
  const float fscale = (float)E / ((float)K * (float)S);
  const int64_t pairs = (int64_t)B * E;
  const int tid = threadIdx.x;
  auto sum_chunks = [&](int64_t pair, int first, int step, float& p, int& c) {
#pragma unroll 8
    for (int k = first; k < chunks; k += step) {
      p += psum[k * pairs + pair];
      c += pcnt[k * pairs + pair];
    }
  };
  float local = 0.0f;
  if (pairs <= kBalFinalThreads / 2) {
    const int n = (int)pairs, R = kBalFinalThreads / n;
    const int part = tid / n;
    float p = 0.0f;
    int c = 0;
    if (part < R) sum_chunks(tid - part * n, part, R, p, c);
    s_p[tid] = p;
    s_c[tid] = c;
    __syncthreads();
    if (tid < n) {
      for (int r = 1; r < R; ++r) {
        p += s_p[r * n + tid];
        c += s_c[r * n + tid];
      }
      local = fscale * (float)c * (p / (float)S);
    }
  } else {
    for (int64_t i = tid; i < pairs; i += kBalFinalThreads) {
      float p = 0.0f;
      int c = 0;
      sum_chunks(i, 0, 1, p, c);
      local += fscale * (float)c * (p / (float)S);
    }
  }
  local = bal_row_sum<kWave>(local);
  if ((tid & (kWave - 1)) == 0) red[tid / kWave] = local;
  __syncthreads();
  if (tid == 0) {
    float t = 0.0f;
#pragma unroll
    for (int w = 0; w < kBalFinalThreads / kWave; ++w) t += red[w];
    loss[0] = t / (float)B;
  }
}

// Gradient of the loss with respect to the scores (the counts are piecewise constant and carry none):
//   d loss / d scores[b,s,e] = g / (B S) * ( f[b,e] / D - (sum_i f[b,i] scores[b,s,i]) / D^2 ),  D = sum_e scores[b,s,e]
// (for D <= 1e-20, where the forward divides by the constant 1e-20 instead: g / (B S) * f[b,e] / 1e-20).
// g is *d_loss, or 1 when d_loss is null.
template <int W, int PL>
__global__ __launch_bounds__(kBalThreads) void balance_backward_kernel(const int32_t* __restrict__ ids,
                                                                       const float* __restrict__ scores,
                                                                       const float* __restrict__ d_loss, int B, int S,
                                                                       int E, int K, int chunk_tokens,
                                                                       float* __restrict__ d_scores) {
  extern __shared__ float smem[];
  constexpr int kRows = kBalWaves * (kWave / W);
  // [sets][E]: a histogram per wave, fewer lanes per counter; a single one where it takes longer to clear and to add
  // up than to fill (16384 sequences of 8 tokens, 256 experts: 52 -> 47 us)
  int* cnt = reinterpret_cast<int*>(smem);
  const int b = blockIdx.y, tid = threadIdx.x, wave = tid / kWave;
  const int row = tid / W, e0 = tid % W;
  const int s_lo = blockIdx.x * chunk_tokens, s_hi = min(S, s_lo + chunk_tokens);
  const int n = S * K, sets = n >= 4 * E ? kBalWaves : 1;
  for (int e = tid; e < sets * E; e += kBalThreads) cnt[e] = 0;
  __syncthreads();
  const int32_t* ids_b = ids + (size_t)b * S * K;
  int* const mine = cnt + (sets > 1 ? wave * E : 0);
  auto count = [&](int id) {
    if (id >= 0 && id < E) atomicAdd(&mine[id], 1);
  };
  int done = 0;
  if (aligned16(ids_b)) {  // four ids per load: the loop is a chain of load latencies
    const int4* ids4 = reinterpret_cast<const int4*>(ids_b);
#pragma unroll 8
    for (int i = tid; i < n / 4; i += kBalThreads) {
      const int4 v = ids4[i];
      count(v.x);
      count(v.y);
      count(v.z);
      count(v.w);
    }
    done = n / 4 * 4;
  }
  for (int i = done + tid; i < n; i += kBalThreads) count(ids_b[i]);
  __syncthreads();
  const float fscale = (float)E / ((float)K * (float)S);
  const float g = (d_loss ? d_loss[0] : 1.0f) / ((float)B * (float)S);
  float f[PL];
#pragma unroll
  for (int j = 0; j < PL; ++j) {
    const int e = e0 + j * W;
    int c = 0;
    if (e < E) {
      c = cnt[e];
      if (sets > 1)
#pragma unroll
        for (int w = 1; w < kBalWaves; ++w) c += cnt[w * E + e];
    }
    f[j] = fscale * (float)c;
  }
#pragma unroll 4
  for (int s = s_lo + row; s < s_hi; s += kRows) {
    const size_t at = ((size_t)b * S + s) * E;
    float v[PL];
    float sum = 0.0f, dot = 0.0f;
#pragma unroll
    for (int j = 0; j < PL; ++j) {
      const int e = e0 + j * W;
      v[j] = e < E ? scores[at + e] : 0.0f;
      sum += v[j];
      dot += f[j] * v[j];
    }
    sum = bal_row_sum<W>(sum);
    dot = bal_row_sum<W>(dot);
    const bool clamped = sum <= 1e-20f;
    const float d = clamped ? 1e-20f : sum;
    const float second = clamped ? 0.0f : dot / (d * d);
#pragma unroll
    for (int j = 0; j < PL; ++j) {
      const int e = e0 + j * W;
      if (e < E) d_scores[at + e] = g * (f[j] / d - second);
    }
  }
}

// lanes per token and experts per lane for E experts
#define JT_BALANCE_WIDTHS(LAUNCH) \
  if (E <= 8)                     \
    LAUNCH(8, 1);                 \
  else if (E <= 16)               \
    LAUNCH(16, 1);                \
  else if (E <= 32)               \
    LAUNCH(32, 1);                \
  else if (E <= 64)               \
    LAUNCH(64, 1);                \
  else if (E <= 128)              \
    LAUNCH(64, 2);                \
  else                            \
    LAUNCH(64, JTMOE_MAX_EXPERTS / 64)

// ---- scalar router statistics (reference moe.py:806-813) -----------------------
// out = {total, load_min, load_max, load_mean, max_vio, load_entropy}
__global__ __launch_bounds__(256) void router_stats_kernel(const float* __restrict__ counts, int E,
                                                           float* __restrict__ out) {
  __shared__ float s_sum[256], s_min[256], s_max[256];
  const int tid = threadIdx.x;
  float sum = 0.0f, mn = 3.402823466e38f, mx = -3.402823466e38f;
  for (int e = tid; e < E; e += 256) {
    const float c = counts[e];
    sum += c;
    mn = fminf(mn, c);
    mx = fmaxf(mx, c);
  }
  s_sum[tid] = sum;
  s_min[tid] = mn;
  s_max[tid] = mx;
  __syncthreads();
  for (int d = 128; d >= 1; d >>= 1) {
    if (tid < d) {
      s_sum[tid] += s_sum[tid + d];
      s_min[tid] = fminf(s_min[tid], s_min[tid + d]);
      s_max[tid] = fmaxf(s_max[tid], s_max[tid + d]);
    }
    __syncthreads();
  }
  const float total = s_sum[0];
  const float lmin = s_min[0], lmax = s_max[0];
  __syncthreads();
  float ent = 0.0f;
  const float denom = fmaxf(total, 1e-6f);
  for (int e = tid; e < E; e += 256) {
    const float p = counts[e] / denom;
    if (p > 0.0f) ent += p * logf(p);
  }
  s_sum[tid] = ent;
  __syncthreads();
  for (int d = 128; d >= 1; d >>= 1) {
    if (tid < d) s_sum[tid] += s_sum[tid + d];
    __syncthreads();
  }
  if (tid == 0) {
    const float mean = total / (float)E;
    out[0] = total;
    out[1] = lmin;
    out[2] = lmax;
    out[3] = mean;
    out[4] = (lmax - mean) / fmaxf(mean, 1e-6f);
    out[5] = -s_sum[0];
  }
}

// ---- SMEBU balancing update (reference steps/moe_balance.py:123-161, 174-184) ----------------
// One workgroup of 16 waves; a wave owns a layer at a time and reduces over its experts with
// shuffles (no barriers inside a layer).  Per layer: mean = sum(counts) / E;
// violation = (mean - counts) / max(mean, 1e-6); delta = load_lr * tanh(clamp * violation), centred on
// its mean; momentum' = f * momentum + (1 - f) * delta; bias' = bias + momentum'.
// metrics = {max over layers of max_vio, min of load_min, max of load_max, mean of the load entropy,
//            sqrt(sum bias'^2), sqrt(sum momentum'^2)}.  Every sum has a fixed order: a lane adds its
// experts in ascending order, the wave combines lanes in a butterfly, thread 0 adds layers in order.
constexpr int kSmebuWaves = 16;

__device__ __forceinline__ float wave_sum_f32(float v) {
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d);
  return v;
}

__global__ __launch_bounds__(kSmebuWaves * 64) void smebu_update_kernel(
    const float* __restrict__ counts, float* __restrict__ momentum, float* __restrict__ bias, int L, int E,
    float load_lr, float factor, float clamp, float* __restrict__ metrics) {
  __shared__ float s_vio[kSmebuWaves], s_min[kSmebuWaves], s_max[kSmebuWaves], s_ent[kSmebuWaves],
      s_bsq[kSmebuWaves], s_msq[kSmebuWaves];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  float all_vio = -3.402823466e38f, all_min = 3.402823466e38f, all_max = -3.402823466e38f;
  float entropy_sum = 0.0f, bias_sq = 0.0f, momentum_sq = 0.0f;  // kept by thread 0
  for (int l0 = 0; l0 < L; l0 += kSmebuWaves) {
    const int l = l0 + wave;
    if (l < L) {
      const float* c = counts + (size_t)l * E;
      float* m = momentum + (size_t)l * E;
      float* b = bias + (size_t)l * E;
      float sum = 0.0f, mn = 3.402823466e38f, mx = -3.402823466e38f;
      for (int e = lane; e < E; e += 64) {
        const float v = c[e];
        sum += v;
        mn = fminf(mn, v);
        mx = fmaxf(mx, v);
      }
      const float total = wave_sum_f32(sum);
#pragma unroll
      for (int d = 32; d > 0; d >>= 1) {
        mn = fminf(mn, __shfl_xor(mn, d));
        mx = fmaxf(mx, __shfl_xor(mx, d));
      }
      const float mean = total / (float)E;
      const float denom = fmaxf(mean, 1e-6f);
      float dsum = 0.0f;
      for (int e = lane; e < E; e += 64) dsum += load_lr * tanhf(clamp * ((mean - c[e]) / denom));
      const float dmean = wave_sum_f32(dsum) / (float)E;
      float ent = 0.0f, bsq = 0.0f, msq = 0.0f;
      const float pden = fmaxf(total, 1e-6f);
      for (int e = lane; e < E; e += 64) {
        const float delta = load_lr * tanhf(clamp * ((mean - c[e]) / denom)) - dmean;
        const float next_m = factor * m[e] + (1.0f - factor) * delta;
        const float next_b = b[e] + next_m;
        m[e] = next_m;
        b[e] = next_b;
        msq += next_m * next_m;
        bsq += next_b * next_b;
        const float p = c[e] / pden;
        if (p > 0.0f) ent += p * logf(p);
      }
      ent = wave_sum_f32(ent);
      bsq = wave_sum_f32(bsq);
      msq = wave_sum_f32(msq);
      if (lane == 0) {
        s_vio[wave] = (mx - mean) / denom;
        s_min[wave] = mn;
        s_max[wave] = mx;
        s_ent[wave] = -ent;
        s_bsq[wave] = bsq;
        s_msq[wave] = msq;
      }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      const int n = min(kSmebuWaves, L - l0);
      for (int w = 0; w < n; ++w) {
        all_vio = fmaxf(all_vio, s_vio[w]);
        all_min = fminf(all_min, s_min[w]);
        all_max = fmaxf(all_max, s_max[w]);
        entropy_sum += s_ent[w];
        bias_sq += s_bsq[w];
        momentum_sq += s_msq[w];
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    metrics[0] = all_vio;
    metrics[1] = all_min;
    metrics[2] = all_max;
    metrics[3] = entropy_sum / (float)L;
    metrics[4] = sqrtf(bias_sq);
    metrics[5] = sqrtf(momentum_sq);
  }
}

struct Carve {
  unsigned char* base;
  size_t used;
  void* take(size_t bytes) {
    void* p = base ? base + used : nullptr;
    used += align_up(bytes, 256);
    return p;
  }
};

struct LayerWorkspace {
  void* router;
  size_t router_bytes;
  void* dispatch;
  size_t dispatch_bytes;
  void* packed_x;
  void* act;
  size_t act_bytes;
  void* packed_y;
  void* shared_act;
  void* shared_y;
  size_t total;
};

LayerWorkspace carve_layer(void* base, int64_t T, int64_t H, int64_t E, int64_t K, int64_t I, int64_t Is, int dtype) {
  const size_t b = dtype_bytes(dtype);
  const size_t A = (size_t)T * (size_t)K;
  Carve c{static_cast<unsigned char*>(base), 0};
  LayerWorkspace w;
  w.router_bytes = jtmoe_router_workspace_bytes(E);
  w.router = c.take(w.router_bytes);
  w.dispatch_bytes = dispatch_layer_workspace_bytes((int64_t)A, E);
  w.dispatch = c.take(w.dispatch_bytes);
  // Room for a permuted copy of x (a third of the workspace at 64 experts x top-8 x 2048) for every shape that the
  // gathering entry point refuses, as the size of the workspace has always been; the layer itself fetches the rows
  // through the permutation up to 1 GiB of x and writes the copy only beyond.
  w.packed_x = jtmoe_grouped_swiglu_gather_supported(T, H, I, dtype) ? nullptr : c.take(A * (size_t)H * b);
  // (the decode path keeps the activations of all tokens through every expert)
  const size_t act_rows = decode_dense_supported(T, H, E, K, I, dtype) ? (size_t)E * (size_t)T : A;
  w.act_bytes = (act_rows > A ? act_rows : A) * (size_t)I * b;
  w.act = c.take(w.act_bytes);
  w.packed_y = c.take(A * (size_t)H * b);
  w.shared_act = Is > 0 ? c.take((size_t)T * (size_t)Is * b) : nullptr;
  w.shared_y = Is > 0 ? c.take((size_t)T * (size_t)H * b) : nullptr;
  w.total = c.used;
  return w;
}

}  // namespace
}  // namespace jtmoe

using namespace jtmoe;

extern "C" int jtmoe_version(void) { return JTMOE_VERSION; }

extern "C" const char* jtmoe_last_error(void) { return g_error; }

extern "C" size_t jtmoe_balance_workspace_bytes(int64_t B, int64_t E) {
  if (B <= 0) return 0;
  if (bal_max_chunks(B) == 1) return align_up((size_t)B * sizeof(float), 256);
  return align_up((size_t)bal_max_chunks(B) * B * (E > 0 ? E : 1) * (sizeof(float) + sizeof(int)), 256);
}

extern "C" int jtmoe_sequence_balance_loss(const int32_t* expert_ids, const float* scores, int64_t B, int64_t S,
                                           int64_t E, int64_t K, float* loss, void* workspace,
                                           size_t workspace_bytes, void* stream) {
  clear_error();
  JT_REQUIRE(B > 0 && S > 0 && E > 0 && K > 0, "sequence_balance_loss: B=%lld S=%lld E=%lld K=%lld out of range",
             (long long)B, (long long)S, (long long)E, (long long)K);
  if (E > JTMOE_MAX_EXPERTS) return fail(JTMOE_EUNSUPPORTED, "sequence_balance_loss: E=%lld exceeds %d", (long long)E, JTMOE_MAX_EXPERTS);
  JT_REQUIRE(B * S * E < ((int64_t)1 << 40) && S * K < ((int64_t)1 << 31) && B < ((int64_t)1 << 24),
             "sequence_balance_loss: sizes out of range");
  JT_REQUIRE(expert_ids && scores && loss && workspace, "sequence_balance_loss: null pointer argument");
  if (workspace_bytes < jtmoe_balance_workspace_bytes(B, E))
    return fail(JTMOE_EWORKSPACE, "sequence_balance_loss: workspace %zu < %zu bytes", workspace_bytes,
                jtmoe_balance_workspace_bytes(B, E));
  hipStream_t s = as_stream(stream);
  const int chunks = bal_chunks(B, S, E);
  const int chunk_tokens = (int)((S + chunks - 1) / chunks);
  float* psum = static_cast<float*>(workspace);
  int* pcnt = reinterpret_cast<int*>(psum + (size_t)chunks * B * E);  // (without a use where a chunk is a sequence)
#define JT_LAUNCH_CHUNKS(W, PL, WHOLE)                                                                              \
  for (int64_t b0 = 0; b0 < B; b0 += 65535)                                                                         \
  balance_partial_kernel<W, PL, WHOLE><<<dim3(chunks, (unsigned)(B - b0 < 65535 ? B - b0 : 65535)), kBalThreads,    \
                                         (size_t)(kBalThreads / W + 1) * E * sizeof(float), s>>>(                   \
      expert_ids + b0 * S * K, scores + b0 * S * E, (int)B, (int)S, (int)E, (int)K, chunk_tokens,                   \
      psum + (WHOLE ? b0 : b0 * E), pcnt + (WHOLE ? 0 : b0 * E))
#define JT_LAUNCH_WHOLE(W, PL) JT_LAUNCH_CHUNKS(W, PL, true)
#define JT_LAUNCH_PARTS(W, PL) JT_LAUNCH_CHUNKS(W, PL, false)
  if (chunks == 1) {
    JT_BALANCE_WIDTHS(JT_LAUNCH_WHOLE);
    balance_mean_kernel<<<1, kBalFinalThreads, 0, s>>>(psum, (int)B, loss);
  } else {
    JT_BALANCE_WIDTHS(JT_LAUNCH_PARTS);
    balance_final_kernel<<<1, kBalFinalThreads, 0, s>>>(psum, pcnt, chunks, (int)B, (int)S, (int)E, (int)K, loss);
  }
#undef JT_LAUNCH_PARTS
#undef JT_LAUNCH_WHOLE
#undef JT_LAUNCH_CHUNKS
  return check_launch("sequence_balance_loss");
}

extern "C" int jtmoe_sequence_balance_loss_backward(const int32_t* expert_ids, const float* scores,
                                                    const float* d_loss, int64_t B, int64_t S, int64_t E, int64_t K,
                                                    float* d_scores, void* stream) {
  clear_error();
  JT_REQUIRE(B > 0 && S > 0 && E > 0 && K > 0,
             "sequence_balance_loss_backward: B=%lld S=%lld E=%lld K=%lld out of range", (long long)B, (long long)S,
             (long long)E, (long long)K);
  if (E > JTMOE_MAX_EXPERTS)
    return fail(JTMOE_EUNSUPPORTED, "sequence_balance_loss_backward: E=%lld exceeds %d", (long long)E, JTMOE_MAX_EXPERTS);
  JT_REQUIRE(B * S * E < ((int64_t)1 << 40) && S * K < ((int64_t)1 << 31) && B < ((int64_t)1 << 24),
             "sequence_balance_loss_backward: sizes out of range");
  JT_REQUIRE(expert_ids && scores && d_scores, "sequence_balance_loss_backward: null pointer argument");
  const int chunks = bal_backward_chunks(B, S, E, K);
  const int chunk_tokens = (int)((S + chunks - 1) / chunks);
#define JT_LAUNCH(W, PL)                                                                                     \
  for (int64_t b0 = 0; b0 < B; b0 += 65535)                                                                  \
  balance_backward_kernel<W, PL><<<dim3(chunks, (unsigned)(B - b0 < 65535 ? B - b0 : 65535)), kBalThreads,   \
                                   (size_t)kBalWaves * E * sizeof(int), as_stream(stream)>>>(                \
      expert_ids + b0 * S * K, scores + b0 * S * E, d_loss, (int)B, (int)S, (int)E, (int)K, chunk_tokens,    \
      d_scores + b0 * S * E)
  JT_BALANCE_WIDTHS(JT_LAUNCH);
#undef JT_LAUNCH
  return check_launch("sequence_balance_loss_backward");
}

extern "C" int jtmoe_router_stats(const float* expert_counts, int64_t E, float* stats6, void* stream) {
  clear_error();
  JT_REQUIRE(E > 0 && E < ((int64_t)1 << 24), "router_stats: E=%lld out of range", (long long)E);
  JT_REQUIRE(expert_counts && stats6, "router_stats: null pointer argument");
  router_stats_kernel<<<1, 256, 0, as_stream(stream)>>>(expert_counts, (int)E, stats6);
  return check_launch("router_stats");
}

extern "C" int jtmoe_smebu_update(const float* router_counts, float* momentum, float* expert_bias, int64_t L,
                                  int64_t E, float load_lr, float momentum_factor, float clamp, float* metrics6,
                                  void* stream) {
  clear_error();
  JT_REQUIRE(L > 0 && L < ((int64_t)1 << 20) && E > 0 && E < ((int64_t)1 << 24), "smebu_update: L=%lld E=%lld out of range",
             (long long)L, (long long)E);
  JT_REQUIRE(load_lr > 0.0f && momentum_factor > 0.0f && clamp > 0.0f,
             "smebu_update: load_lr, momentum and clamp must be positive");
  JT_REQUIRE(router_counts && momentum && expert_bias && metrics6, "smebu_update: null pointer argument");
  smebu_update_kernel<<<1, kSmebuWaves * 64, 0, as_stream(stream)>>>(router_counts, momentum, expert_bias, (int)L, (int)E, load_lr,
                                                       momentum_factor, clamp, metrics6);
  return check_launch("smebu_update");
}

extern "C" int jtmoe_moe_forward_takes_decode_path(int64_t T, int64_t H, int64_t E, int64_t K, int64_t I, int dtype) {
  if (T < 0 || H <= 0 || E <= 0 || K <= 0 || I <= 0 || !dtype_ok(dtype)) return 0;
  return decode_dense_supported(T, H, E, K, I, dtype) ? 1 : 0;
}

extern "C" size_t jtmoe_workspace_bytes(int64_t T, int64_t H, int64_t E, int64_t K, int64_t I, int64_t Is,
                                        int dtype) {
  if (T < 0 || H <= 0 || E <= 0 || K <= 0 || I <= 0 || Is < 0 || !dtype_ok(dtype)) return 0;
  return carve_layer(nullptr, T, H, E, K, I, Is, dtype).total;
}

// gate_pre .. shared_up_pre: where the training forward keeps the four rounded products that the
// backward pass reads; all null for the plain forward
static int moe_forward_impl(const void* x, const void* w_router, const float* expert_bias, const void* gate,
                            const void* up, const void* down, const void* shared_gate, const void* shared_up,
                            const void* shared_down, int64_t T, int64_t H, int64_t E, int64_t K, int64_t I,
                            int64_t Is, double route_scale, int dtype, void* y, int32_t* expert_ids, void* weights,
                            float* scores, float* expert_counts, float* importance, int32_t* group_sizes,
                            int32_t* offsets, int32_t* source_order, int32_t* inverse, void* workspace,
                            size_t workspace_bytes, void* stream, void* gate_pre, void* up_pre,
                            void* shared_gate_pre, void* shared_up_pre, const void* residual = nullptr,
                            const float* post_scale = nullptr, double eps = 0.0,
                            int score_func = JTMOE_SCORE_SIGMOID) {
  clear_error();
  const bool train = gate_pre != nullptr;
  JT_REQUIRE(dtype_ok(dtype), "moe_forward: unknown dtype %d", dtype);
  JT_REQUIRE(T >= 0 && H > 0 && E > 0 && K > 0 && I > 0 && Is >= 0, "moe_forward: shape out of range");
  JT_REQUIRE((Is == 0) == (shared_gate == nullptr) && (Is == 0) == (shared_up == nullptr) &&
                 (Is == 0) == (shared_down == nullptr),
             "moe_forward: shared expert matrices and Is=%lld disagree", (long long)Is);
  JT_REQUIRE(workspace != nullptr && (reinterpret_cast<uintptr_t>(workspace) & 255u) == 0,
             "moe_forward: workspace must be non-null and 256-byte aligned");
  const LayerWorkspace w = carve_layer(workspace, T, H, E, K, I, Is, dtype);
  if (workspace_bytes < w.total)
    return fail(JTMOE_EWORKSPACE, "moe_forward: workspace %zu < %zu bytes", workspace_bytes, w.total);
  // where the GEMM can apply the permutation while it fetches its A tiles, the permuted copy of
  // x is never written: dispatch then only computes the histogram, offsets and permutation
  const bool no_copy = !train && T > 0 && jtmoe_grouped_swiglu_gather_supported(T, H, I, dtype);
  const bool gather = train || no_copy || (T > 0 && T * H * (int64_t)dtype_bytes(dtype) < ((int64_t)1 << 30));
  // the workspace of such a shape holds no permuted copy of x to fall back on
  if (no_copy &&
      ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(gate) | reinterpret_cast<uintptr_t>(up) |
        reinterpret_cast<uintptr_t>(down)) & 15u) != 0)
    return fail(JTMOE_EINVAL, "moe_forward: x and the expert matrices must be 16-byte aligned");
  // The router of a layer call leaves out what the dispatch behind it can do in passing: at large
  // batches the statistics (no zeroing and no finalising launch, no global atomics), at small ones
  // its finishing workgroup writes the dispatch plan as well.
  // Decode path (a handful of tokens): one launch runs every token through every expert's gate and up
  // matrices, which needs nothing of the routing, and a few of its workgroups are the router and write
  // the dispatch plan; the down launch then picks the routed rows.
  hipStream_t main_stream = as_stream(stream);
  const bool decode = !train && decode_dense_supported(T, H, E, K, I, dtype);
  bool stats_done = false, plan_done = false, shared_done = Is == 0;
  // (a timed call keeps the shared experts in launches of their own, so that their stages are theirs)
  const bool offer_shared = Is > 0 && g_stage_timer == nullptr;
  SharedExperts shared{shared_gate, shared_up, shared_down, Is, w.shared_act, w.shared_y, shared_gate_pre,
                       shared_up_pre, I, false, false, false};
  int rc;
  if (decode) {
    rc = launch_decode_gate_up_router(x, w_router, expert_bias, gate, up, w.act, T, H, E, K, I, route_scale,
                                      score_func, expert_ids, weights, scores, expert_counts, importance, group_sizes,
                                      offsets, source_order, inverse, w.router, main_stream,
                                      offer_shared ? &shared : nullptr);
    if (rc) return rc;
    stage_mark(kStageGateUp, main_stream);
    rc = launch_down_from_all_tokens(w.act, down, group_sizes, offsets, source_order, T, K, H, I, E, w.packed_y,
                                     main_stream, shared.gate_up_done ? &shared : nullptr);
    if (rc) return rc;
    shared_done = shared_done || shared.gate_up_done;
    stage_mark(kStageDown, main_stream);
    rc = check_launch("grouped gemm");
  } else {
    rc = router_for_layer(x, w_router, expert_bias, T, H, E, K, route_scale, dtype, expert_ids, weights, scores,
                          expert_counts, importance, group_sizes, offsets, source_order, inverse, w.router,
                          w.router_bytes, score_func, &stats_done, &plan_done, main_stream, w.act, w.act_bytes,
                          offer_shared && gather ? &shared : nullptr);
    if (rc) return rc;
    stage_mark(kStageRouter, main_stream);
    rc = dispatch_for_layer(expert_ids, weights, (T > 0 && !gather) ? x : nullptr, T, H, E, K, dtype, group_sizes,
                            offsets, source_order, inverse, w.packed_x, expert_counts, importance, w.dispatch,
                            !stats_done, plan_done, main_stream, x, offer_shared && gather ? &shared : nullptr);
  }
  if (rc) return rc;
  if (!decode) {  // (the decode path has enqueued both of its GEMM launches above)
    if (train || gather) {
      const bool take = offer_shared && T > 0;
      rc = launch_swiglu_gather(x, source_order, gate, up, down, group_sizes, offsets, T, K, H, I, E, dtype, w.act,
                                w.packed_y, main_stream, take ? &shared : nullptr, gate_pre, up_pre);
      shared_done = shared_done || take;
    }
    else
      rc = jtmoe_grouped_swiglu(w.packed_x, gate, up, down, group_sizes, offsets, T * K, H, I, E, dtype, w.act,
                                w.packed_y, stream);
    if (rc) return rc;
  }
  if (!shared_done) {
    if (train)
      rc = jtmoe_shared_swiglu_train(x, shared_gate, shared_up, shared_down, T, H, Is, dtype, shared_gate_pre,
                                     shared_up_pre, w.shared_act, w.shared_y, stream);
    else
      rc = jtmoe_shared_swiglu(x, shared_gate, shared_up, shared_down, T, H, Is, dtype, w.shared_act, w.shared_y,
                               stream);
    if (rc) return rc;
  }
  if (residual)  // the decoder block's tail fused into the combine: y = residual + rmsnorm(layer output)
    rc = jtmoe_combine_norm_residual(w.packed_y, inverse, weights, Is > 0 ? w.shared_y : nullptr, residual, post_scale,
                                     eps, T, H, K, dtype, y, stream);
  else
    rc = jtmoe_combine(w.packed_y, inverse, weights, Is > 0 ? w.shared_y : nullptr, T, H, K, dtype, y, stream);
  stage_mark(kStageCombine, as_stream(stream));
  return rc;
}

extern "C" int jtmoe_moe_forward(const void* x, const void* w_router, const float* expert_bias, const void* gate,
                                 const void* up, const void* down, const void* shared_gate, const void* shared_up,
                                 const void* shared_down, int64_t T, int64_t H, int64_t E, int64_t K, int64_t I,
                                 int64_t Is, double route_scale, int dtype, void* y, int32_t* expert_ids,
                                 void* weights, float* scores, float* expert_counts, float* importance,
                                 int32_t* group_sizes, int32_t* offsets, int32_t* source_order, int32_t* inverse,
                                 void* workspace, size_t workspace_bytes, void* stream) {
  return moe_forward_impl(x, w_router, expert_bias, gate, up, down, shared_gate, shared_up, shared_down, T, H, E, K, I,
                          Is, route_scale, dtype, y, expert_ids, weights, scores, expert_counts, importance,
                          group_sizes, offsets, source_order, inverse, workspace, workspace_bytes, stream, nullptr,
                          nullptr, nullptr, nullptr);
}

extern "C" int jtmoe_moe_forward_sf(const void* x, const void* w_router, const float* expert_bias, const void* gate,
                                    const void* up, const void* down, const void* shared_gate, const void* shared_up,
                                    const void* shared_down, int64_t T, int64_t H, int64_t E, int64_t K, int64_t I,
                                    int64_t Is, double route_scale, int score_func, int dtype, void* y,
                                    int32_t* expert_ids, void* weights, float* scores, float* expert_counts,
                                    float* importance, int32_t* group_sizes, int32_t* offsets, int32_t* source_order,
                                    int32_t* inverse, void* workspace, size_t workspace_bytes, void* stream) {
  return moe_forward_impl(x, w_router, expert_bias, gate, up, down, shared_gate, shared_up, shared_down, T, H, E, K, I,
                          Is, route_scale, dtype, y, expert_ids, weights, scores, expert_counts, importance,
                          group_sizes, offsets, source_order, inverse, workspace, workspace_bytes, stream, nullptr,
                          nullptr, nullptr, nullptr, nullptr, nullptr, 0.0, score_func);
}

extern "C" int jtmoe_moe_forward_train(const void* x, const void* w_router, const float* expert_bias,
                                       const void* gate, const void* up, const void* down, const void* shared_gate,
                                       const void* shared_up, const void* shared_down, int64_t T, int64_t H,
                                       int64_t E, int64_t K, int64_t I, int64_t Is, double route_scale, int dtype,
                                       void* y, int32_t* expert_ids, void* weights, float* scores,
                                       float* expert_counts, float* importance, int32_t* group_sizes,
                                       int32_t* offsets, int32_t* source_order, int32_t* inverse, void* gate_pre,
                                       void* up_pre, void* shared_gate_pre, void* shared_up_pre, void* workspace,
                                       size_t workspace_bytes, void* stream) {
  return jtmoe_moe_forward_train_sf(x, w_router, expert_bias, gate, up, down, shared_gate, shared_up, shared_down, T, H,
                                    E, K, I, Is, route_scale, JTMOE_SCORE_SIGMOID, dtype, y, expert_ids, weights, scores,
                                    expert_counts, importance, group_sizes, offsets, source_order, inverse, gate_pre,
                                    up_pre, shared_gate_pre, shared_up_pre, workspace, workspace_bytes, stream);
}

extern "C" int jtmoe_moe_forward_train_sf(const void* x, const void* w_router, const float* expert_bias,
                                          const void* gate, const void* up, const void* down,
                                          const void* shared_gate, const void* shared_up, const void* shared_down,
                                          int64_t T, int64_t H, int64_t E, int64_t K, int64_t I, int64_t Is,
                                          double route_scale, int score_func, int dtype, void* y, int32_t* expert_ids,
                                          void* weights, float* scores, float* expert_counts, float* importance,
                                          int32_t* group_sizes, int32_t* offsets, int32_t* source_order,
                                          int32_t* inverse, void* gate_pre, void* up_pre, void* shared_gate_pre,
                                          void* shared_up_pre, void* workspace, size_t workspace_bytes, void* stream) {
  if (T > 0 && (gate_pre == nullptr || up_pre == nullptr || (Is > 0 && (!shared_gate_pre || !shared_up_pre)))) {
    clear_error();
    return fail(JTMOE_EINVAL, "moe_forward_train: null residual buffer");
  }
  // without tokens there is nothing to keep and the plain path (which launches nothing) serves
  return moe_forward_impl(x, w_router, expert_bias, gate, up, down, shared_gate, shared_up, shared_down, T, H, E, K, I,
                          Is, route_scale, dtype, y, expert_ids, weights, scores, expert_counts, importance,
                          group_sizes, offsets, source_order, inverse, workspace, workspace_bytes, stream,
                          gate_pre, up_pre, shared_gate_pre, shared_up_pre, nullptr, nullptr, 0.0, score_func);
}

extern "C" size_t jtmoe_ffn_block_workspace_bytes(int64_t T, int64_t H, int64_t E, int64_t K, int64_t I, int64_t Is,
                                                  int dtype) {
  const size_t layer = jtmoe_workspace_bytes(T, H, E, K, I, Is, dtype);
  if (layer == 0) return 0;
  return layer + align_up((size_t)T * (size_t)H * dtype_bytes(dtype), 256);
}

extern "C" int jtmoe_ffn_block_forward(const void* x, const float* pre_scale, const float* post_scale, double eps,
                                       const void* w_router, const float* expert_bias, const void* gate,
                                       const void* up, const void* down, const void* shared_gate,
                                       const void* shared_up, const void* shared_down, int64_t T, int64_t H,
                                       int64_t E, int64_t K, int64_t I, int64_t Is, double route_scale, int dtype,
                                       void* out, int32_t* expert_ids, void* weights, float* scores,
                                       float* expert_counts, float* importance, int32_t* group_sizes,
                                       int32_t* offsets, int32_t* source_order, int32_t* inverse, void* workspace,
                                       size_t workspace_bytes, void* stream) {
  clear_error();
  JT_REQUIRE(dtype_ok(dtype), "ffn_block_forward: unknown dtype %d", dtype);
  JT_REQUIRE(T >= 0 && H > 0 && E > 0 && K > 0 && I > 0 && Is >= 0, "ffn_block_forward: shape out of range");
  JT_REQUIRE(pre_scale && post_scale, "ffn_block_forward: null norm scale");
  JT_REQUIRE(workspace != nullptr && (reinterpret_cast<uintptr_t>(workspace) & 255u) == 0,
             "ffn_block_forward: workspace must be non-null and 256-byte aligned");
  const size_t layer_bytes = jtmoe_workspace_bytes(T, H, E, K, I, Is, dtype);
  const size_t need = jtmoe_ffn_block_workspace_bytes(T, H, E, K, I, Is, dtype);
  if (workspace_bytes < need)
    return fail(JTMOE_EWORKSPACE, "ffn_block_forward: workspace %zu < %zu bytes", workspace_bytes, need);
  void* normed = static_cast<unsigned char*>(workspace) + layer_bytes;
  int rc = jtmoe_rmsnorm(x, pre_scale, T, H, eps, dtype, normed, stream);
  if (rc) return rc;
  return moe_forward_impl(normed, w_router, expert_bias, gate, up, down, shared_gate, shared_up, shared_down, T, H, E,
                          K, I, Is, route_scale, dtype, out, expert_ids, weights, scores, expert_counts, importance,
                          group_sizes, offsets, source_order, inverse, workspace, layer_bytes, stream, nullptr,
                          nullptr, nullptr, nullptr, T > 0 ? x : nullptr, post_scale, eps);
}

extern "C" int jtmoe_moe_forward_timed(const void* x, const void* w_router, const float* expert_bias,
                                       const void* gate, const void* up, const void* down, const void* shared_gate,
                                       const void* shared_up, const void* shared_down, int64_t T, int64_t H,
                                       int64_t E, int64_t K, int64_t I, int64_t Is, double route_scale, int dtype,
                                       void* y, int32_t* expert_ids, void* weights, float* scores,
                                       float* expert_counts, float* importance, int32_t* group_sizes,
                                       int32_t* offsets, int32_t* source_order, int32_t* inverse, void* workspace,
                                       size_t workspace_bytes, void* stream, float* stage_ms) {
  clear_error();
  JT_REQUIRE(stage_ms != nullptr, "moe_forward_timed: stage_ms is null");
  StageTimer timer;
  int created = 0;
  for (; created < kStageCount; ++created)
    if (hipEventCreate(&timer.ev[created]) != hipSuccess) break;
  int rc = JTMOE_OK;
  if (created != kStageCount) {
    rc = fail(JTMOE_ELAUNCH, "moe_forward_timed: hipEventCreate failed");
  } else {
    hipStream_t s = as_stream(stream);
    // every event is recorded once up front so that a skipped stage reads as zero
    for (int i = kStageCount - 1; i >= 0; --i) (void)hipEventRecord(timer.ev[i], s);
    g_stage_timer = &timer;
    rc = jtmoe_moe_forward(x, w_router, expert_bias, gate, up, down, shared_gate, shared_up, shared_down, T, H, E, K,
                           I, Is, route_scale, dtype, y, expert_ids, weights, scores, expert_counts, importance,
                           group_sizes, offsets, source_order, inverse, workspace, workspace_bytes, stream);
    g_stage_timer = nullptr;
    if (hipStreamSynchronize(s) != hipSuccess && rc == JTMOE_OK)
      rc = fail(JTMOE_ELAUNCH, "moe_forward_timed: stream synchronisation failed");
    if (rc == JTMOE_OK) {
      int last = kStageBegin;
      for (int i = 1; i < kStageCount; ++i) {
        float ms = 0.0f;
        // a stage that did not run keeps its up-front record, which precedes kStageBegin
        if (hipEventElapsedTime(&ms, timer.ev[last], timer.ev[i]) != hipSuccess || ms < 0.0f) {
          stage_ms[i - 1] = 0.0f;
          continue;
        }
        stage_ms[i - 1] = ms;
        last = i;
      }
    }
  }
  for (int i = 0; i < created; ++i) (void)hipEventDestroy(timer.ev[i]);
  return rc;
}
