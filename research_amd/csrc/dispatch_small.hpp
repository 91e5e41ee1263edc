// The dispatch plan of a small batch, computed by ONE workgroup: a histogram of the expert ids per wave in LDS, one
// scan over experts and waves, then the stable rank of every assignment (ballots inside a wave, the wave's own next free
// rows).  Same results as the three-pass plan of dispatch.hip (local_dispatch of the reference at ep_size == 1,
// moe.py:583-602).
//
// Latency bounds it.  A wave owns a run of consecutive assignments, so that the waves meet four times in all,
// whatever the number of assignments, and the ids arrive kDispatchBatch loads at a time.  us without statistics, in rounds
// of the whole workgroup with two meetings and a load each / so; 64 experts, 6 assignments 3.3 / 3.2, 296 3.5 / 3.4, 3096
// 8.4 / 5.5, 4096 9.1 / 6.0, 8192 16.3 / 9.4 (with the counts of the waves read one after the other and the ids a second time
// 3.7, 3.8, 6.0, 6.4 and 9.7).
//
// The body is a device function so that two kernels can end in it: the stand-alone small dispatch,
// and the last workgroup of the small-batch router, which then goes on from the ids it still holds
// in LDS instead of a second launch reading them back.
#pragma once

#include "common.hpp"

namespace jtmoe {

constexpr int kSmallMaxAssignments = 8192;
constexpr int64_t kSmallLayerAssignments = 4096;  // in a layer call (dispatch.hip says why)
constexpr int kSmallMaxExperts = JTMOE_MAX_EXPERTS;
constexpr float kImportanceScale = 4294967296.0f;  // importance is summed in 32.32 fixed point: any order, same sum
// A route weight as a 32.32 fixed-point term.  Route weights are finite, non-negative and far below 2^32
// (at most route_scale); anything else (a NaN from non-finite logits, a negative or huge value handed
// to the dispatcher by a caller) would make the float -> integer conversion undefined, so NaN and
// negative values count as 0 and the rest is clamped to the largest float below 2^32.
__device__ __forceinline__ unsigned long long importance_term(float w) {
  w = fminf(fmaxf(w, 0.0f), 4294967040.0f);  // fmaxf(NaN, 0) = 0
  return (unsigned long long)(w * kImportanceScale);
}

constexpr int kDispatchBatch = 4;  // loads of a lane in flight

// LDS of the body: next[waves][E], wave_sums[waves] ints, then (kStats) imp[E] of 8 bytes
__host__ __device__ inline size_t dispatch_small_smem_bytes(int E, int threads, bool stats) {
  const int waves = threads / kWave;
  size_t n = ((size_t)E * waves + waves) * sizeof(int);
  n = (n + 7) / 8 * 8;
  if (stats) n += (size_t)E * 8;
  return n;
}

// ids: A expert ids in assignment order (global memory or LDS); ids outside [0, E) are dropped.
// kStats: also expert_counts[e] = number of assignments of e (as float) and importance[e] = the sum
// of their route weights (the two vectors of _router_stats, moe.py:802-805).
// Requires A > 0, blockDim.x == kThreads and, for the scan, E <= kThreads.  Ends without a barrier.
template <int kThreads, bool kStats, typename WT>
__device__ __forceinline__ void dispatch_small_body(const int32_t* ids, const WT* weights, int A, int E,
                                                    int32_t* __restrict__ group_sizes, int32_t* __restrict__ offsets,
                                                    int32_t* __restrict__ source_order, int32_t* __restrict__ inverse,
                                                    float* __restrict__ expert_counts, float* __restrict__ importance,
                                                    unsigned char* smem_raw) {
  constexpr int kWaves = kThreads / kWave;
  int* const next = reinterpret_cast<int*>(smem_raw);  // [kWaves][E] assignments of the wave, then its next packed row
  int* const wave_sums = next + kWaves * E;            // [kWaves]
  unsigned long long* const imp =
      reinterpret_cast<unsigned long long*>(smem_raw + (((size_t)E * kWaves + kWaves) * sizeof(int) + 7) / 8 * 8);
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  if (kStats)
    for (int e = tid; e < E; e += kThreads) imp[e] = 0ull;
  const int run = (A + kThreads - 1) / kThreads * kWave;                // assignments of a wave
  const int waves = A <= kThreads ? (A + kWave - 1) / kWave : kWaves;  // no wave behind these has any
  for (int i = tid; i < waves * E; i += kThreads) next[i] = 0;
  __syncthreads();
  const int first = wave * run, end = min(first + run, A);
  int* const mine = next + wave * E;
  int id[kDispatchBatch];  // (a run of one batch keeps its ids for the ranks)
  for (int base = first; base < end; base += kDispatchBatch * kWave) {
    float w[kDispatchBatch];
#pragma unroll
    for (int i = 0; i < kDispatchBatch; ++i) {
      const int a = base + i * kWave + lane;
      id[i] = a < end ? ids[a] : -1;
      if (kStats) w[i] = a < end ? Elem<WT>::load(weights + a) : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < kDispatchBatch; ++i)
      if (base + i * kWave < end && id[i] >= 0 && id[i] < E) {
        atomicAdd(&mine[id[i]], 1);
        if (kStats) atomicAdd(&imp[id[i]], importance_term(w[i]));
      }
  }
  __syncthreads();
  // exclusive scan over the experts: thread e owns expert e
  // (the reads of a wave's threads without a condition, so that they are all on their way at once)
  int of_wave[kWaves] = {}, count = 0;
  if (wave * kWave < E) {
    const int mine_or_last = min(tid, E - 1);
#pragma unroll
    for (int w = 0; w < kWaves; ++w) of_wave[w] = next[min(w, waves - 1) * E + mine_or_last];
#pragma unroll
    for (int w = 0; w < kWaves; ++w) count += of_wave[w] = tid < E && w < waves ? of_wave[w] : 0;
  }
  int incl = count;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int v = __shfl_up(incl, d);
    if (lane >= d) incl += v;
  }
  if (lane == kWave - 1) wave_sums[wave] = incl;
  __syncthreads();
  int before = 0;
  for (int w = 0; w < wave; ++w) before += wave_sums[w];
  if (tid < E) {
    int row = incl + before - count;
    offsets[tid] = row;
    group_sizes[tid] = count;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      if (w < waves) next[w * E + tid] = row;
      row += of_wave[w];
    }
    if (kStats) {
      expert_counts[tid] = (float)count;
      importance[tid] = (float)((double)imp[tid] * (1.0 / 4294967296.0));
    }
  }
  __syncthreads();
  int nbits = 0;
  while ((1 << nbits) < E) ++nbits;
  for (int base = first; base < end; base += kDispatchBatch * kWave) {
    if (run > kDispatchBatch * kWave)
#pragma unroll
      for (int i = 0; i < kDispatchBatch; ++i) {
        const int a = base + i * kWave + lane;
        id[i] = a < end ? ids[a] : -1;
      }
#pragma unroll
    for (int i = 0; i < kDispatchBatch; ++i) {
      const int a = base + i * kWave + lane;
      const bool valid = id[i] >= 0 && id[i] < E;
      unsigned long long peers = __ballot(valid);  // lanes of this wave holding the same expert id
      for (int b = 0; b < nbits; ++b) {
        const bool bit = (id[i] >> b) & 1;
        const unsigned long long m = __ballot(valid && bit);
        peers &= bit ? m : ~m;
      }
      const int rank = __popcll(peers & ((1ull << lane) - 1ull));
      if (valid) {
        const int pos = mine[id[i]] + rank;
        inverse[a] = pos;
        source_order[pos] = a;
      } else if (a < end) {
        inverse[a] = -1;
      }
      if (base + (i + 1) * kWave >= end) break;
      // (the table is the wave's own, and its LDS accesses are done in order)
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (valid && rank == 0) mine[id[i]] += __popcll(peers);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  }
}

}  // namespace jtmoe
