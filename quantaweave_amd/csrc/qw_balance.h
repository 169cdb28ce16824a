// The balance loss (src/quantweave_moe_model.py:152-154) in pieces that run
// beside other kernels' work: partial sums of the probabilities per 64 tokens,
// then importance and the balance term, every addition in a fixed order.  As
// kernels of their own they cost two launches (4.8 us each at 8192 x 64) for
// about 1 us of work; as extra workgroups of the plan and combine launches they
// run on compute units those leave idle.
#pragma once
#include "qw_common.h"

namespace qw {

constexpr int kImpRows = 64;  // tokens per partial sum

struct BalanceJob {
  const float* probs = nullptr;     // [T, E]
  const int32_t* counts = nullptr;  // [E] routes per expert
  const int32_t* totals = nullptr;  // kept, dropped
  float* partial = nullptr;         // [nb, E] workspace (nb > 1)
  int nb = 0, T = 0, K = 0, E = 0;  // nb = ceil(T / 64)
  float* importance = nullptr;      // [E]
  float* balance = nullptr;
  int64_t* overflow = nullptr;      // the dropped count, 64 bits
  float* zero = nullptr;            // one 0.0f (a loss that was not asked for)
};

// Sum of expert e's probabilities over this quarter's tokens (every fourth) of
// a 64-token chunk, in token order: all 16 loads in flight at once (a token
// past the end adds +0, which leaves the non-negative sum as it is).
__device__ __forceinline__ float importance_quarter(const float* __restrict__ probs, int T, int E, int chunk,
                                                    int quarter, int e) {
  const int t0 = chunk * kImpRows, t1 = min(T, t0 + kImpRows);
  float v[kImpRows / 4];
#pragma unroll
  for (int i = 0; i < kImpRows / 4; ++i) {
    const int t = t0 + quarter + 4 * i;
    v[i] = (e < E && t < t1) ? probs[static_cast<int64_t>(t) * E + e] : 0.0f;
  }
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < kImpRows / 4; ++i) s += v[i];
  return s;
}

// Units (chunk, block of 64 experts) of partial sums; a unit takes four waves.
__host__ __device__ inline int partial_units(int nb, int E) { return nb * ((E + kWave - 1) / kWave); }

// One unit by waves 0..3 of a group; red holds the group's four rows of 64.
// Every thread of the block must call it (it holds a barrier).
__device__ __forceinline__ void importance_unit(const BalanceJob& j, int unit, float (*red)[kWave]) {
  const int lane = threadIdx.x % kWave, quarter = threadIdx.x / kWave % 4;
  const int chunk = unit % j.nb, e = unit / j.nb * kWave + lane;
  red[quarter][lane] = importance_quarter(j.probs, j.T, j.E, chunk < j.nb ? chunk : 0, quarter, e);
  __syncthreads();
  if (quarter == 0 && e < j.E && unit < partial_units(j.nb, j.E))
    j.partial[static_cast<int64_t>(chunk) * j.E + e] = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
}

// Sum w of expert e: partial rows w, w + 16, ... in order, eight in flight.
__device__ __forceinline__ float importance_sum(const BalanceJob& j, int w, int e) {
  constexpr int kRowsPerLoad = 8;
  float s = 0.0f;
#pragma unroll 1
  for (int b0 = w; b0 < j.nb; b0 += 16 * kRowsPerLoad) {
    float v[kRowsPerLoad];
#pragma unroll
    for (int i = 0; i < kRowsPerLoad; ++i) {
      const int b = b0 + 16 * i;
      v[i] = (b < j.nb && e < j.E) ? j.partial[static_cast<int64_t>(b) * j.E + e] : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < kRowsPerLoad; ++i) s += v[i];  // rows in order; +0 past the end (sums are >= 0)
  }
  return s;
}

// Importance and balance by one 256-thread workgroup: sixteen sums per expert
// (a single chunk: its four quarters, straight from the probabilities) added
// in order, then the balance term over experts in ascending order by one
// thread.  Up to 64 experts the sums are dealt over the four waves, beyond
// that the blocks of 64 experts.  It runs beside the combining workgroups, so
// it keeps few loads in flight: 32 took 138 registers per thread, which every
// one of them paid for (combine 16 -> 24 us at 8192 x 2048).
__device__ __forceinline__ void balance_final(const BalanceJob& j, float (*red)[kWave], float* term) {
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const float routes = static_cast<float>(static_cast<int64_t>(j.T) * j.K);
  const int sums = j.nb == 1 ? 4 : 16;
  auto sum = [&](int w, int e) {
    return j.nb == 1 ? importance_quarter(j.probs, j.T, j.E, 0, w, e) : importance_sum(j, w, e);
  };
  auto finish = [&](float t, int e) {
    const float imp = t / static_cast<float>(j.T);
    j.importance[e] = imp;
    term[e] = imp * (static_cast<float>(j.counts[e]) / routes);
  };
  if (j.E <= kWave) {
#pragma unroll 1
    for (int w = wave; w < sums; w += 4) red[w][lane] = sum(w, lane);
    __syncthreads();
    if (wave == 0 && lane < j.E) {
      float t = 0.0f;  // 0 + the first sum is that sum: all are >= 0
      for (int w = 0; w < sums; ++w) t += red[w][lane];
      finish(t, lane);
    }
  } else {
#pragma unroll 1
    for (int e = threadIdx.x; e - lane < j.E; e += 256) {
      float t = 0.0f;
      if (j.nb > 1 && j.nb <= 16) {  // one row per sum: all of them in flight
        float v[16];
#pragma unroll
        for (int w = 0; w < 16; ++w)
          v[w] = (w < j.nb && e < j.E) ? j.partial[static_cast<int64_t>(w) * j.E + e] : 0.0f;
#pragma unroll
        for (int w = 0; w < 16; ++w) t += v[w];
      } else {
#pragma unroll 1
        for (int w = 0; w < sums; ++w) t += sum(w, e);
      }
      if (e < j.E) finish(t, e);
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    // ascending order; 16 reads in flight at a time (the terms are >= 0, so
    // the +0 past E changes nothing)
    float s = 0.0f;
#pragma unroll 1
    for (int e0 = 0; e0 < j.E; e0 += 16) {
      float v[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = e0 + i < j.E ? term[e0 + i] : 0.0f;
#pragma unroll
      for (int i = 0; i < 16; ++i) s += v[i];
    }
    *j.balance = static_cast<float>(j.E) * s;
    if (j.overflow) *j.overflow = j.totals[1];
    if (j.zero) *j.zero = 0.0f;
  }
}

}  // namespace qw
