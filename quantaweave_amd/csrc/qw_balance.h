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

// Sums w, w + 16 / NS, ... (NS of the sixteen) of expert e, sum i over the partial rows
// i, i + 16, ... in order: eight rows of each in flight.  w is uniform: one row
// address per wave and load.
template <int NS>
__device__ __forceinline__ void importance_sums(const BalanceJob& j, int w, int e, float (&s)[NS]) {
  constexpr int kRows = 8, kStep = 16 / NS;
  const int col = min(e, j.E - 1);
#pragma unroll
  for (int i = 0; i < NS; ++i) s[i] = 0.0f;
#pragma unroll 1
  for (int b0 = w; b0 < j.nb; b0 += 16 * kRows) {
    float v[NS * kRows];
#pragma unroll
    for (int k = 0; k < NS * kRows; ++k)  // rows past the end: the last one, not added
      v[k] = (j.partial + static_cast<int64_t>(min(b0 + kStep * k, j.nb - 1)) * j.E)[col];
#pragma unroll
    for (int k = 0; k < NS * kRows; ++k) s[k % NS] += b0 + kStep * k < j.nb ? v[k] : 0.0f;  // +0: sums are >= 0
  }
}

// Importance and balance by one workgroup of WAVES waves (4 or 16): sixteen sums per
// expert (a single chunk: its four quarters, straight from the probabilities)
// added in order, then the balance term over experts in ascending order by one
// thread.  Bound by the rounds of dependent loads.  64 experts at a time, the sums
// dealt over the waves: one round per 128 partial rows and 64 experts (184 experts:
// 3 at 8192 tokens; a thread per expert, its sums one after the other, took 16: whole
// layer of d 64, 71.7 -> 66.9 us, 1024 experts 201 -> 193).  With at most 16 partial
// rows a sum is one row: a thread per expert then holds all of them in one round
// (184 experts, 256 tokens: 37.8 us against 40.7).  With 4 waves it runs beside the
// combining workgroups, which pay for its registers: 49 here, 138 with 64-bit
// addresses per lane (combine 16 -> 24 us at 8192 x 2048).
// A kernel of its own is built for one form (kThreadPerExpert: more than 64 experts
// and at most 16 partial rows; kManyRows: several partial rows): its instructions
// come from memory at each launch, and those of the other forms cost it 1 us.
enum BalanceForm { kAnyForm, kThreadPerExpert, kManyRows };

template <int WAVES, BalanceForm FORM = kAnyForm>
__device__ __forceinline__ void balance_final(const BalanceJob& j, float (*red)[kWave], float* term) {
  static_assert(WAVES == 4 || WAVES == 16, "sixteen sums dealt evenly, at least four quarters");
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const float routes = static_cast<float>(static_cast<int64_t>(j.T) * j.K);
  const bool one = FORM != kManyRows && j.nb == 1;
  const int sums = one ? 4 : 16;
  auto finish = [&](float t, int e) {
    const float imp = t / static_cast<float>(j.T);
    j.importance[e] = imp;
    term[e] = imp * (static_cast<float>(j.counts[e]) / routes);
  };
  if (FORM == kThreadPerExpert || (FORM == kAnyForm && j.E > kWave && j.nb <= 16)) {
#pragma unroll 1
    for (int e = threadIdx.x; e < j.E; e += WAVES * kWave) {
      float t = 0.0f;  // 0 + the first sum is that sum: all are >= 0
      if (j.nb == 1) {
#pragma unroll 1
        for (int q = 0; q < 4; ++q) t += importance_quarter(j.probs, j.T, j.E, 0, q, e);
      } else {
        float v[16];
#pragma unroll
        for (int w = 0; w < 16; ++w) v[w] = (j.partial + static_cast<int64_t>(min(w, j.nb - 1)) * j.E)[e];
#pragma unroll
        for (int w = 0; w < 16; ++w) t += w < j.nb ? v[w] : 0.0f;
      }
      finish(t, e);
    }
    __syncthreads();
  } else {
#pragma unroll 1
    for (int e0 = 0; e0 < j.E; e0 += kWave) {
      const int e = e0 + lane;
      if (one) {
        if (wave < 4) red[wave][lane] = importance_quarter(j.probs, j.T, j.E, 0, wave, e);
      } else {
        float s[16 / WAVES];
        importance_sums<16 / WAVES>(j, wave, e, s);
#pragma unroll
        for (int i = 0; i < 16 / WAVES; ++i) red[wave + WAVES * i][lane] = s[i];
      }
      __syncthreads();
      if (wave == 0 && e < j.E) {
        float t = 0.0f;
        for (int w = 0; w < sums; ++w) t += red[w][lane];
        finish(t, e);
      }
      __syncthreads();
    }
  }
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
