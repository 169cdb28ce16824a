// Pieces shared by the matrix-core kernels that stage operands with
// global_load_lds: operand types, waits, the ring barrier, the MFMA step in the
// activation type, and the kernel view of a stacked projection.
#pragma once
#include <algorithm>
#include <cmath>

#include "qw_ffn.h"

namespace qw {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));  // 16-bit operands (bf16 or fp16 bits)
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;

// s_waitcnt immediate waiting for vmcnt <= n only (expcnt, lgkmcnt left at max).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | (((N >> 4) & 3) << 14));
}

// Barrier for an LDS ring: the slice's loads were already waited for with an
// explicit vmcnt, so no fence is needed (a workgroup fence would wait for every
// load still in flight, including the slices requested ahead).  The empty asm
// statements keep the compiler from moving LDS accesses across the barrier.
__device__ __forceinline__ void ring_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Weights of one projection for the kernels: bytes per expert and per stored
// row; scales (quantised formats) per expert, per row, and the group size.
struct MfW {
  const char* w;
  const float* scales;
  int64_t expert_bytes, row_bytes, expert_scales;
  int groups, group;
};

inline MfW mf_view(int wf, const WView& v) {
  const int64_t esize = wf == QW_I8 || wf == QW_U4 ? 1 : 2;  // QW_U4 strides are in bytes already
  MfW m;
  m.w = static_cast<const char*>(v.w);
  m.scales = v.scales;
  m.expert_bytes = v.expert_elems * esize;
  m.row_bytes = v.row_stride * esize;
  m.expert_scales = v.expert_scales;
  m.groups = static_cast<int>(v.groups);
  m.group = static_cast<int>(v.group > 0 ? v.group : 1);
  return m;
}

// One 16x16x32 MFMA step in the activation type: bf16, or fp16 bits carried
// in the same 16-byte operand registers.
template <int ACT>
__device__ __forceinline__ f32x4 mfma_step(bf16x8 a, bf16x8 b, f32x4 c) {
  if constexpr (ACT == QW_F16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                   0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Four unsigned bytes of `even` and `odd` each -> act(u * s + c), interleaved:
// columns 2b from even, 2b + 1 from odd.  The bytes are opaque, so each
// conversion is one v_cvt_f32_ubyte<n>.
template <int ACT>
__device__ __forceinline__ bf16x8 scale_bytes(uint32_t even, uint32_t odd, float s, float c) {
  asm("" : "+v"(even), "+v"(odd));
  u32x4 r;
#pragma unroll
  for (int b = 0; b < 4; ++b)
    r[b] = pack_half2<ACT>(__builtin_fmaf(static_cast<float>((even >> (8 * b)) & 0xffu), s, c),
                           __builtin_fmaf(static_cast<float>((odd >> (8 * b)) & 0xffu), s, c));
  return __builtin_bit_cast(bf16x8, r);
}

// The same with consecutive columns in lo (0..3) and hi (4..7).
template <int ACT>
__device__ __forceinline__ bf16x8 scale_bytes_seq(uint32_t lo, uint32_t hi, float s, float c) {
  asm("" : "+v"(lo), "+v"(hi));
  u32x4 r;
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    r[b] = pack_half2<ACT>(__builtin_fmaf(static_cast<float>((lo >> (16 * b)) & 0xffu), s, c),
                           __builtin_fmaf(static_cast<float>((lo >> (16 * b + 8)) & 0xffu), s, c));
    r[2 + b] = pack_half2<ACT>(__builtin_fmaf(static_cast<float>((hi >> (16 * b)) & 0xffu), s, c),
                               __builtin_fmaf(static_cast<float>((hi >> (16 * b + 8)) & 0xffu), s, c));
  }
  return __builtin_bit_cast(bf16x8, r);
}

// The quantised projection suits the matrix-core kernels: rows of whole
// 64-column slices, groups of whole MFMA K steps, 16-byte aligned rows and base.
inline bool quant_fits(const WView& v, int wf) {
  return (wf == QW_I8 || wf == QW_U4) && v.cols % 64 == 0 && v.group > 0 && v.group % 32 == 0 &&
         v.row_stride % 16 == 0 && reinterpret_cast<uintptr_t>(v.w) % 16 == 0 &&
         reinterpret_cast<uintptr_t>(v.scales) % 4 == 0;
}

// Rows of an expert to size a row chunk for: even routing with room for
// `sigmas` standard deviations, within the bound.  A loose bound (no capacity)
// says nothing about the usual expert; one with more rows takes another chunk.
inline int64_t likely_rows(const FfnArgs& a, double sigmas) {
  const int64_t cap = a.row_cap > 0 ? a.row_cap : a.max_rows;
  return std::min(cap, a.avg_rows + static_cast<int64_t>(sigmas * std::sqrt(static_cast<double>(a.avg_rows))));
}

// Row chunks of one expert that follow each other on one XCD where the row bound is
// loose: as many as an expert of the average size has, at least two, so that the
// usual expert's weights are fetched by one L2, while a popular expert's chunks go
// round the XCDs in such runs instead of queueing on one (d 2048, f 1024, 64 experts,
// no capacity, popularity r^-1.2: 8192 rows bf16 353 -> 241 us, int8 391 -> 215; one
// expert with all of 1024 rows 146 -> 47; even routing as before).
inline int loose_run(int64_t rows, int64_t experts, int64_t chunk) {
  return static_cast<int>(std::max<int64_t>(2, ceil_div(ceil_div(rows, experts), chunk)));
}

// Chunks of that order one XCD can own: its share of the runs that hold all rows, one of
// them partial per expert.
inline int64_t loose_chunks(int64_t rows, int64_t experts, int64_t chunk, int run) {
  return run * ceil_div(ceil_div(rows, run * chunk) + experts, kXcds);
}

// The at-th chunk of XCD xcd: runs of `run` chunks of `gran` rows, expert after expert,
// dealt to the XCDs in turn, without the empty places of runs that are not full.
// Returns the expert (-1 past the last) and its chunk.  One wave works it out: a
// scan of the experts' runs gives their XCDs, one of their chunks here the place.
__device__ __forceinline__ int find_run_chunk(const int32_t* __restrict__ offsets, int E, int rows, int gran, int run,
                                              int xcd, int at, int* chunk) {
  const int lane = threadIdx.x % kWave;
  int runs_before = 0, chunks_before = 0;
  for (int e0 = 0; e0 < E; e0 += kWave) {
    const int e = e0 + lane;
    int c = 0;
    if (e < E) {
      const int lo = min(max(offsets[e], 0), rows), hi = min(offsets[e + 1], rows);
      c = hi > lo ? (hi - lo + gran - 1) / gran : 0;
    }
    const int k = (c + run - 1) / run;
    int incl = k;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const int v = __shfl_up(incl, o, kWave);
      if (lane >= o) incl += v;
    }
    const int first = (xcd - (runs_before + incl - k)) & (kXcds - 1);  // the expert's first run on this XCD
    const int n = first < k ? (k - first + kXcds - 1) / kXcds : 0;     // its runs here
    const bool last = n > 0 && first + kXcds * (n - 1) == k - 1;       // among them its last, perhaps partial one
    const int here = n * run - (last ? k * run - c : 0);
    runs_before += __shfl(incl, kWave - 1, kWave);
    incl = here;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const int v = __shfl_up(incl, o, kWave);
      if (lane >= o) incl += v;
    }
    const unsigned long long hit = __ballot(chunks_before + incl > at);
    if (hit) {
      const int l = __ffsll(static_cast<long long>(hit)) - 1;
      const int q = at - chunks_before - __shfl(incl - here, l, kWave);
      *chunk = (__shfl(first, l, kWave) + kXcds * (q / run)) * run + q % run;
      return e0 + l;
    }
    chunks_before += __shfl(incl, kWave - 1, kWave);
  }
  return -1;
}

// Quantised experts of up to this many rows take the kernel that dequantises
// each weight once; with more, the one whose larger row chunks read fewer
// weights.  Whole layer, this one against the other: int4 (d 4096, f 1408) 342
// against 561 us at 64 rows per expert, 562 / 596 at 128, 646 / 660 at 188,
// 870 / 753 at 256; int8 (d 2048, f 1024) 151 / 213, 220 / 251, 261 / 269,
// 378 / 301 us.  fp16 activations (expert stage): int4 308 / 463 at 64 rows, 512 /
// 568 at 128, 553 / 596 at 160, int8 119 / 195, 193 / 225, 213 / 231.
constexpr int64_t kQuantRows = 192;

}  // namespace qw
