// Permute, combine, balance loss, weight quantisation and the plain grouped
// matmul.
#include "qw_balance.h"
#include "qw_ffn.h"
#include "qw_weights.h"

namespace qw {

// ---------------------------------------------------------------------------
// Permute: out[s] = x[slot_token[s]] (src/quantweave_moe_model.py:195).
// One block per row; 16-byte vectors when the row is 16-byte aligned.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void permute_kernel(const char* __restrict__ x, int64_t row_bytes,
                                                      const int32_t* __restrict__ slot_token,
                                                      const int32_t* __restrict__ totals, int max_rows,
                                                      char* __restrict__ out) {
  const int s = blockIdx.x;
  const int n = min(*totals, max_rows);
  if (s >= n) return;
  const char* src = x + static_cast<int64_t>(slot_token[s]) * row_bytes;
  char* dst = out + static_cast<int64_t>(s) * row_bytes;
  if ((row_bytes & 15) == 0) {
    const int64_t nv = row_bytes / 16;
    for (int64_t i = threadIdx.x; i < nv; i += blockDim.x)
      reinterpret_cast<uint4*>(dst)[i] = reinterpret_cast<const uint4*>(src)[i];
  } else {
    for (int64_t i = threadIdx.x; i < row_bytes; i += blockDim.x) dst[i] = src[i];
  }
}

int permute(const void* x, int dtype, int64_t D, const int32_t* slot_token, const int32_t* totals, int64_t max_rows,
            void* out, hipStream_t stream) {
  QW_REQUIRE(dtype == QW_F32 || dtype == QW_BF16 || dtype == QW_F16, "permute dtype must be f32, bf16 or f16");
  QW_REQUIRE(D >= 1 && max_rows >= 0 && max_rows <= INT32_MAX, "bad permute sizes");
  if (max_rows == 0) return QW_OK;
  QW_REQUIRE(x && slot_token && totals && out, "permute pointers are required");
  const int64_t row_bytes = D * (dtype == QW_F32 ? 4 : 2);
  permute_kernel<<<static_cast<unsigned>(max_rows), 256, 0, stream>>>(
      static_cast<const char*>(x), row_bytes, slot_token, totals, static_cast<int>(max_rows), static_cast<char*>(out));
  QW_LAUNCH_CHECK("permute_kernel");
  return QW_OK;
}

// The same with the rows rounded to another activation type on the way, eight
// elements per thread and step (the cast of the whole input and its extra pass
// over memory fall away: 20 us of 8192 x 2048 fp32 rows).
template <int IN, int OUT, int VEC>
__global__ __launch_bounds__(256) void permute_cast_kernel(const void* __restrict__ x, int D,
                                                           const int32_t* __restrict__ slot_token,
                                                           const int32_t* __restrict__ totals, int max_rows,
                                                           void* __restrict__ out) {
  const int s = blockIdx.x;
  if (s >= min(*totals, max_rows)) return;
  const int64_t src = static_cast<int64_t>(slot_token[s]) * D, dst = static_cast<int64_t>(s) * D;
  for (int c = threadIdx.x * VEC; c < D; c += 256 * VEC) {
    float v[VEC];
    load_vec<IN, VEC>(x, src + c, v);
    store_vec<OUT, VEC>(out, dst + c, v);
  }
}

int permute_cast(const void* x, int dtype, int64_t D, const int32_t* slot_token, const int32_t* totals,
                 int64_t max_rows, void* out, int out_dtype, hipStream_t stream) {
  if (dtype == out_dtype) return permute(x, dtype, D, slot_token, totals, max_rows, out, stream);
  QW_REQUIRE(D >= 1 && D <= INT32_MAX / 2 && max_rows >= 0 && max_rows <= INT32_MAX, "bad permute sizes");
  if (max_rows == 0) return QW_OK;
  QW_REQUIRE(x && slot_token && totals && out, "permute pointers are required");
  const bool vec = D % 8 == 0 && (reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out)) % 16 == 0;
  const unsigned g = static_cast<unsigned>(max_rows);
  const int d = static_cast<int>(D), m = static_cast<int>(max_rows);
#define QW_PC(I, O)                                                                                       \
  if (dtype == I && out_dtype == O) {                                                                     \
    if (vec) permute_cast_kernel<I, O, 8><<<g, 256, 0, stream>>>(x, d, slot_token, totals, m, out);       \
    else permute_cast_kernel<I, O, 1><<<g, 256, 0, stream>>>(x, d, slot_token, totals, m, out);           \
    QW_LAUNCH_CHECK("permute_cast_kernel");                                                               \
    return QW_OK;                                                                                         \
  }
  QW_PC(QW_F32, QW_BF16)
  QW_PC(QW_F32, QW_F16)
  QW_PC(QW_BF16, QW_F32)
  QW_PC(QW_BF16, QW_F16)
  QW_PC(QW_F16, QW_F32)
  QW_PC(QW_F16, QW_BF16)
#undef QW_PC
  return set_error(QW_ERR_INVALID, "permute dtypes must be f32, bf16 or f16 (got %d, %d)", dtype, out_dtype);
}

// ---------------------------------------------------------------------------
// Combine: out[t] = the kept routes of t added in ascending expert order (the
// plan order of `tokens`) in fp32, starting from zero, and rounded to the
// output dtype once — the arithmetic of torch's
// `zeros_like(flat).index_add_(0, tokens, y)` (src/quantweave_moe_model.py:192,
// :201, :211), which for a bf16 output accumulates in fp32 in index order and
// rounds at the end.  One block per token.
// WEIGHTED: each row enters as (y * w).to(out dtype), w the route's router
// weight — `expert_output * weights[:, None]` (:201) with unweighted rows.
// The same kernel with weights off and OUT = fp32 is the backward of the row
// gather flat[tokens] (:192): index_add of the rows' gradients.
// ---------------------------------------------------------------------------
// STATIC: the accumulation of the capacity-free static dispatch
// (TopKMoE._static_output, src/quantweave_moe_model.py:235-245): the route
// weight is cast to the output dtype before the product
// (`dense_weights[:, e].to(flat_hidden.dtype)`), and `output = output + term`
// rounds after every add, expert by expert in ascending order (the experts
// with weight zero add exact zeros and are skipped).
// KMAX >= K bounds the routes per token; the token's kept routes are put in
// ascending expert order in registers (a static ranking network, no indexed
// private memory).
template <int ACT, int OUT, int VEC, int KMAX, bool WEIGHTED, bool STATIC = false>
__global__ __launch_bounds__(256) void combine_kernel(const void* __restrict__ y, const int32_t* __restrict__ route_slot,
                                                      const int32_t* __restrict__ top_idx,
                                                      const float* __restrict__ top_w, int K, int D,
                                                      void* __restrict__ out, const BalanceJob job) {
  // products and sums rounded one by one (no fused multiply-add): the weighted
  // term is the reference's y * w, rounded to the output dtype before its
  // index_add; the sum is rounded when it is stored
#pragma clang fp contract(off)
  if constexpr (WEIGHTED && !STATIC) {  // the first workgroup finishes the balance loss, where it is asked for
    __shared__ float red[16][kWave];
    __shared__ float term[1024];
    if (job.balance != nullptr && blockIdx.x == 0) {
      balance_final<4>(job, red, term);
      return;
    }
  }
  const int t = blockIdx.x - (WEIGHTED && !STATIC && job.balance != nullptr ? 1 : 0);
  int sl[KMAX], ex[KMAX];
  float wt[KMAX];
#pragma unroll
  for (int j = 0; j < KMAX; ++j) {
    sl[j] = j < K ? route_slot[static_cast<int64_t>(t) * K + j] : -1;
    ex[j] = j < K ? top_idx[static_cast<int64_t>(t) * K + j] : 0;
    wt[j] = (WEIGHTED && j < K) ? top_w[static_cast<int64_t>(t) * K + j] : 1.0f;
    if (STATIC) wt[j] = round_act<OUT>(wt[j]);
  }
  // rank of each kept route among the kept routes by expert id (experts of a token are distinct)
  int rk[KMAX];
  int nk = 0;
#pragma unroll
  for (int j = 0; j < KMAX; ++j) {
    int r = 0;
#pragma unroll
    for (int i = 0; i < KMAX; ++i) r += (sl[i] >= 0 && ex[i] < ex[j]) ? 1 : 0;
    rk[j] = sl[j] >= 0 ? r : KMAX;
    nk += sl[j] >= 0 ? 1 : 0;
  }
  int slot[KMAX];
  float wsl[KMAX];
#pragma unroll
  for (int p = 0; p < KMAX; ++p) {
    int s = 0;
    float w = 1.0f;
#pragma unroll
    for (int j = 0; j < KMAX; ++j) {
      s = rk[j] == p ? sl[j] : s;
      w = rk[j] == p ? wt[j] : w;
    }
    slot[p] = s;
    wsl[p] = w;
  }
  const int64_t row = static_cast<int64_t>(t) * D;
  // the rows of up to G routes are requested together, then added in order
  // (a route past the kept ones reads the first kept route's row and adds
  // nothing; the empty volatile asm keeps each load ahead of the additions
  // instead of sunk into its route's branch)
  constexpr int G = KMAX < 4 ? KMAX : 4;
  static_assert(KMAX % G == 0, "whole groups of routes");
  for (int c = threadIdx.x * VEC; c < D; c += blockDim.x * VEC) {
    float acc[VEC];
#pragma unroll
    for (int v = 0; v < VEC; ++v) acc[v] = 0.0f;
    auto add = [&](const float (&yr)[VEC], float w) {
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        const float term = WEIGHTED ? round_act<OUT>(yr[v] * w) : yr[v];
        acc[v] = STATIC ? round_act<OUT>(acc[v] + term) : acc[v] + term;
      }
    };
    if constexpr (KMAX <= 16) {
#pragma unroll
      for (int j0 = 0; j0 < KMAX; j0 += G) {
        if (j0 >= nk) break;
        float yv[G][VEC];
#pragma unroll
        for (int g = 0; g < G; ++g)
          load_vec<ACT, VEC>(y, static_cast<int64_t>(j0 + g < nk ? slot[j0 + g] : slot[0]) * D + c, yv[g]);
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
          for (int v = 0; v < VEC; ++v) asm volatile("" : "+v"(yv[g][v]));
#pragma unroll
        for (int g = 0; g < G; ++g)
          if (j0 + g < nk) add(yv[g], wsl[j0 + g]);
      }
    } else {  // one route at a time
#pragma unroll
      for (int j = 0; j < KMAX; ++j) {
        if (j < nk) {
          float yv[VEC];
          load_vec<ACT, VEC>(y, static_cast<int64_t>(slot[j]) * D + c, yv);
          add(yv, wsl[j]);
        }
      }
    }
    store_vec<OUT, VEC>(out, row + c, acc);
  }
}

template <int ACT, int OUT, int KMAX, bool WEIGHTED, bool STATIC>
void launch_combine_vec(const void* y, const int32_t* route_slot, const int32_t* top_idx, const float* top_w,
                        unsigned g, int k, int d, void* out, const BalanceJob& job, hipStream_t stream) {
  constexpr int V = (ACT != QW_F32 || OUT != QW_F32) ? 8 : 4;
  if (d % V == 0)
    combine_kernel<ACT, OUT, V, KMAX, WEIGHTED, STATIC>
        <<<g, 256, 0, stream>>>(y, route_slot, top_idx, top_w, k, d, out, job);
  else
    combine_kernel<ACT, OUT, 1, KMAX, WEIGHTED, STATIC>
        <<<g, 256, 0, stream>>>(y, route_slot, top_idx, top_w, k, d, out, job);
}

template <int KMAX, bool WEIGHTED, bool STATIC>
int launch_combine(const void* y, int dtype, const int32_t* route_slot, const int32_t* top_idx, const float* top_w,
                   unsigned g, int k, int d, void* out, int out_dtype, const BalanceJob& job, hipStream_t stream) {
#define QW_CB(A, O)                                                                                             \
  if (dtype == A && out_dtype == O)                                                                             \
    launch_combine_vec<A, O, KMAX, WEIGHTED, STATIC>(y, route_slot, top_idx, top_w, g, k, d, out, job, stream); \
  else
  QW_CB(QW_F32, QW_F32)
  QW_CB(QW_F32, QW_BF16)
  QW_CB(QW_BF16, QW_F32)
  QW_CB(QW_BF16, QW_BF16)
  QW_CB(QW_F16, QW_F16)
  QW_CB(QW_F16, QW_F32)
  QW_CB(QW_F32, QW_F16)
  return set_error(QW_ERR_INVALID, "combine does not take rows of dtype %d into an output of dtype %d", dtype,
                   out_dtype);
#undef QW_CB
  QW_LAUNCH_CHECK("combine_kernel");
  return QW_OK;
}

template <bool WEIGHTED, bool STATIC = false>
int combine_k(const void* y, int dtype, const int32_t* route_slot, const int32_t* top_idx, const float* top_w,
              int64_t T, int64_t K, int64_t D, void* out, int out_dtype, hipStream_t stream,
              const BalanceJob& job = BalanceJob()) {
  const unsigned g = static_cast<unsigned>(T) + (job.balance != nullptr ? 1 : 0);
  const int k = static_cast<int>(K), d = static_cast<int>(D);
#define QW_CK(N)                                                                                                 \
  if (K <= N)                                                                                                    \
    return launch_combine<N, WEIGHTED, STATIC>(y, dtype, route_slot, top_idx, top_w, g, k, d, out, out_dtype, job, stream);
  QW_CK(2)
  QW_CK(4)
  QW_CK(8)
  QW_CK(16)
#undef QW_CK
  return launch_combine<64, WEIGHTED, STATIC>(y, dtype, route_slot, top_idx, top_w, g, k, d, out, out_dtype, job, stream);
}

static int combine_check(const void* y, int dtype, const int32_t* route_slot, const int32_t* top_idx, int64_t T,
                         int64_t K, int64_t D, void* out, int out_dtype) {
  QW_REQUIRE((dtype == QW_F32 || dtype == QW_BF16 || dtype == QW_F16) &&
                 (out_dtype == QW_F32 || out_dtype == QW_BF16 || out_dtype == QW_F16),
             "combine dtypes must be f32, bf16 or f16");
  QW_REQUIRE(!(is_half(dtype) && is_half(out_dtype) && dtype != out_dtype),
             "combine does not mix bf16 and f16 (rows %d, output %d)", dtype, out_dtype);
  QW_REQUIRE(K >= 1 && K <= 64, "combine supports top_k in [1, 64], got %lld", (long long)K);
  QW_REQUIRE(T >= 0 && T <= INT32_MAX && D >= 1 && D <= INT32_MAX, "bad combine sizes");
  QW_REQUIRE(T == 0 || (y && route_slot && top_idx && out), "combine pointers are required");
  return QW_OK;
}

int combine_weighted(const void* y, int dtype, const int32_t* route_slot, const int32_t* top_idx, const float* top_w,
                     int64_t T, int64_t K, int64_t D, void* out, int out_dtype, hipStream_t stream) {
  if (const int st = combine_check(y, dtype, route_slot, top_idx, T, K, D, out, out_dtype)) return st;
  if (T == 0) return QW_OK;
  if (top_w) return combine_k<true>(y, dtype, route_slot, top_idx, top_w, T, K, D, out, out_dtype, stream);
  return combine_k<false>(y, dtype, route_slot, top_idx, nullptr, T, K, D, out, out_dtype, stream);
}

// The weighted combine that also finishes the balance loss of `job`.
int combine_balance(const void* y, int dtype, const int32_t* route_slot, const int32_t* top_idx, const float* top_w,
                    int64_t T, int64_t K, int64_t D, void* out, int out_dtype, const BalanceJob& job,
                    hipStream_t stream) {
  if (const int st = combine_check(y, dtype, route_slot, top_idx, T, K, D, out, out_dtype)) return st;
  return combine_k<true>(y, dtype, route_slot, top_idx, top_w, T, K, D, out, out_dtype, stream, job);
}

int combine_static(const void* y, int dtype, const int32_t* route_slot, const int32_t* top_idx, const float* top_w,
                   int64_t T, int64_t K, int64_t D, void* out, int out_dtype, hipStream_t stream) {
  if (const int st = combine_check(y, dtype, route_slot, top_idx, T, K, D, out, out_dtype)) return st;
  QW_REQUIRE(T == 0 || top_w, "the static combine needs the route weights");
  if (T == 0) return QW_OK;
  return combine_k<true, true>(y, dtype, route_slot, top_idx, top_w, T, K, D, out, out_dtype, stream);
}

int combine(const void* y, int dtype, const int32_t* route_slot, const int32_t* top_idx, int64_t T, int64_t K,
            int64_t D, void* out, hipStream_t stream) {
  return combine_weighted(y, dtype, route_slot, top_idx, nullptr, T, K, D, out, dtype, stream);
}

// ---------------------------------------------------------------------------
// Decode-step combine, the last line of the one-token MoE step
// (src/fast_decode.py:177):
//   out[t] = residual[t] + ((y_0 * w_0 + y_1 * w_1) + ...)
// with y_j the expert output row of route j of token t (activation dtype,
// widened to fp32), w_j its renormalised router weight, products and sums
// rounded in fp32 in top-k order, and no rounding to the activation dtype.
// Routes without a slot (route_slot < 0) add nothing.  One block per token;
// `out` may be `residual` (each element is read, then written, by one thread).
// ---------------------------------------------------------------------------
template <int ACT, int VEC, int KMAX>
__global__ __launch_bounds__(256) void decode_combine_kernel(const void* __restrict__ y,
                                                             const int32_t* __restrict__ route_slot,
                                                             const float* __restrict__ top_w, const float* residual,
                                                             int K, int D, float* out) {
  const int t = blockIdx.x;
  const int64_t row = static_cast<int64_t>(t) * D;
  const int64_t first = static_cast<int64_t>(t) * K;
  if constexpr (KMAX > 0) {
    // K <= KMAX: the token's slots and weights are read once, the rows of up
    // to G routes and the residual are requested together, then added in
    // top-k order (a route without a slot reads the row of the token's first
    // slotted route and adds nothing; the empty volatile asm keeps each row's
    // load ahead of the additions instead of sunk into its route's branch)
    int sl[KMAX];
    float wt[KMAX];
#pragma unroll
    for (int j = 0; j < KMAX; ++j) {
      sl[j] = j < K ? route_slot[first + j] : -1;
      wt[j] = j < K ? top_w[first + j] : 0.0f;
    }
    int any = -1;
#pragma unroll
    for (int j = KMAX - 1; j >= 0; --j) any = sl[j] >= 0 ? sl[j] : any;
    constexpr int G = KMAX < 4 ? KMAX : 4;
    static_assert(KMAX % G == 0, "whole groups of routes");
    for (int c = threadIdx.x * VEC; c < D; c += blockDim.x * VEC) {
      float rv[VEC];
      if (residual != nullptr) {
#pragma unroll
        for (int v = 0; v < VEC; ++v) rv[v] = residual[row + c + v];
      }
      float acc[VEC];
#pragma unroll
      for (int v = 0; v < VEC; ++v) acc[v] = 0.0f;
#pragma unroll
      for (int j0 = 0; j0 < KMAX; j0 += G) {
        if (j0 >= K || any < 0) break;
        float yv[G][VEC];
#pragma unroll
        for (int g = 0; g < G; ++g)
          load_vec<ACT, VEC>(y, static_cast<int64_t>(sl[j0 + g] >= 0 ? sl[j0 + g] : any) * D + c, yv[g]);
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
          for (int v = 0; v < VEC; ++v) asm volatile("" : "+v"(yv[g][v]));
#pragma unroll
        for (int g = 0; g < G; ++g) {
          if (sl[j0 + g] < 0) continue;
#pragma unroll
          for (int v = 0; v < VEC; ++v) acc[v] = __fadd_rn(acc[v], __fmul_rn(yv[g][v], wt[j0 + g]));
        }
      }
      if (residual != nullptr) {
#pragma unroll
        for (int v = 0; v < VEC; ++v) acc[v] = __fadd_rn(rv[v], acc[v]);
      }
#pragma unroll
      for (int v = 0; v < VEC; ++v) out[row + c + v] = acc[v];
    }
  } else {
    for (int c = threadIdx.x * VEC; c < D; c += blockDim.x * VEC) {
      float acc[VEC];
#pragma unroll
      for (int v = 0; v < VEC; ++v) acc[v] = 0.0f;
      for (int j = 0; j < K; ++j) {
        const int s = route_slot[first + j];
        if (s < 0) continue;
        const float w = top_w[first + j];
        float yv[VEC];
        load_vec<ACT, VEC>(y, static_cast<int64_t>(s) * D + c, yv);
#pragma unroll
        for (int v = 0; v < VEC; ++v) acc[v] = __fadd_rn(acc[v], __fmul_rn(yv[v], w));
      }
      if (residual != nullptr) {
#pragma unroll
        for (int v = 0; v < VEC; ++v) acc[v] = __fadd_rn(residual[row + c + v], acc[v]);
      }
#pragma unroll
      for (int v = 0; v < VEC; ++v) out[row + c + v] = acc[v];
    }
  }
}

template <int ACT, int VEC>
void launch_decode_combine(const void* y, const int32_t* route_slot, const float* top_w, const float* residual,
                           unsigned g, int k, int d, float* out, hipStream_t stream) {
  if (k <= 2)
    decode_combine_kernel<ACT, VEC, 2><<<g, 256, 0, stream>>>(y, route_slot, top_w, residual, k, d, out);
  else if (k <= 4)
    decode_combine_kernel<ACT, VEC, 4><<<g, 256, 0, stream>>>(y, route_slot, top_w, residual, k, d, out);
  else if (k <= 8)
    decode_combine_kernel<ACT, VEC, 8><<<g, 256, 0, stream>>>(y, route_slot, top_w, residual, k, d, out);
  else
    decode_combine_kernel<ACT, VEC, 0><<<g, 256, 0, stream>>>(y, route_slot, top_w, residual, k, d, out);
}

int decode_combine(const void* y, int dtype, const int32_t* route_slot, const float* top_w, const float* residual,
                   int64_t T, int64_t K, int64_t D, float* out, hipStream_t stream) {
  QW_REQUIRE(dtype == QW_F32 || dtype == QW_BF16 || dtype == QW_F16, "decode combine dtype must be f32, bf16 or f16");
  QW_REQUIRE(T >= 0 && T <= INT32_MAX && K >= 1 && D >= 1 && D <= INT32_MAX, "bad decode combine sizes");
  if (T == 0) return QW_OK;
  QW_REQUIRE(y && route_slot && top_w && out, "decode combine pointers are required");
  const unsigned g = static_cast<unsigned>(T);
  const int k = static_cast<int>(K), d = static_cast<int>(D);
  if (dtype == QW_F16 && d % 8 == 0)
    launch_decode_combine<QW_F16, 8>(y, route_slot, top_w, residual, g, k, d, out, stream);
  else if (dtype == QW_F16)
    launch_decode_combine<QW_F16, 1>(y, route_slot, top_w, residual, g, k, d, out, stream);
  else if (dtype == QW_BF16 && d % 8 == 0)
    launch_decode_combine<QW_BF16, 8>(y, route_slot, top_w, residual, g, k, d, out, stream);
  else if (dtype == QW_BF16)
    launch_decode_combine<QW_BF16, 1>(y, route_slot, top_w, residual, g, k, d, out, stream);
  else if (d % 4 == 0)
    launch_decode_combine<QW_F32, 4>(y, route_slot, top_w, residual, g, k, d, out, stream);
  else
    launch_decode_combine<QW_F32, 1>(y, route_slot, top_w, residual, g, k, d, out, stream);
  QW_LAUNCH_CHECK("decode_combine_kernel");
  return QW_OK;
}

// fp32 -> bf16 or fp16, round to nearest even (`normed.to(dtype)`,
// src/fast_decode.py:174).  Four elements per thread when n % 4 == 0.
template <int DT>
__global__ __launch_bounds__(256) void cast_half_kernel(const float* __restrict__ x, int64_t n,
                                                        uint16_t* __restrict__ out) {
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) * 4;
  if (i >= n) return;
  if ((n & 3) == 0) {
    const float4 v = *reinterpret_cast<const float4*>(x + i);
    uint2 o;
    o.x = pack_half2<DT>(v.x, v.y);
    o.y = pack_half2<DT>(v.z, v.w);
    *reinterpret_cast<uint2*>(out + i) = o;
  } else {
    for (int64_t j = i; j < i + 4 && j < n; ++j) out[j] = f32_to_half<DT>(x[j]);
  }
}

int cast_half(const float* x, int64_t n, uint16_t* out, int dtype, hipStream_t stream) {
  QW_REQUIRE(n >= 0, "bad cast size");
  QW_REQUIRE(is_half(dtype), "the cast is to bf16 or f16");
  if (n == 0) return QW_OK;
  QW_REQUIRE(x && out, "cast pointers are required");
  const unsigned g = static_cast<unsigned>(ceil_div(ceil_div(n, 4), 256));
  if (dtype == QW_F16) cast_half_kernel<QW_F16><<<g, 256, 0, stream>>>(x, n, out);
  else cast_half_kernel<QW_BF16><<<g, 256, 0, stream>>>(x, n, out);
  QW_LAUNCH_CHECK("cast_half_kernel");
  return QW_OK;
}

// ---------------------------------------------------------------------------
// QW_BF16T packing: one thread per 16-byte piece of the tiled output, which is
// written in order (the reads are 16-byte pieces of the plain rows).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void pack_bf16_tiles_kernel(const uint16_t* __restrict__ w, int64_t pieces,
                                                              int64_t rows, int64_t cols,
                                                              uint16_t* __restrict__ out) {
  const int64_t o = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (o >= pieces) return;
  const int64_t per_expert = rows * cols / 8;
  const int64_t e = o / per_expert, rem = o % per_expert;
  const int64_t tile = rem / 64, i = rem % 64;
  const int64_t kt = cols / 64;
  const int64_t rb = tile / kt, kb = tile % kt;
  const int64_t row = 8 * rb + i / 8;
  const int64_t p = (i % 8) ^ ((row >> 1) & 7);
  const uint4 v = *reinterpret_cast<const uint4*>(w + e * rows * cols + row * cols + kb * 64 + p * 8);
  *reinterpret_cast<uint4*>(out + o * 8) = v;
}

int pack_bf16_tiles(const void* w, int64_t E, int64_t rows, int64_t cols, void* out, hipStream_t stream) {
  QW_REQUIRE(E >= 1 && rows >= 1 && cols >= 1, "bad tile packing sizes");
  QW_REQUIRE(rows % 8 == 0 && cols % 64 == 0,
             "tiled bf16 weights need out_features %% 8 == 0 and in_features %% 64 == 0 (got %lld, %lld)",
             (long long)rows, (long long)cols);
  QW_REQUIRE(w && out, "packing pointers are required");
  QW_REQUIRE(w != out, "packing cannot run in place");
  QW_REQUIRE((reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(out)) % 16 == 0,
             "packing needs 16-byte aligned buffers");
  const int64_t pieces = E * rows * cols / 8;
  pack_bf16_tiles_kernel<<<static_cast<unsigned>(ceil_div(pieces, 256)), 256, 0, stream>>>(
      static_cast<const uint16_t*>(w), pieces, rows, cols, static_cast<uint16_t*>(out));
  QW_LAUNCH_CHECK("pack_bf16_tiles_kernel");
  return QW_OK;
}

// ---------------------------------------------------------------------------
// Experts' own weight matrices -> one stack [E, rows, cols], cast and tiled on
// the way: what a training step needs after every weight update.  As torch
// operations it was a stack, a cast and a packing pass per projection, and
// another stack and cast for the backward (16 experts of 2048 x 1024 fp32:
// 640 us a step); here each weight is read once and written once, at 16 bytes
// per access, bound by HBM.  The matrices come as a table in the kernel's
// arguments, so nothing is copied to the device first.
// ---------------------------------------------------------------------------
constexpr int kPackTable = 64;  // matrices per launch
constexpr int kPackPieces = 4;  // 8-element pieces per thread

struct PackTable {
  const void* w[kPackTable];
};

template <int SRC, int DST, bool TILED>
__global__ __launch_bounds__(256) void pack_experts_kernel(const PackTable table, int64_t pieces, int64_t cols,
                                                           void* __restrict__ out) {
  const void* const w = table.w[blockIdx.y];
  const int64_t first = static_cast<int64_t>(blockIdx.x) * (256 * kPackPieces) + threadIdx.x;
  const int64_t base = static_cast<int64_t>(blockIdx.y) * pieces;  // the expert's first piece of the stack
  float v[kPackPieces][8];
#pragma unroll
  for (int u = 0; u < kPackPieces; ++u) {
    const int64_t o = first + 256 * u;
    if (o >= pieces) break;
    int64_t src = 8 * o;
    if constexpr (TILED) {  // output piece o of the QW_BF16T tiles
      const int64_t tile = o / 64, i = o % 64, kt = cols / 64;
      const int64_t row = 8 * (tile / kt) + i / 8;
      src = row * cols + (tile % kt) * 64 + ((i % 8) ^ ((row >> 1) & 7)) * 8;
    }
    load_vec<SRC, 8>(w, src, v[u]);
  }
#pragma unroll
  for (int u = 0; u < kPackPieces; ++u) {
    const int64_t o = first + 256 * u;
    if (o >= pieces) break;
    store_vec<DST, 8>(out, 8 * (base + o), v[u]);
  }
}

int pack_experts(const void* const* weights, int src, int64_t E, int64_t rows, int64_t cols, void* out, int fmt,
                 hipStream_t stream) {
  QW_REQUIRE(E >= 1 && rows >= 1 && cols >= 1 && rows <= INT32_MAX / 2 && cols <= INT32_MAX / 2, "bad packing sizes");
  QW_REQUIRE(weights && out, "packing pointers are required");
  QW_REQUIRE(src == QW_F32 || src == QW_BF16 || src == QW_F16, "packed weights must be f32, bf16 or f16");
  const bool tiled = fmt == QW_BF16T || fmt == QW_F16T;
  const int dst = fmt == QW_BF16T ? QW_BF16 : fmt == QW_F16T ? QW_F16 : fmt;
  QW_REQUIRE(dst == QW_F32 || dst == QW_BF16 || dst == QW_F16, "packing makes plain or tiled float stacks");
  QW_REQUIRE(cols % 8 == 0 && (!tiled || (rows % 8 == 0 && cols % 64 == 0)),
             "packing needs in_features %% 8 == 0, tiles out_features %% 8 == 0 and in_features %% 64 == 0");
  QW_REQUIRE(reinterpret_cast<uintptr_t>(out) % 16 == 0, "packing needs 16-byte aligned buffers");
  const int64_t pieces = rows * cols / 8;
  const int64_t blocks = ceil_div(pieces, 256 * kPackPieces);
  QW_REQUIRE(blocks <= INT32_MAX, "matrix too large to pack");
  for (int64_t e0 = 0; e0 < E; e0 += kPackTable) {
    PackTable t{};
    const int n = static_cast<int>(E - e0 < kPackTable ? E - e0 : kPackTable);
    for (int i = 0; i < n; ++i) {
      t.w[i] = weights[e0 + i];
      QW_REQUIRE(t.w[i] != nullptr && reinterpret_cast<uintptr_t>(t.w[i]) % 16 == 0,
                 "packing needs 16-byte aligned matrices");
    }
    void* const to = static_cast<char*>(out) + e0 * rows * cols * (dst == QW_F32 ? 4 : 2);
    const dim3 g(static_cast<unsigned>(blocks), static_cast<unsigned>(n));
#define QW_PK(S, D, T)                                                            \
  if (src == S && dst == D && tiled == T) {                                       \
    pack_experts_kernel<S, D, T><<<g, 256, 0, stream>>>(t, pieces, cols, to);     \
  }
    QW_PK(QW_F32, QW_F32, false)
    QW_PK(QW_F32, QW_BF16, false)
    QW_PK(QW_F32, QW_BF16, true)
    QW_PK(QW_F32, QW_F16, false)
    QW_PK(QW_F32, QW_F16, true)
    QW_PK(QW_BF16, QW_F32, false)
    QW_PK(QW_BF16, QW_BF16, false)
    QW_PK(QW_BF16, QW_BF16, true)
    QW_PK(QW_BF16, QW_F16, false)
    QW_PK(QW_BF16, QW_F16, true)
    QW_PK(QW_F16, QW_F32, false)
    QW_PK(QW_F16, QW_F16, false)
    QW_PK(QW_F16, QW_F16, true)
    QW_PK(QW_F16, QW_BF16, false)
    QW_PK(QW_F16, QW_BF16, true)
#undef QW_PK
    QW_LAUNCH_CHECK("pack_experts_kernel");
  }
  return QW_OK;
}

// ---------------------------------------------------------------------------
// Balance loss (src/quantweave_moe_model.py:152-154).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void importance_kernel(const float* __restrict__ probs, int T, int E,
                                                         float* __restrict__ importance) {
  __shared__ float red[256];
  const int e = blockIdx.x;
  float s = 0.0f;
  for (int t = threadIdx.x; t < T; t += 256) s += probs[static_cast<int64_t>(t) * E + e];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int o = 128; o >= 1; o >>= 1) {
    if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) importance[e] = red[0] / static_cast<float>(T);
}

__global__ void balance_kernel(const float* __restrict__ importance, const int32_t* __restrict__ counts, int T, int K,
                               int E, float* __restrict__ balance) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  const float routes = static_cast<float>(static_cast<int64_t>(T) * K);
  float s = 0.0f;
  for (int e = 0; e < E; ++e) s += importance[e] * (static_cast<float>(counts[e]) / routes);
  *balance = static_cast<float>(E) * s;
}

// The same with partial sums per 64 tokens (coalesced row reads) summed
// afterwards in a fixed order: deterministic, and the probs matrix is read by
// many CUs instead of one workgroup per strided column.
__global__ __launch_bounds__(256) void importance_partial_kernel(const BalanceJob job) {
  __shared__ float red[4][kWave];
  importance_unit(job, blockIdx.x, red);
}

// Alone on the chip it takes 16 waves (8192 tokens, 184 experts: 11.2 us with the
// partial sums, 17.3 with 4 waves in all forms).
template <int WAVES, BalanceForm FORM>
__global__ __launch_bounds__(WAVES * kWave) void importance_final_kernel(const BalanceJob job) {
  __shared__ float red[16][kWave];
  __shared__ float term[1024];
  balance_final<WAVES, FORM>(job, red, term);
}

size_t balance_workspace_bytes(int64_t T, int64_t E) {
  return static_cast<size_t>(ceil_div(T, kImpRows)) * static_cast<size_t>(E) * sizeof(float) + 256;
}

int balance_ws(const float* probs, const int32_t* counts, int64_t T, int64_t K, int64_t E, float* importance,
               float* bal, void* ws, size_t ws_bytes, hipStream_t stream) {
  QW_REQUIRE(T >= 1 && T <= INT32_MAX && E >= 1 && E <= 1024 && K >= 1, "bad balance sizes");
  QW_REQUIRE(probs && counts && bal && importance, "balance pointers are required");
  const size_t need = balance_workspace_bytes(T, E);
  if (!ws || ws_bytes < need)
    return set_error(QW_ERR_WORKSPACE, "balance workspace needs %zu bytes, got %zu", need, ws_bytes);
  BalanceJob job;
  job.probs = probs;
  job.counts = counts;
  job.partial = static_cast<float*>(ws);
  job.nb = static_cast<int>(ceil_div(T, kImpRows));
  job.T = static_cast<int>(T);
  job.K = static_cast<int>(K);
  job.E = static_cast<int>(E);
  job.importance = importance;
  job.balance = bal;
  if (job.nb > 1) {
    importance_partial_kernel<<<static_cast<unsigned>(partial_units(job.nb, job.E)), 256, 0, stream>>>(job);
    QW_LAUNCH_CHECK("importance_partial_kernel");
  }
  if (job.nb <= 16 && E > kWave) importance_final_kernel<16, kThreadPerExpert><<<1, 1024, 0, stream>>>(job);
  else if (job.nb > 1) importance_final_kernel<16, kManyRows><<<1, 1024, 0, stream>>>(job);
  else importance_final_kernel<4, kAnyForm><<<1, 256, 0, stream>>>(job);
  QW_LAUNCH_CHECK("importance_final_kernel");
  return QW_OK;
}

int balance(const float* probs, const int32_t* counts, int64_t T, int64_t K, int64_t E, float* importance,
            float* bal, hipStream_t stream, float* scratch_importance) {
  QW_REQUIRE(T >= 1 && T <= INT32_MAX && E >= 1 && E <= 1024 && K >= 1, "bad balance sizes");
  QW_REQUIRE(probs && counts && bal, "balance pointers are required");
  float* imp = importance ? importance : scratch_importance;
  QW_REQUIRE(imp != nullptr, "balance needs an importance buffer");
  importance_kernel<<<static_cast<unsigned>(E), 256, 0, stream>>>(probs, static_cast<int>(T), static_cast<int>(E), imp);
  QW_LAUNCH_CHECK("importance_kernel");
  balance_kernel<<<1, 64, 0, stream>>>(imp, counts, static_cast<int>(T), static_cast<int>(K), static_cast<int>(E), bal);
  QW_LAUNCH_CHECK("balance_kernel");
  return QW_OK;
}

// ---------------------------------------------------------------------------
// Quantisation, QuantizedLinear.from_linear (src/quantization.py:43-59).
// One thread per (row, group).
// ---------------------------------------------------------------------------
template <int WDT, int BITS>
__global__ void quantize_kernel(const void* __restrict__ w, int64_t rows, int64_t cols, int64_t group,
                                int64_t groups, void* __restrict__ qweight, float* __restrict__ scales) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= rows * groups) return;
  const int64_t row = i / groups, g = i % groups;
  const int64_t c0 = g * group;
  const float limit = BITS == 8 ? 127.0f : 7.0f;
  const float lo = BITS == 8 ? -127.0f : -8.0f;
  float amax = 0.0f;
  for (int64_t c = c0; c < c0 + group; ++c) {
    const float v = c < cols ? load_act<WDT>(w, row * cols + c) : 0.0f;
    amax = fmaxf(amax, fabsf(v));
  }
  const float s = fmaxf(amax / limit, 1e-8f);
  scales[row * groups + g] = s;
  if (BITS == 8) {
    int8_t* q = static_cast<int8_t*>(qweight) + row * groups * group;
    for (int64_t c = c0; c < c0 + group; ++c) {
      const float v = c < cols ? load_act<WDT>(w, row * cols + c) : 0.0f;
      const float r = fminf(fmaxf(__builtin_rintf(v / s), lo), limit);
      q[c] = static_cast<int8_t>(r);
    }
  } else {
    uint8_t* q = static_cast<uint8_t*>(qweight) + row * (groups * group / 2);
    for (int64_t c = c0; c < c0 + group; c += 2) {
      const float v0 = c < cols ? load_act<WDT>(w, row * cols + c) : 0.0f;
      const float v1 = c + 1 < cols ? load_act<WDT>(w, row * cols + c + 1) : 0.0f;
      const int q0 = static_cast<int>(fminf(fmaxf(__builtin_rintf(v0 / s), lo), limit)) + 8;
      const int q1 = static_cast<int>(fminf(fmaxf(__builtin_rintf(v1 / s), lo), limit)) + 8;
      q[c / 2] = static_cast<uint8_t>(q0 | (q1 << 4));
    }
  }
}

int quantize(const void* w, int wdt, int64_t rows, int64_t cols, int bits, int64_t group, void* qweight, float* scales,
             hipStream_t stream) {
  QW_REQUIRE(bits == 4 || bits == 8, "bits must be 4 or 8");
  QW_REQUIRE(wdt == QW_F32 || wdt == QW_BF16 || wdt == QW_F16, "weight dtype must be f32, bf16 or f16");
  QW_REQUIRE(group >= 1, "group_size must be positive");
  QW_REQUIRE(!(bits == 4 && (group % 2)), "group_size must be even for 4-bit weights");
  QW_REQUIRE(rows >= 0 && cols >= 1, "bad quantize sizes");
  if (rows == 0) return QW_OK;
  QW_REQUIRE(w && qweight && scales, "quantize pointers are required");
  const int64_t groups = ceil_div(cols, group);
  const int64_t n = rows * groups;
  const unsigned g = static_cast<unsigned>(ceil_div(n, 256));
  if (wdt == QW_F32 && bits == 8) quantize_kernel<QW_F32, 8><<<g, 256, 0, stream>>>(w, rows, cols, group, groups, qweight, scales);
  else if (wdt == QW_F32) quantize_kernel<QW_F32, 4><<<g, 256, 0, stream>>>(w, rows, cols, group, groups, qweight, scales);
  else if (wdt == QW_F16 && bits == 8) quantize_kernel<QW_F16, 8><<<g, 256, 0, stream>>>(w, rows, cols, group, groups, qweight, scales);
  else if (wdt == QW_F16) quantize_kernel<QW_F16, 4><<<g, 256, 0, stream>>>(w, rows, cols, group, groups, qweight, scales);
  else if (bits == 8) quantize_kernel<QW_BF16, 8><<<g, 256, 0, stream>>>(w, rows, cols, group, groups, qweight, scales);
  else quantize_kernel<QW_BF16, 4><<<g, 256, 0, stream>>>(w, rows, cols, group, groups, qweight, scales);
  QW_LAUNCH_CHECK("quantize_kernel");
  return QW_OK;
}

template <int WF>
__global__ void dequantize_kernel(WView v, float* __restrict__ out) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= v.rows * v.cols) return;
  const int64_t row = i / v.cols, col = i % v.cols;
  out[i] = load_weight<WF>(v, 0, row, col);
}

int dequantize(const void* qweight, const float* scales, int bits, int64_t rows, int64_t cols, int64_t group,
               float* out, hipStream_t stream) {
  QW_REQUIRE(bits == 4 || bits == 8, "bits must be 4 or 8");
  QW_REQUIRE(group >= 1 && !(bits == 4 && (group % 2)), "bad group_size");
  QW_REQUIRE(rows >= 0 && cols >= 1, "bad dequantize sizes");
  if (rows == 0) return QW_OK;
  QW_REQUIRE(qweight && scales && out, "dequantize pointers are required");
  const WView v = make_wview(bits == 8 ? QW_I8 : QW_U4, qweight, scales, rows, cols, group);
  const unsigned g = static_cast<unsigned>(ceil_div(rows * cols, 256));
  if (bits == 8) dequantize_kernel<QW_I8><<<g, 256, 0, stream>>>(v, out);
  else dequantize_kernel<QW_U4><<<g, 256, 0, stream>>>(v, out);
  QW_LAUNCH_CHECK("dequantize_kernel");
  return QW_OK;
}

}  // namespace qw
