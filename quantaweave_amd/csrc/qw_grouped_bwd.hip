// Backward of the grouped matmul y[rows of e] = x[rows of e] @ W[e]^T.
//
// Reference: _GroupedMatmul.backward (src/moe_kernels.py:146-164) with its two
// kernels: grad_x through the forward kernel with the weight transposed
// (:118-135, transpose=True), and _grouped_dw_kernel (:66-89):
//   grad_x[r, k]    = sum_n grad_y[r, n] * W[e][n, k]          (r in rows of e)
//   grad_W[e][n, k] = sum_{r in rows of e} grad_y[r, n] * x[r, k]
// An expert without rows gets an exactly zero grad_W.  fp32 accumulation,
// output in the operands' dtype (fp32 or bf16); with `accumulate` grad_x
// receives grad_x + result (one rounding), which sums the gate and up
// projections' input gradients of a SwiGLU expert in place.
//
// bf16 and fp16 with a workspace run on the matrix cores (gemm_grouped_backward,
// qw_gemm_mfma.hip, or gemm_tr_dx and gemm_tr_dw, qw_gemm_tr.hip); fp32 runs on
// the fp32 matrix cores (grouped_f32_kernel below) when rows are 16-byte aligned.  Otherwise two
// vector-ALU kernels compute a 64x64 output tile per 256-thread
// block (4x4 per thread) from 16-deep slices of the reduction staged in LDS;
// the reduction runs in ascending order, so results do not depend on
// scheduling.
#include "qw_mfma.h"

namespace qw {

namespace {

constexpr int BT = 64;  // output tile edge
constexpr int BR = 16;  // reduction slice

// grad_x: block (k tile, row tile, expert)
template <int DT>
__global__ __launch_bounds__(256) void grouped_dx_kernel(const void* __restrict__ gy, const void* __restrict__ w,
                                                         const int32_t* __restrict__ offsets, int N, int K,
                                                         int rows, int accumulate, void* __restrict__ gx) {
  __shared__ float gs[BR][BT + 4];  // [n][row]
  __shared__ float ws[BR][BT + 4];  // [n][k]
  const int e = blockIdx.z;
  const int lo = min(max(offsets[e], 0), rows), hi = min(offsets[e + 1], rows);
  const int r0 = lo + blockIdx.y * BT;
  if (r0 >= hi) return;
  const int k0 = blockIdx.x * BT;
  const int tid = threadIdx.x, ty = tid / 16, tx = tid % 16;
  const int64_t wbase = static_cast<int64_t>(e) * N * K;
  float acc[4][4] = {};
  for (int n0 = 0; n0 < N; n0 += BR) {
    for (int i = tid; i < BT * BR; i += 256) {
      const int m = i / BR, nn = i % BR;
      const int r = r0 + m, n = n0 + nn;
      gs[nn][m] = (r < hi && n < N) ? load_act<DT>(gy, static_cast<int64_t>(r) * N + n) : 0.0f;
      const int wn = i / BT, kk = i % BT;
      const int n2 = n0 + wn, k = k0 + kk;
      ws[wn][kk] = (n2 < N && k < K) ? load_act<DT>(w, wbase + static_cast<int64_t>(n2) * K + k) : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int nn = 0; nn < BR; ++nn) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = gs[nn][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = ws[nn][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = r0 + ty * 4 + i;
    if (r >= hi) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = k0 + tx * 4 + j;
      if (k >= K) continue;
      const int64_t o = static_cast<int64_t>(r) * K + k;
      store_act<DT>(gx, o, accumulate ? load_act<DT>(gx, o) + acc[i][j] : acc[i][j]);
    }
  }
}

// grad_W: block (k tile, n tile, expert); ODT the output dtype
template <int DT, int ODT>
__global__ __launch_bounds__(256) void grouped_dw_kernel(const void* __restrict__ gy, const void* __restrict__ x,
                                                         const int32_t* __restrict__ offsets, int N, int K,
                                                         int rows, void* __restrict__ gw) {
  __shared__ float gs[BR][BT + 4];  // [row][n]
  __shared__ float xs[BR][BT + 4];  // [row][k]
  const int e = blockIdx.z;
  const int lo = min(max(offsets[e], 0), rows), hi = min(offsets[e + 1], rows);
  const int n0 = blockIdx.y * BT, k0 = blockIdx.x * BT;
  const int tid = threadIdx.x, ty = tid / 16, tx = tid % 16;
  float acc[4][4] = {};
  for (int m0 = lo; m0 < hi; m0 += BR) {
    for (int i = tid; i < BR * BT; i += 256) {
      const int m = i / BT, c = i % BT;
      const int r = m0 + m;
      const bool ok = r < hi;
      gs[m][c] = (ok && n0 + c < N) ? load_act<DT>(gy, static_cast<int64_t>(r) * N + n0 + c) : 0.0f;
      xs[m][c] = (ok && k0 + c < K) ? load_act<DT>(x, static_cast<int64_t>(r) * K + k0 + c) : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < BR; ++m) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = gs[m][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = xs[m][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
  const int64_t wbase = static_cast<int64_t>(e) * N * K;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int n = n0 + ty * 4 + i;
    if (n >= N) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = k0 + tx * 4 + j;
      if (k < K) store_act<ODT>(gw, wbase + static_cast<int64_t>(n) * K + k, acc[i][j]);
    }
  }
}

// ---------------------------------------------------------------------------
// fp32 on the matrix cores (v_mfma_f32_16x16x4_f32, one fp32 per lane and
// operand: lane group q of the four instructions j of a 16-wide step takes
// reduction index 4q + j).  A 256-thread workgroup (2 x 2 waves) computes a
// 64 x 64 output tile.  The matrix cores bound it (32 clocks an instruction), as
// long as nothing waits: operands go straight to LDS (global_load_lds, a ring
// of four 32-deep slices, three requested ahead) as they lie in memory.  A
// reduction-major one is read one fp32 per lane, 16 columns of 4 rows: the
// 16-column group c of row r sits at c ^ ((r / 4) % 4), so the four rows
// cover all banks.  The other kind (rows of gy for grad_x) is read 16 bytes
// per lane.  Transposing on the way into LDS, through registers, cost as many
// LDS clocks as the products.  16 experts, 16000 rows, out x in 512 x 256: grad_x
// 59 -> 51 us, grad_W 66 -> 46 (92 of the 157 TFLOP/s); 1408 x 1024, 2000 rows:
// 71 -> 61 and 94 -> 70.
// The reduction runs in ascending order.
// ---------------------------------------------------------------------------
typedef float bf32x4 __attribute__((ext_vector_type(4)));
constexpr int FB_T = 64, FB_R = 32, FB_ST = 4, FB_OPER = FB_T * FB_R;  // tile, slice, stages, floats per operand

__device__ const uint4 g_fb_zero = {0u, 0u, 0u, 0u};  // pieces past the end of the reduction

// RED: grad_W_e[n, k] = sum over the rows r of expert e of gy[r, n] a[r, k], a = x
//      (exactly zero without rows); block (k tile, n tile, expert).
// else: grad_x[r, k] (+)= sum_n gy[r, n] a[n, k], a = W_e; block (k tile, row tile, expert).
template <bool RED>
__global__ __launch_bounds__(256) void grouped_f32_kernel(const float* __restrict__ gy, const float* __restrict__ a,
                                                          const int32_t* __restrict__ offsets, int N, int K, int rows,
                                                          int accumulate, float* __restrict__ out) {
  __shared__ __attribute__((aligned(1024))) float ring[FB_ST][2][FB_OPER];
  const int e = blockIdx.z;
  const int lo = min(max(offsets[e], 0), rows), hi = min(offsets[e + 1], rows);
  const int m0 = blockIdx.y * FB_T, k0 = blockIdx.x * FB_T;  // first row of the tile (of the expert's), first column
  const int mcount = min(FB_T, (RED ? N : hi - lo) - m0);
  if (mcount <= 0) return;
  const int red = RED ? max(hi - lo, 0) : N;
  const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int wm = wave / 2, wn = wave % 2, l16 = lane % 16, lq = lane / 16;
  // this lane's piece of load group wave + 4 q (1 KiB): source at the first
  // slice, and the first reduction index it holds
  const float *a_src[2], *b_src[2];
  int a_red[2], b_red[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int g = wave + 4 * q;
    const int r = 4 * g + lane / 16, c = 4 * ((lane % 16) ^ ((g & 3) << 2));
    a_red[q] = r;
    a_src[q] = a + (RED ? static_cast<int64_t>(lo) : static_cast<int64_t>(e) * N) * K + static_cast<int64_t>(r) * K +
               min(k0 + c, K - 4);
    if constexpr (RED) {
      b_red[q] = r;
      b_src[q] = gy + static_cast<int64_t>(lo + r) * N + min(m0 + c, N - 4);
    } else {
      const int row = 8 * g + lane / 8;
      b_red[q] = 4 * ((lane % 8) ^ ((row >> 1) & 7));
      b_src[q] = gy + static_cast<int64_t>(lo + m0 + min(row, mcount - 1)) * N + b_red[q];
    }
  }
  const int64_t a_step = static_cast<int64_t>(FB_R) * K, b_step = RED ? static_cast<int64_t>(FB_R) * N : FB_R;
  auto issue = [&](int s) {
    float* st = &ring[s % FB_ST][0][0];
    const int left = red - s * FB_R;  // reduction indices from this slice on
    const float* zero = reinterpret_cast<const float*>(&g_fb_zero);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const float* src = a_red[q] < left ? a_src[q] + s * a_step : zero;
      __builtin_amdgcn_global_load_lds(static_cast<const void*>(src), (lds_void*)(st + (wave + 4 * q) * 256), 16, 0, 0);
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const float* src = b_red[q] < left ? b_src[q] + s * b_step : zero;
      __builtin_amdgcn_global_load_lds(static_cast<const void*>(src), (lds_void*)(st + FB_OPER + (wave + 4 * q) * 256),
                                       16, 0, 0);
    }
  };
  bf32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int t = 0; t < 2; ++t) acc[i][t] = bf32x4{0.f, 0.f, 0.f, 0.f};
  const int S = (red + FB_R - 1) / FB_R;  // 0 for an expert without rows
  for (int s = 0; s < FB_ST - 1 && s < S; ++s) issue(s);
  static_assert(FB_ST == 4, "the waits below");
  for (int s = 0; s < S; ++s) {
    // four loads per wave and slice; the two slices after this one stay in flight
    if (s + 2 < S) wait_vmcnt<8>();
    else if (s + 1 < S) wait_vmcnt<4>();
    else wait_vmcnt<0>();
    ring_barrier();
    if (s + FB_ST - 1 < S) issue(s + FB_ST - 1);  // into the stage of slice s - 1
    const float* As = &ring[s % FB_ST][0][0];
    const float* Bs = As + FB_OPER;
#pragma unroll
    for (int kk = 0; kk < FB_R; kk += 16) {
      float av[2][4], bv[2][4];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) av[t][j] = As[(kk + 4 * lq + j) * FB_T + (((2 * wn + t) ^ lq) << 4) + l16];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if constexpr (RED) {
#pragma unroll
          for (int j = 0; j < 4; ++j) bv[i][j] = Bs[(kk + 4 * lq + j) * FB_T + (((2 * wm + i) ^ lq) << 4) + l16];
        } else {
          const int row = wm * 32 + 16 * i + l16;
          const bf32x4 v = *reinterpret_cast<const bf32x4*>(Bs + row * FB_R + 4 * ((kk / 4 + lq) ^ ((row >> 1) & 7)));
#pragma unroll
          for (int j = 0; j < 4; ++j) bv[i][j] = v[j];
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int t = 0; t < 2; ++t)
            acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[t][j], bv[i][j], acc[i][t], 0, 0, 0);
    }
  }
  // lane holds row wm*32 + 16i + l16, columns wn*32 + 16t + 4lq .. +3
  float* const base = out + (RED ? static_cast<int64_t>(e) * N + m0 : static_cast<int64_t>(lo) + m0) * K;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int m = wm * 32 + 16 * i + l16;
    if (m >= mcount) continue;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int k = k0 + wn * 32 + 16 * t + 4 * lq;
      if (k >= K) continue;  // K % 4 == 0: wholly inside or past the end
      bf32x4* o = reinterpret_cast<bf32x4*>(base + static_cast<int64_t>(m) * K + k);
      bf32x4 v = acc[i][t];
      if (!RED && accumulate) {
        const bf32x4 old = *o;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = old[j] + v[j];
      }
      *o = v;
    }
  }
}

}  // namespace

size_t gemm_backward_workspace_bytes(int64_t E, int64_t N, int64_t K, int64_t rows);
bool gemm_backward_fits(int64_t rows, int64_t E);
int gemm_grouped_backward(const void* gy, const void* x, const void* w, int dtype, int64_t E, int64_t N, int64_t K,
                          const int32_t* offsets, int64_t rows, int64_t rows_per_expert, void* gx, int accumulate,
                          void* gw, int gw_f32, bool tiled, void* ws, size_t ws_bytes, hipStream_t stream);

bool gemm_tr_dx_fits(const void* gy, const void* w, const void* gx, int64_t E, int64_t N, int64_t K, int64_t rows,
                     bool pair, bool tiles128);
int gemm_tr_dx(const void* gy0, const void* gy1, const void* w0, const void* w1, int dtype, bool tiled, int64_t E,
               int64_t N, int64_t K, const int32_t* offsets, int64_t rows, void* gx, hipStream_t stream);
bool gemm_tr_dw_fits(const void* gy, const void* x, const void* gw, int64_t E, int64_t N, int64_t K);
int gemm_tr_dw(const void* gy0, const void* gy1, const void* x, int dtype, int64_t E, int64_t N, int64_t K,
               const int32_t* offsets, int64_t rows, void* gw0, void* gw1, int gw_f32, hipStream_t stream);

size_t grouped_backward_workspace_bytes(int64_t E, int64_t N, int64_t K, int64_t rows, int dtype) {
  return is_half(dtype) ? gemm_backward_workspace_bytes(E, N, K, rows) : 256;
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

int grouped_matmul_backward(const void* gy, const void* x, const void* w, int dtype, int wfmt, int64_t E, int64_t N,
                            int64_t K, const int32_t* offsets, int64_t rows, int64_t max_rows_per_expert, void* gx,
                            int accumulate, void* gw, int gw_dtype, void* ws, size_t ws_bytes, hipStream_t stream) {
  const bool tiled = wfmt != dtype;
  QW_REQUIRE(dtype == QW_F32 || dtype == QW_BF16 || dtype == QW_F16, "grouped backward dtype must be f32, bf16 or f16");
  QW_REQUIRE(gw_dtype == dtype || gw_dtype == QW_F32, "grad_w dtype must be the operands' dtype or f32");
  QW_REQUIRE(E >= 1 && E <= 65535 && N >= 1 && K >= 1 && N <= INT32_MAX && K <= INT32_MAX && rows >= 0 &&
                 rows <= INT32_MAX && max_rows_per_expert >= 0,
             "bad grouped backward sizes");
  QW_REQUIRE(!tiled || (dtype == QW_BF16 && wfmt == QW_BF16T) || (dtype == QW_F16 && wfmt == QW_F16T),
             "grouped backward weights must be of the operands' dtype, plain or tiled");
  QW_REQUIRE(!tiled || (N % 64 == 0 && K % 64 == 0), "tiled weights need sizes that are multiples of 64");
  QW_REQUIRE(offsets != nullptr, "offsets are required");
  if (gx != nullptr && rows > 0) QW_REQUIRE(gy && w, "grad_x needs grad_out and w");
  if (gw != nullptr) QW_REQUIRE(rows == 0 || (gy && x), "grad_w needs grad_out and x");
  const int64_t per = max_rows_per_expert > 0 && max_rows_per_expert < rows ? max_rows_per_expert : rows;
  QW_REQUIRE(ceil_div(per, BT) <= 65535 && ceil_div(N, BT) <= 65535, "grouped backward sizes out of range");
  // 128 x 128 tiles (bf16/fp16 with a workspace): dX needs out_features % 64 == 0, dW any shape
  const bool core = is_half(dtype) && ws != nullptr && ws_bytes >= gemm_backward_workspace_bytes(E, N, K, rows) &&
                    aligned16(gy) && aligned16(x) && aligned16(w) && gemm_backward_fits(rows, E);
  const bool core_dx = core && aligned16(gx) && N % 64 == 0 && K % 4 == 0;
  const bool core_dw = core && aligned16(gw);
  // 256-column tiles over the operands as they lie (no workspace used)
  if (is_half(dtype) && gx != nullptr && !accumulate && rows > 0 &&
      gemm_tr_dx_fits(gy, w, gx, E, N, K, rows, false, core_dx)) {
    const int st = gemm_tr_dx(gy, nullptr, w, nullptr, dtype, tiled, E, N, K, offsets, rows, gx, stream);
    if (st) return st;
    gx = nullptr;
  }
  if (is_half(dtype) && gw != nullptr && gemm_tr_dw_fits(gy, x, gw, E, N, K)) {
    const int st = gemm_tr_dw(gy, nullptr, x, dtype, E, N, K, offsets, rows, gw, nullptr, gw_dtype == QW_F32, stream);
    if (st) return st;
    gw = nullptr;
  }
  if ((core_dx && gx != nullptr) || (core_dw && gw != nullptr)) {
    const int st = gemm_grouped_backward(gy, x, w, dtype, E, N, K, offsets, rows, per, core_dx ? gx : nullptr, accumulate,
                                         core_dw ? gw : nullptr, gw_dtype == QW_F32, tiled, ws, ws_bytes, stream);
    if (st) return st;
    if (core_dx) gx = nullptr;
    if (core_dw) gw = nullptr;
  }
  if (tiled && gx != nullptr && rows > 0)
    return set_error(QW_ERR_UNSUPPORTED, "tiled weights need the matrix-core backward (workspace, aligned buffers)");
  const int n = static_cast<int>(N), k = static_cast<int>(K), r = static_cast<int>(rows);
  // fp32 matrix-core path: 16-byte rows and bases
  const bool f32_core = dtype == QW_F32 && N % 4 == 0 && K % 4 == 0 && aligned16(gy) && aligned16(x) &&
                        aligned16(w) && (gx == nullptr || aligned16(gx)) && (gw == nullptr || aligned16(gw));
  if (f32_core && gx != nullptr && rows > 0) {
    const dim3 g(static_cast<unsigned>(ceil_div(K, FB_T)), static_cast<unsigned>(ceil_div(per, FB_T)),
                 static_cast<unsigned>(E));
    grouped_f32_kernel<false><<<g, 256, 0, stream>>>(static_cast<const float*>(gy), static_cast<const float*>(w),
                                                     offsets, n, k, r, accumulate, static_cast<float*>(gx));
    QW_LAUNCH_CHECK("grouped_f32_kernel");
    gx = nullptr;
  }
  if (f32_core && gw != nullptr && gw_dtype == QW_F32) {
    const dim3 g(static_cast<unsigned>(ceil_div(K, FB_T)), static_cast<unsigned>(ceil_div(N, FB_T)),
                 static_cast<unsigned>(E));
    grouped_f32_kernel<true><<<g, 256, 0, stream>>>(static_cast<const float*>(gy), static_cast<const float*>(x),
                                                    offsets, n, k, r, 0, static_cast<float*>(gw));
    QW_LAUNCH_CHECK("grouped_f32_kernel");
    gw = nullptr;
  }
  if (gx != nullptr && rows > 0) {
    const dim3 g(static_cast<unsigned>(ceil_div(K, BT)), static_cast<unsigned>(ceil_div(per, BT)),
                 static_cast<unsigned>(E));
    if (dtype == QW_F32) grouped_dx_kernel<QW_F32><<<g, 256, 0, stream>>>(gy, w, offsets, n, k, r, accumulate, gx);
    else if (dtype == QW_F16) grouped_dx_kernel<QW_F16><<<g, 256, 0, stream>>>(gy, w, offsets, n, k, r, accumulate, gx);
    else grouped_dx_kernel<QW_BF16><<<g, 256, 0, stream>>>(gy, w, offsets, n, k, r, accumulate, gx);
    QW_LAUNCH_CHECK("grouped_dx_kernel");
  }
  if (gw != nullptr) {
    const dim3 g(static_cast<unsigned>(ceil_div(K, BT)), static_cast<unsigned>(ceil_div(N, BT)),
                 static_cast<unsigned>(E));
    if (dtype == QW_F32) grouped_dw_kernel<QW_F32, QW_F32><<<g, 256, 0, stream>>>(gy, x, offsets, n, k, r, gw);
    else if (dtype == QW_F16 && gw_dtype == QW_F32)
      grouped_dw_kernel<QW_F16, QW_F32><<<g, 256, 0, stream>>>(gy, x, offsets, n, k, r, gw);
    else if (dtype == QW_F16) grouped_dw_kernel<QW_F16, QW_F16><<<g, 256, 0, stream>>>(gy, x, offsets, n, k, r, gw);
    else if (gw_dtype == QW_F32) grouped_dw_kernel<QW_BF16, QW_F32><<<g, 256, 0, stream>>>(gy, x, offsets, n, k, r, gw);
    else grouped_dw_kernel<QW_BF16, QW_BF16><<<g, 256, 0, stream>>>(gy, x, offsets, n, k, r, gw);
    QW_LAUNCH_CHECK("grouped_dw_kernel");
  }
  return QW_OK;
}

// Two products of the same x: gx = gy_a . w_a + gy_b . w_b, gw_a and gw_b.
int grouped_matmul_backward_pair(const void* gy_a, const void* gy_b, const void* x, const void* w_a, const void* w_b,
                                 int dtype, int wfmt, int64_t E, int64_t N, int64_t K, const int32_t* offsets,
                                 int64_t rows, int64_t max_rows_per_expert, void* gx, void* gw_a, void* gw_b,
                                 int gw_dtype, void* ws, size_t ws_bytes, hipStream_t stream) {
  // the checks of the single product, which launches nothing here
  int st = grouped_matmul_backward(gy_a, x, w_a, dtype, wfmt, E, N, K, offsets, rows, max_rows_per_expert, nullptr, 0,
                                   nullptr, gw_dtype, ws, ws_bytes, stream);
  if (st) return st;
  if (gx != nullptr && rows > 0) QW_REQUIRE(gy_a && gy_b && w_a && w_b, "grad_x needs grad_out and w");
  if (gw_a != nullptr || gw_b != nullptr) QW_REQUIRE(rows == 0 || (gy_a && gy_b && x), "grad_w needs grad_out and x");
  // one accumulator for both: one rounding instead of two, and grad_x written once
  if (is_half(dtype) && gx != nullptr && rows > 0 && gemm_tr_dx_fits(gy_a, w_a, gx, E, N, K, rows, true, false) &&
      gemm_tr_dx_fits(gy_b, w_b, gx, E, N, K, rows, true, false)) {
    st = gemm_tr_dx(gy_a, gy_b, w_a, w_b, dtype, wfmt != dtype, E, N, K, offsets, rows, gx, stream);
    if (st) return st;
    gx = nullptr;
  }
  if (is_half(dtype) && gw_a != nullptr && gw_b != nullptr && gemm_tr_dw_fits(gy_a, x, gw_a, E, N, K) &&
      gemm_tr_dw_fits(gy_b, x, gw_b, E, N, K)) {
    st = gemm_tr_dw(gy_a, gy_b, x, dtype, E, N, K, offsets, rows, gw_a, gw_b, gw_dtype == QW_F32, stream);
    if (st) return st;
    gw_a = gw_b = nullptr;
  }
  if (gx != nullptr || gw_a != nullptr)
    st = grouped_matmul_backward(gy_a, x, w_a, dtype, wfmt, E, N, K, offsets, rows, max_rows_per_expert, gx, 0, gw_a,
                                 gw_dtype, ws, ws_bytes, stream);
  if (!st && (gx != nullptr || gw_b != nullptr))
    st = grouped_matmul_backward(gy_b, x, w_b, dtype, wfmt, E, N, K, offsets, rows, max_rows_per_expert, gx, 1, gw_b,
                                 gw_dtype, ws, ws_bytes, stream);
  return st;
}

}  // namespace qw
