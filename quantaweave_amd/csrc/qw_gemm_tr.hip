// Grouped 16-bit GEMMs whose operands lie reduction-major in memory, for the
// backward of the grouped matmul y[rows of e] = x[rows of e] . W[e]^T
// (src/moe_kernels.py:66-89, :118-135, :146-164):
//
//   MODE rows:  dX[r, k]    = sum_n dY[r, n] W[e][n, k]   A = dY rows, B = W[e] as stored
//   MODE red:   dW[e][n, k] = sum_r dY[r, n] x[r, k]      A = dY, B = x, both row-major
//
// Two products that share an operand go as one launch (the gate and up
// projections of a SwiGLU expert): rows sums both in one accumulator, red
// doubles the tiles.
//
// What bounds it: the matrix cores and the LDS together.  A 256 x 256 tile
// takes 2048 clocks of MFMA per 64-deep slice and moves 192 KiB of fragments
// and 64 KiB of staging through the LDS (about 2000 clocks at 128 B).  The
// 128 x 128 tiles of gemm_nt_kernel move half as much again, and its operands
// went through registers (B) or two transposed, padded copies in memory (dW).
// Here operands go straight to LDS (global_load_lds) as they lie, and
// ds_read_b64_tr_b16 transposes them on the way into the registers: the 16
// lanes of a group read 4 reduction rows of 16 columns and each gets one
// column, so two reads make the 8 reduction values of a lane.
//
// Workgroup: 8 waves (2 x 4), 32 SM rows x 256 columns, each wave SM
// 16-row sub-tiles (wm, wm + 2, ...) x 64 columns.  A reduction-major slice is
// 64 rows of 2 x tile bytes; the 32-byte column group s of row r sits at
// s ^ ((r & 3) | (r >> 3 & 1) << 2), so the 8 rows that 32 lanes read at once
// fall into 8 different bank groups.  Rows of the last slice past the
// expert's end come from a zero block; columns past the matrix read its last
// 8 (never stored).
#include <type_traits>

#include "qw_mfma.h"

namespace qw {

namespace {

constexpr int TR_THREADS = 512, TR_WAVES = 8;
constexpr int TR_N = 256;   // columns per tile
constexpr int TR_K = 64;    // reduction slice
constexpr int TR_LDS = 160 * 1024;
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

__device__ const uint4 g_tr_zero = {0u, 0u, 0u, 0u};  // rows past an expert's end

struct TrArgs {
  const uint16_t *a0, *a1, *b0, *b1;  // the second pair only where parts == 2
  void *c0, *c1;
  const int32_t* offsets;
  int64_t b_stride, c_stride;  // elements per expert
  int lda, ldb, ldc;
  int rows, m, n, k, experts, parts;  // m: rows of an output matrix (red); k: reduction per part (rows)
};

template <int SM>
constexpr int tr_stages() {
  return 3 * (32 * SM + TR_N) * TR_K * 2 <= TR_LDS ? 3 : 2;
}

// Column group permutation of reduction row r.
__device__ __forceinline__ int tr_swz(int r) { return (r & 3) | (((r >> 3) & 1) << 2); }

// One transposing read.  The restrict argument is what gives the read alias
// information once inlined: without any, the compiler takes it to touch the
// slices still in flight and waits for them before every read.
__device__ __forceinline__ s16x4 tr_read(const lds_s16x4* __restrict__ at) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(const_cast<lds_s16x4*>(at));
}

template <int DT, int SM, bool RED, bool BT, bool C32>
__global__ __launch_bounds__(TR_THREADS) void gemm_tr_kernel(const TrArgs p) {
  constexpr int TM = 32 * SM, NP = SM / 2, NT = 4;
  constexpr int A_STAGE = TM * TR_K * 2, B_STAGE = TR_N * TR_K * 2;
  constexpr int AL = A_STAGE / 1024 / TR_WAVES, BL = B_STAGE / 1024 / TR_WAVES;
  constexpr int ST = tr_stages<SM>(), AHEAD = ST - 1;
  constexpr int A_ROWB = RED ? TM * 2 : TR_K * 2, A_LPR = A_ROWB / 16, A_RPG = 64 / A_LPR;
  constexpr int B_ROWB = TR_N * 2, B_LPR = B_ROWB / 16, B_RPG = 64 / B_LPR;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  char* const a_ring = smem;
  char* const b_ring = smem + ST * A_STAGE;

  // ---- tile.  rows: XCD x takes row tiles x, x + 8, ... with all their column
  //      tiles; red: every expert's tiles are split over the XCDs (experts'
  //      rows differ, so whole experts would leave XCDs idle), each a run of
  //      tiles that share dY columns. ----
  const int blk = blockIdx.x, xcd = blk % kXcds, j = blk / kXcds;
  const int n_nt = (p.n + TR_N - 1) / TR_N;
  int e, nt, m0, mcount, len, KT, which = 0;
  int64_t row0;
  if constexpr (!RED) {
    int local = 0;
    nt = j % n_nt;
    e = find_tile(p.offsets, p.experts, p.rows, TM, (j / n_nt) * kXcds + xcd, &local);
    if (e < 0) return;
    const int lo = min(max(p.offsets[e], 0), p.rows), hi = min(p.offsets[e + 1], p.rows);
    row0 = lo + local * TM;
    m0 = 0;
    mcount = min(TM, hi - static_cast<int>(row0));
    if (mcount <= 0) return;
    len = p.k;
    KT = p.parts * (p.k / TR_K);
  } else {
    const int tiles = ((p.m + TM - 1) / TM) * n_nt, share = (tiles + kXcds - 1) / kXcds;
    const int t = xcd * share + j % share, q = j / share;
    which = q % p.parts;
    e = q / p.parts;
    if (t >= tiles || e >= p.experts) return;
    nt = t % n_nt;
    m0 = (t / n_nt) * TM;
    mcount = min(TM, p.m - m0);
    const int lo = min(max(p.offsets[e], 0), p.rows), hi = min(p.offsets[e + 1], p.rows);
    row0 = lo;
    len = max(hi - lo, 0);
    KT = (len + TR_K - 1) / TR_K;
  }
  const int n0 = nt * TR_N;
  const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int wm = wave / 4, wn = wave % 4, l16 = lane % 16, lq = lane / 16;

  // ---- per-lane byte offsets of this wave's 1 KiB load groups from the slice's first row ----
  uint32_t a_off[AL], b_off[BL];
#pragma unroll
  for (int q = 0; q < AL; ++q) {
    const int r = A_RPG * (wave + q * TR_WAVES) + lane / A_LPR, piece = lane % A_LPR;
    if constexpr (RED)
      a_off[q] = 2u * (static_cast<uint32_t>(r) * p.lda + min(m0 + 8 * (piece ^ (tr_swz(r) << 1)), p.m - 8));
    else
      a_off[q] = 2u * (static_cast<uint32_t>(min(r, mcount - 1)) * p.lda + 8 * (piece ^ ((r >> 1) & 7)));
  }
#pragma unroll
  for (int q = 0; q < BL; ++q) {
    const int r = B_RPG * (wave + q * TR_WAVES) + lane / B_LPR, piece = lane % B_LPR;
    const int c = min(n0 + 8 * (piece ^ (tr_swz(r) << 1)), p.n - 8);
    if constexpr (BT)  // 8 x 64 tiles of 1 KiB, 16-byte pieces XORed by the row
      b_off[q] = 2u * ((static_cast<uint32_t>(r / 8) * (p.n / 64) + c / 64) * 512u + (r % 8) * 64 +
                       8 * ((c / 8 % 8) ^ ((r >> 1) & 7)));
    else
      b_off[q] = 2u * (static_cast<uint32_t>(r) * p.ldb + c);
  }
  const int kt_part = RED ? INT32_MAX : p.k / TR_K;  // slices of the first part
  const char* const a_first = reinterpret_cast<const char*>((which ? p.a1 : p.a0) + row0 * p.lda);
  const char* const a_second = RED ? nullptr : reinterpret_cast<const char*>(p.a1 + row0 * p.lda);
  const int64_t b_base = RED ? row0 * p.ldb : e * p.b_stride;
  const char* const b_first = reinterpret_cast<const char*>((which ? p.b1 : p.b0) + b_base);
  const char* const b_second = RED ? nullptr : reinterpret_cast<const char*>(p.b1 + b_base);
  const int64_t a_step = RED ? int64_t{2} * TR_K * p.lda : 2 * TR_K, b_step = int64_t{2} * TR_K * p.ldb;
  auto issue = [&](int kt) {
    const bool second = kt >= kt_part;
    const int ks = second ? kt - kt_part : kt;
    const char* as = (second ? a_second : a_first) + ks * a_step;
    const char* bs = (second ? b_second : b_first) + ks * b_step;
    char* const sa = a_ring + (kt % ST) * A_STAGE;
    char* const sb = b_ring + (kt % ST) * B_STAGE;
    const int valid = len - kt * TR_K;  // rows of the slice that exist (red)
    if (RED && valid < TR_K) {
      const char* zero = reinterpret_cast<const char*>(&g_tr_zero);
#pragma unroll
      for (int q = 0; q < AL; ++q) {
        const int g = wave + q * TR_WAVES;
        const char* src = A_RPG * g + lane / A_LPR < valid ? as + a_off[q] : zero;
        __builtin_amdgcn_global_load_lds(static_cast<const void*>(src), (lds_void*)(sa + g * 1024), 16, 0, 0);
      }
#pragma unroll
      for (int q = 0; q < BL; ++q) {
        const int g = wave + q * TR_WAVES;
        const char* src = B_RPG * g + lane / B_LPR < valid ? bs + b_off[q] : zero;
        __builtin_amdgcn_global_load_lds(static_cast<const void*>(src), (lds_void*)(sb + g * 1024), 16, 0, 0);
      }
    } else {
#pragma unroll
      for (int q = 0; q < AL; ++q)
        __builtin_amdgcn_global_load_lds(static_cast<const void*>(as + a_off[q]),
                                         (lds_void*)(sa + (wave + q * TR_WAVES) * 1024), 16, 0, 0);
#pragma unroll
      for (int q = 0; q < BL; ++q)
        __builtin_amdgcn_global_load_lds(static_cast<const void*>(bs + b_off[q]),
                                         (lds_void*)(sb + (wave + q * TR_WAVES) * 1024), 16, 0, 0);
    }
  };

  f32x4 acc[SM][NT];
#pragma unroll
  for (int i = 0; i < SM; ++i)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  // fragment addresses: reduction row 8 lq + l16 / 4 (+ 4 h + 32 ks), 4 columns at 4 (l16 % 4)
  const int fr = 8 * lq + l16 / 4, fs = tr_swz(fr), fc = 8 * (l16 % 4);
  auto read_tr = [&](const char* st, int rowb, int slot, int ks) -> bf16x8 {
    const char* at = st + fr * rowb + ((slot ^ fs) * 32 + fc) + 32 * ks * rowb;
    union {
      s16x4 h[2];
      bf16x8 v;
    } u;
    u.h[0] = tr_read((const lds_s16x4*)(at));
    u.h[1] = tr_read((const lds_s16x4*)(at + 4 * rowb));
    return u.v;
  };
  constexpr int AR = RED ? 2 : 1;  // LDS reads per A fragment (B: 2)
  static_assert(AHEAD >= 1 && AHEAD <= 2 && 2 * (AL + BL) < 64, "ring depth");

  for (int i = 0; i < AHEAD && i < KT; ++i) issue(i);
  // The ring and the order of the fragment reads behind the MFMAs are those of
  // ffn_mfma_kernel: wait for slice kt, barrier, first fragments, request slice
  // kt + AHEAD into the stage of slice kt - 1, multiply.
  auto k_loop = [&](auto npa) {
    constexpr int NPA = decltype(npa)::value;
    for (int kt = 0; kt < KT; ++kt) {
      if (AHEAD == 2 && kt + 1 < KT) wait_vmcnt<AL + BL>();
      else wait_vmcnt<0>();
      ring_barrier();
      const char* st_a = a_ring + (kt % ST) * A_STAGE;
      const char* st_b = b_ring + (kt % ST) * B_STAGE;
      auto read_a = [&](int i, int ks) -> bf16x8 {
        if constexpr (RED) {
          return read_tr(st_a, A_ROWB, wm + 2 * i, ks);
        } else {
          const int row = (wm + 2 * i) * 16 + l16;
          return *reinterpret_cast<const bf16x8*>(st_a + row * A_ROWB + (((lq + 4 * ks) ^ ((row >> 1) & 7)) * 16));
        }
      };
      auto read_b = [&](int t, int ks) -> bf16x8 { return read_tr(st_b, B_ROWB, wn * 4 + t, ks); };
      bf16x8 wfr[2][NT], xb[2][2];
#pragma unroll
      for (int t = 0; t < NT; ++t) wfr[0][t] = read_b(t, 0);
      xb[0][0] = read_a(0, 0);
      xb[0][1] = read_a(1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2 * NT + 2 * AR, 0);
      if (kt + AHEAD < KT) issue(kt + AHEAD);
#pragma unroll
      for (int u = 0; u < 2 * NPA; ++u) {
        const int ks = u / NPA, pr = u % NPA;
        const bf16x8 x0 = xb[u & 1][0], x1 = xb[u & 1][1];
        acc[2 * pr][0] = mfma_step<DT>(wfr[ks][0], x0, acc[2 * pr][0]);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (u + 1 < 2 * NPA) {
          const int ks1 = (u + 1) / NPA, p1 = (u + 1) % NPA;
          if (ks1 != ks) {
#pragma unroll
            for (int t = 0; t < NT; ++t) wfr[1][t] = read_b(t, 1);
          }
          xb[(u + 1) & 1][0] = read_a(2 * p1, ks1);
          xb[(u + 1) & 1][1] = read_a(2 * p1 + 1, ks1);
          if (ks1 != ks) __builtin_amdgcn_sched_group_barrier(0x100, 2 * NT + 2 * AR, 0);
          else __builtin_amdgcn_sched_group_barrier(0x100, 2 * AR, 0);
        }
#pragma unroll
        for (int t = 1; t < NT; ++t) acc[2 * pr][t] = mfma_step<DT>(wfr[ks][t], x0, acc[2 * pr][t]);
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[2 * pr + 1][t] = mfma_step<DT>(wfr[ks][t], x1, acc[2 * pr + 1][t]);
        __builtin_amdgcn_sched_group_barrier(0x008, 2 * NT - 1, 0);
      }
    }
  };
  // pairs of sub-tiles wholly past the tile's rows are not multiplied
  const int active = (mcount + 15) / 16;
  const int npa = __builtin_amdgcn_readfirstlane(((active > wm ? (active - wm + 1) / 2 : 0) + 1) / 2);
  if (npa >= NP) k_loop(std::integral_constant<int, NP>{});
  else if (NP == 4 && npa == 3) k_loop(std::integral_constant<int, NP == 4 ? 3 : 1>{});
  else if (NP == 4 && npa == 2) k_loop(std::integral_constant<int, NP == 4 ? 2 : 1>{});
  else k_loop(std::integral_constant<int, 1>{});

  // ---- lane holds row l16 of sub-tile (wm + 2 i), columns 4 lq .. 4 lq + 3 of each 16-column tile ----
  const int64_t c_row0 = RED ? m0 : row0;
  char* const c = static_cast<char*>(which ? p.c1 : p.c0) + (RED ? e * p.c_stride : 0) * (C32 ? 4 : 2);
#pragma unroll
  for (int i = 0; i < SM; ++i) {
    const int m = (wm + 2 * i) * 16 + l16;
    if (m >= mcount) continue;
    const int64_t row = (c_row0 + m) * p.ldc + n0;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int n = wn * 64 + 16 * t + 4 * lq;
      if (n0 + n >= p.n) continue;
      const f32x4 v = acc[i][t];
      if constexpr (C32)
        *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(c) + row + n) = v;
      else
        *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(c) + row + n) =
            make_uint2(pack_half2<DT>(v[0], v[1]), pack_half2<DT>(v[2], v[3]));
    }
  }
}

template <int DT, int SM, bool RED, bool BT, bool C32>
int launch_tr(const TrArgs& a, int64_t blocks, hipStream_t stream) {
  constexpr int lds = tr_stages<SM>() * (32 * SM + TR_N) * TR_K * 2;
  const hipError_t attr = reserve_lds<gemm_tr_kernel<DT, SM, RED, BT, C32>>(lds);
  if (attr != hipSuccess) return set_error(QW_ERR_HIP, "cannot reserve LDS: %s", hipGetErrorString(attr));
  gemm_tr_kernel<DT, SM, RED, BT, C32><<<static_cast<unsigned>(blocks), TR_THREADS, lds, stream>>>(a);
  QW_LAUNCH_CHECK("gemm_tr_kernel");
  return QW_OK;
}

// 256-row tiles where they come near filling the compute units once (`tiles`, one
// workgroup each), else 128-row ones.  Measured on 2048 x 1024 to 256 x 512
// matrices of 8 to 32 experts, 4000 and 16000 rows: 216 tiles dX 36.7 us against
// 46.2 (128 rows), 282 tiles 48.6 against 70.9, 512 tiles dW 75 against 113;
// 189 tiles dX 34.8 against 28.6, 64 tiles dW 56 against 39.
bool tall_tiles(double tiles) { return tiles >= 200; }

// Row tiles of all experts at `height` rows: on average half a tile per expert is a remainder.
double row_tiles(int64_t rows, int64_t E, int height) { return static_cast<double>(rows) / height + 0.5 * E; }

bool aligned(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace

// dX of one product, or of two summed (gy1, w1 non-null): N columns of gy are the
// reduction.  tiles128: gemm_nt_kernel would take the product otherwise.
bool gemm_tr_dx_fits(const void* gy, const void* w, const void* gx, int64_t E, int64_t N, int64_t K, int64_t rows,
                     bool pair, bool tiles128) {
  // One product: 128 x 128 tiles (gemm_nt_kernel) are level or faster where 256-row
  // tiles do not fill the chip (1024 x 2048, 16 experts, 4000 rows: 28.0 us against
  // 28.6; 512 x 256, 16000 rows: 14.4 against 15.7), except below 96 rows an
  // expert, where whole sub-tiles are skipped (1000 rows: 16.2 us against 19.6).
  // They need a workspace; without one the product would go to the vector-ALU kernel
  // (1024 x 512, 8 experts, 4000 rows: 174 us, 21 here).
  // Two products would be two such launches and a second pass over grad_x
  // (2816 x 1024, 8 experts, 5003 rows: the step of 669 us takes 30 more).
  if (!pair && tiles128 && !tall_tiles(row_tiles(rows, E, 256) * ceil_div(K, TR_N)) && rows >= 96 * E) return false;
  return N % TR_K == 0 && K % 8 == 0 && K >= 192 && N <= (1 << 22) && K <= (1 << 22) &&
         (ceil_div(rows, 128) + E + kXcds) * ceil_div(K, TR_N) <= INT32_MAX / 8 && aligned(gy) && aligned(w) &&
         aligned(gx);
}

int gemm_tr_dx(const void* gy0, const void* gy1, const void* w0, const void* w1, int dtype, bool tiled, int64_t E,
               int64_t N, int64_t K, const int32_t* offsets, int64_t rows, void* gx, hipStream_t stream) {
  TrArgs a{};
  a.a0 = static_cast<const uint16_t*>(gy0);
  a.a1 = static_cast<const uint16_t*>(gy1 ? gy1 : gy0);
  a.b0 = static_cast<const uint16_t*>(w0);
  a.b1 = static_cast<const uint16_t*>(w1 ? w1 : w0);
  a.c0 = a.c1 = gx;
  a.offsets = offsets;
  a.b_stride = N * K;
  a.lda = static_cast<int>(N);
  a.ldb = a.ldc = a.n = static_cast<int>(K);
  a.rows = static_cast<int>(rows);
  a.k = static_cast<int>(N);
  a.experts = static_cast<int>(E);
  a.parts = gy1 ? 2 : 1;
  const int64_t nt = ceil_div(K, TR_N);
  const bool tall = tall_tiles(row_tiles(rows, E, 256) * nt);
  const int64_t blocks = kXcds * nt * ceil_div(ceil_div(rows, tall ? 256 : 128) + E, kXcds);
  auto go = [&](auto dt, auto bt) {
    return tall ? launch_tr<decltype(dt)::value, 8, false, decltype(bt)::value, false>(a, blocks, stream)
                : launch_tr<decltype(dt)::value, 4, false, decltype(bt)::value, false>(a, blocks, stream);
  };
  using H = std::integral_constant<int, QW_F16>;
  using B = std::integral_constant<int, QW_BF16>;
  if (dtype == QW_F16) return tiled ? go(H{}, std::true_type{}) : go(H{}, std::false_type{});
  return tiled ? go(B{}, std::true_type{}) : go(B{}, std::false_type{});
}

// dW of one product, or of two with the same x (gy1, gw1 non-null).
bool gemm_tr_dw_fits(const void* gy, const void* x, const void* gw, int64_t E, int64_t N, int64_t K) {
  return N % 8 == 0 && K % 8 == 0 && N >= 96 && K >= 192 && N <= (1 << 22) && K <= (1 << 22) &&
         2 * E * (ceil_div(N, 128) * ceil_div(K, TR_N) + kXcds) <= INT32_MAX && aligned(gy) && aligned(x) && aligned(gw);
}

int gemm_tr_dw(const void* gy0, const void* gy1, const void* x, int dtype, int64_t E, int64_t N, int64_t K,
               const int32_t* offsets, int64_t rows, void* gw0, void* gw1, int gw_f32, hipStream_t stream) {
  TrArgs a{};
  a.a0 = static_cast<const uint16_t*>(gy0);
  a.a1 = static_cast<const uint16_t*>(gy1 ? gy1 : gy0);
  a.b0 = a.b1 = static_cast<const uint16_t*>(x);
  a.c0 = gw0;
  a.c1 = gw1;
  a.offsets = offsets;
  a.c_stride = N * K;
  a.lda = a.m = static_cast<int>(N);
  a.ldb = a.ldc = a.n = static_cast<int>(K);
  a.rows = static_cast<int>(rows);
  a.experts = static_cast<int>(E);
  a.parts = gy1 ? 2 : 1;
  const int64_t nt = ceil_div(K, TR_N), per = a.parts * E;
  const bool tall = tall_tiles(static_cast<double>(per * nt * ceil_div(N, 256)));
  const int64_t blocks = kXcds * per * ceil_div(nt * ceil_div(N, tall ? 256 : 128), kXcds);
  auto go = [&](auto dt, auto c32) {
    return tall ? launch_tr<decltype(dt)::value, 8, true, false, decltype(c32)::value>(a, blocks, stream)
                : launch_tr<decltype(dt)::value, 4, true, false, decltype(c32)::value>(a, blocks, stream);
  };
  using H = std::integral_constant<int, QW_F16>;
  using B = std::integral_constant<int, QW_BF16>;
  if (dtype == QW_F16) return gw_f32 ? go(H{}, std::true_type{}) : go(H{}, std::false_type{});
  return gw_f32 ? go(B{}, std::true_type{}) : go(B{}, std::false_type{});
}

}  // namespace qw
