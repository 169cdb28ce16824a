// Grouped SwiGLU and grouped matmul over weight-only quantised rows (QW_I8,
// QW_U4; src/quantization.py:61-72) on 16-bit MFMA, for prefill-sized rows per
// expert and for one quantised matrix applied on its own.
//
// What bounds it: an int4 weight costs 3 vector instructions to become bf16
// (convert, fma, half a pair conversion, a share of the nibble split: 24 per 8
// codes), a 16x16x32 MFMA step 16 cycles of the matrix core, so at 64 to 96
// rows per expert the dequantisation weighs as much as the products.  Each
// weight is therefore dequantised once per workgroup: a wave owns 64 weight
// rows for all rows of the chunk (4 waves, 256 weight rows; gate/up: 32 gate
// rows and the matching 32 up rows, so silu(g) * u is formed in registers), its
// codes go straight from global memory to registers, requested one to two K
// slices ahead, and only the activations are staged in LDS (a ring of three
// slices).  In the built loops of most variants the compiler adds a wait for
// everything in flight per two slices (it moves the codes between registers on
// the way back, or takes its own count of the loads), so the lead holds for
// every other slice only.  Two workgroups share a compute unit, so one wave's
// conversions run under another's MFMAs.  Against the 16-bit kernel's layout,
// whose eight waves dequantise every weight twice: int4 layer of 64 rows per
// expert (T 2049, d 4096, f 1408) 571 -> 346 us, int8 (d 2048, f 1024) 213 -> 151
// us; the int4 matrix 2048 x 7168 over 1023 rows 1476 us on the general kernel
// -> 55 us.
// With two slices fetched together (whole 128-byte lines per request) and one
// slice of lead: 375 us for that int4 layer, no gain.
//
// A lane loads 16 bytes of codes per 16-row tile and slice (whole 64-byte row
// pieces per quarter wave), which are not the codes its MFMA operand needs:
// step s takes columns 32 s + 8 q .. + 7 from quarter q (lanes 16 q .. 16 q +
// 15).  The quarters exchange dwords with v_permlane32_swap /
// v_permlane16_swap (one instruction per two dwords), so the operands, and
// the order of every sum, are those of the 16-bit kernel on the dequantised
// weights.  Weights are formed as w = act(q * scale), the fp32 product rounded
// once, exactly the reference's `dequantize().to(dtype)`: the stored value
// u = q + bias (bias 128 after flipping the int8 sign bit, 8 for int4 nibbles)
// is converted to fp32 and fma(u, s, -bias * s) rounds once (bias * s is a
// power-of-two multiple of s, so exact).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "qw_mfma.h"

namespace qw {

namespace {

constexpr int QP_THREADS = 256;
constexpr int QP_NT = 4;     // 16-row weight tiles per wave
constexpr int QP_NB = 256;   // weight rows per workgroup

// Dwords of codes per lane, tile and slice.
template <int WF, int KS>
constexpr int qp_dwords() {
  return WF == QW_I8 ? KS / 16 : KS / 32;
}

__device__ __forceinline__ void swap16(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
__device__ __forceinline__ void swap32(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

// Exchange between the quarters of a wave: a slice's codes as loaded become
// cw[t][s] (int4) or cw[t][2 s], [2 s + 1] (int8), the operand codes of step s;
// its scales (one per lane, tile and slice; one per row: RS) become s4[t][s].
template <int WF, int KS, bool RS, int DW, int STEPS>
__device__ __forceinline__ void exchange(uint32_t (&cw)[QP_NT][DW], const float (&cs)[QP_NT],
                                         float (&s4)[QP_NT][STEPS]) {
  static_assert(STEPS == KS / 32, "MFMA steps of a slice");
#pragma unroll
  for (int t = 0; t < QP_NT; ++t) {
    if constexpr (WF == QW_U4 && KS == 128) {
      swap32(cw[t][0], cw[t][2]);
      swap32(cw[t][1], cw[t][3]);
      swap16(cw[t][0], cw[t][1]);
      swap16(cw[t][2], cw[t][3]);
    } else if constexpr (WF == QW_U4) {
      swap16(cw[t][0], cw[t][1]);
    } else {  // dwords (0, 1) and (2, 3) are the halves of the lane's 16 codes
      swap16(cw[t][0], cw[t][2]);
      swap16(cw[t][1], cw[t][3]);
    }
    if constexpr (RS) {
#pragma unroll
      for (int s = 0; s < STEPS; ++s) s4[t][s] = cs[t];
    } else {
      uint32_t a = __float_as_uint(cs[t]), c = a;
      if constexpr (KS == 128) {
        swap32(a, c);
        uint32_t a2 = a, c2 = c;
        swap16(a, a2);
        swap16(c, c2);
        s4[t][0] = __uint_as_float(a);
        s4[t][1] = __uint_as_float(a2);
        s4[t][2] = __uint_as_float(c);
        s4[t][3] = __uint_as_float(c2);
      } else {
        swap16(a, c);
        s4[t][0] = __uint_as_float(a);
        s4[t][1] = __uint_as_float(c);
      }
    }
  }
}

// Tile t's weight operand of step s: act(q * scale) of 8 columns.
template <int ACT, int WF, int DW>
__device__ __forceinline__ bf16x8 weight_operand(const uint32_t (&c)[DW], int s, float scale) {
  if constexpr (WF == QW_I8) {
    return scale_bytes_seq<ACT>(c[2 * s] ^ 0x80808080u, c[2 * s + 1] ^ 0x80808080u, scale, -128.0f * scale);
  } else {
    const uint32_t r = c[s];
    return scale_bytes<ACT>(r & 0x0f0f0f0fu, (r >> 4) & 0x0f0f0f0fu, scale, -8.0f * scale);
  }
}

// Loads one tile's codes of a slice from p.
template <int DW>
__device__ __forceinline__ void load_codes(const char* p, uint32_t (&r)[DW]) {
  if constexpr (DW == 4) {
    const u32x4 v = *reinterpret_cast<const u32x4*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = v[i];
  } else {
    const u32x2 v = *reinterpret_cast<const u32x2*>(p);
    r[0] = v[0];
    r[1] = v[1];
  }
}

// KS: K columns per slice (128 for int4 rows of whole 128-code pieces, else
// 64).  SUB: 16-row sub-tiles of activations per workgroup.
// RS: one scale per row.
template <int ACT, int WF, bool GATEUP, int SUB, int KS, bool RS>
__global__ __launch_bounds__(QP_THREADS, 2) void ffn_quant_kernel(
    const uint16_t* __restrict__ x, const int32_t* __restrict__ row_index, const int32_t* __restrict__ offsets,
    int max_rows, const MfW wa, const MfW wb, int n_w, int K, const float* __restrict__ row_weight,
    uint16_t* __restrict__ out, int n_out, int n_tiles, int m_chunks, int experts, uint16_t* __restrict__ save_a,
    uint16_t* __restrict__ save_b) {
  constexpr int MCH = 16 * SUB;
  constexpr int ROWB = KS * 2;                 // bytes per LDS row
  constexpr int PIECES = ROWB / 16;            // 16-byte pieces per row (8 or 16)
  constexpr int A_STAGE = MCH * ROWB;
  constexpr int GROWS = 64 / PIECES;           // rows per 1 KiB load group
  constexpr int AL = A_STAGE / 1024 / 4;       // load groups per wave and slice
  constexpr int STEPS = KS / 32;               // MFMA steps per slice
  constexpr int DW = qp_dwords<WF, KS>();      // code dwords per lane, tile and slice
  static_assert(DW == 4 || DW == 2, "16- or 8-byte code loads");
  static_assert(A_STAGE % 4096 == 0, "whole load groups per wave");
  // When the codes of the slice after the next are requested.  At first, over a copy
  // of the present ones, where the registers hold the copy.  With 96 rows (SUB 6)
  // they do so for bf16 int4 only; elsewhere 4 to 46 registers went to scratch, for
  // fp16 inside the loop, so there the codes are multiplied where they lie and
  // requested behind the slice's last conversions (64 rows per expert, fp16: int4 d
  // 4096, f 1408 383 -> 306 us, int8 d 2048, f 1024 156 -> 121; bf16 int8 124 -> 117).
  // Smaller chunks spend less time on a slice and need the longer lead (18 rows,
  // int4: 223 us against 241).
  constexpr bool LATE = SUB >= 6 && (WF == QW_I8 || ACT == QW_F16);
  extern __shared__ __attribute__((aligned(1024))) char smem[];

  // ---- tile: 8 experts or more: expert e's tiles go to XCD e % 8, so its rows
  //      stay in one L2; fewer: the (expert, column tile) pairs are dealt over
  //      the XCDs, row chunks fastest, so a pair's weights are fetched by one
  //      L2. ----
  const int b = blockIdx.x, xcd = b % kXcds, j = b / kXcds;
  int nt, mc = 0, e;
  if (experts >= kXcds) {
    if (m_chunks > 0) {  // an expert's chunks of one column tile together: they share its weights in the L2
      mc = j % m_chunks;
      nt = j / m_chunks % n_tiles;
      e = xcd + kXcds * (j / m_chunks / n_tiles);
      if (e >= experts) return;
    } else {  // a loose bound: the chunks that hold rows are found here, in runs of -m_chunks on one XCD
      nt = j % n_tiles;
      e = find_run_chunk(offsets, experts, max_rows, MCH, -m_chunks, xcd, j / n_tiles, &mc);
      if (e < 0) return;
    }
  } else {
    const int pair = xcd + kXcds * (j / m_chunks);
    mc = j % m_chunks;
    e = pair / n_tiles;
    nt = pair % n_tiles;
    if (e >= experts) return;
  }
  const int e_lo = offsets ? max(offsets[e], 0) : 0;  // no offsets: one expert holds every row
  const int e_hi = offsets ? offsets[e + 1] : max_rows;
  const int r0 = e_lo + mc * MCH;
  const int count = min(min(e_hi, r0 + MCH), max_rows) - r0;
  if (count <= 0) return;

  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const int l16 = lane % 16, lq = lane / 16;
  const int n0 = nt * (GATEUP ? QP_NB / 2 : QP_NB);

  // ---- activation sources: lane i of a group writes LDS row GROWS g + i /
  //      PIECES, physical piece i % PIECES ----
  auto swz = [](int row, int piece) { return piece ^ (PIECES == 16 ? (row & 15) : ((row >> 1) & 7)); };
  const uint16_t* a_src[AL];
#pragma unroll
  for (int q = 0; q < AL; ++q) {
    const int row = GROWS * (wave + 4 * q) + lane / PIECES;
    const int rr = min(row, count - 1);  // rows past the end load a valid row
    const int64_t src = row_index ? row_index[r0 + rr] : (r0 + rr);
    a_src[q] = x + src * K + swz(row, lane % PIECES) * 8;
  }
  // ---- code sources: quarter q loads 16-byte (DW 4) or 8-byte (DW 2) piece
  //      `part` of its row's slice, so that the exchange below leaves each
  //      quarter with its own columns ----
  const int part = (WF == QW_U4 && KS == 128) ? lq : ((lq & 1) << 1 | (lq >> 1));
  const char* b_src[QP_NT];
  const float* s_src[QP_NT];
#pragma unroll
  for (int t = 0; t < QP_NT; ++t) {
    const bool second = GATEUP && t >= QP_NT / 2;
    const MfW& v = second ? wb : wa;
    const int wrow = min(GATEUP ? n0 + 32 * wave + 16 * (t % 2) + l16 : n0 + 64 * wave + 16 * t + l16, n_w - 1);
    b_src[t] = v.w + static_cast<int64_t>(e) * v.expert_bytes + wrow * v.row_bytes + part * (4 * DW);
    s_src[t] = v.scales + static_cast<int64_t>(e) * v.expert_scales + static_cast<int64_t>(wrow) * v.groups;
  }
  const int step32 = KS == 128 ? lq : (lq & 1);  // the MFMA step whose scale this lane loads
  const int group32 = wa.group / 32;             // MFMA steps per scale
  const int KT = K / KS;

  // Codes and scales of the next two slices, requested into registers.
  uint32_t raw[2][QP_NT][DW];
  float sc[2][QP_NT];
  constexpr int BL = QP_NT * (RS ? 1 : 2);  // loads per slice
  auto load_b = [&](int kt, uint32_t (&r)[QP_NT][DW], float (&f)[QP_NT]) {
#pragma unroll
    for (int t = 0; t < QP_NT; ++t) load_codes<DW>(b_src[t] + kt * (16 * DW), r[t]);
    if constexpr (!RS) {
      const int step = kt * STEPS + step32;
      const int idx = group32 == 1 ? step : step / group32;
#pragma unroll
      for (int t = 0; t < QP_NT; ++t) f[t] = s_src[t][idx];
    }
  };
  auto issue_a = [&](int kt, int stage) {
    char* st = smem + stage * A_STAGE;
#pragma unroll
    for (int q = 0; q < AL; ++q)
      __builtin_amdgcn_global_load_lds(static_cast<const void*>(a_src[q] + kt * KS),
                                       (lds_void*)(st + (wave + 4 * q) * 1024), 16, 0, 0);
  };

  f32x4 acc[SUB][QP_NT];
#pragma unroll
  for (int i = 0; i < SUB; ++i)
#pragma unroll
    for (int t = 0; t < QP_NT; ++t) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  float row_sc[QP_NT];
  if constexpr (RS) {
#pragma unroll
    for (int t = 0; t < QP_NT; ++t) row_sc[t] = s_src[t][0];
  }
  issue_a(0, 0);
  load_b(0, raw[0], sc[0]);
  __builtin_amdgcn_sched_barrier(0);
  issue_a(min(1, KT - 1), 1);
  load_b(min(1, KT - 1), raw[1], sc[1]);
  // NA: sub-tiles that hold rows (rounded up to even); the others are loaded
  // with the rest and not multiplied.
  auto k_loop = [&](auto na) {
    constexpr int NA = decltype(na)::value;
    int stage = 0;  // kt % 3
    auto slice = [&](int kt, auto buf) {
      constexpr int BUF = decltype(buf)::value;
      // slice kt has landed (activations in LDS, codes in registers); slice
      // kt + 1 may stay in flight.  Every slice issues the same loads (past the
      // end those of the last one), so the count is fixed.
      wait_vmcnt<AL + BL>();
      ring_barrier();  // visible to every wave, and every wave is done with slice kt - 1
      const int next = min(kt + 2, KT - 1);
      const int nstage = stage == 0 ? 2 : stage - 1;
      issue_a(next, nstage);
      uint32_t copy[QP_NT][DW];
      uint32_t (&cw)[QP_NT][DW] = LATE ? raw[BUF] : copy;
      float cs[QP_NT], s4[QP_NT][STEPS];
#pragma unroll
      for (int t = 0; t < QP_NT; ++t) {
#pragma unroll
        for (int i = 0; i < (LATE ? 0 : DW); ++i) copy[t][i] = raw[BUF][t][i];
        cs[t] = RS ? row_sc[t] : sc[BUF][t];
      }
      if constexpr (!LATE) load_b(next, raw[BUF], sc[BUF]);
      exchange<WF, KS, RS>(cw, cs, s4);
      const char* st = smem + stage * A_STAGE;
      stage = stage == 2 ? 0 : stage + 1;
      auto read_a = [&](int i, int s) {
        const int row = 16 * i + l16;
        return *reinterpret_cast<const bf16x8*>(st + row * ROWB + swz(row, 4 * s + lq) * 16);
      };
#pragma unroll
      for (int s = 0; s < STEPS; ++s) {
        bf16x8 w[QP_NT];
#pragma unroll
        for (int t = 0; t < QP_NT; ++t) w[t] = weight_operand<ACT, WF, DW>(cw[t], s, s4[t][s]);
        if (LATE && s == STEPS - 1) {
          if constexpr (WF == QW_I8) __builtin_amdgcn_sched_barrier(0);
          load_b(next, raw[BUF], sc[BUF]);
          if constexpr (WF == QW_I8 && ACT == QW_F16) __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int i = 0; i < NA; ++i) {
          const bf16x8 xr = read_a(i, s);
#pragma unroll
          for (int t = 0; t < QP_NT; ++t) acc[i][t] = mfma_step<ACT>(w[t], xr, acc[i][t]);
        }
      }
    };
    int kt = 0;
    for (; kt + 1 < KT; kt += 2) {
      slice(kt, std::integral_constant<int, 0>{});
      slice(kt + 1, std::integral_constant<int, 1>{});
    }
    if (kt < KT) slice(kt, std::integral_constant<int, 0>{});
  };
  const int active = (count + 15) / 16;  // uniform over the workgroup
  if (SUB >= 6 && active > 4) k_loop(std::integral_constant<int, SUB>{});
  else if (SUB >= 4 && active > 2) k_loop(std::integral_constant<int, SUB < 4 ? SUB : 4>{});
  else k_loop(std::integral_constant<int, 2>{});
  // The last two slices asked for once too often still write to the stages, which
  // the epilogue reuses and the workgroup's end gives back.
  wait_vmcnt<0>();

  // ---- epilogue: lane holds row l16 of a sub-tile, columns 4 lq .. 4 lq + 3
  //      of each weight tile ----
  constexpr int OC = GATEUP ? QP_NB / 2 : QP_NB;  // output columns of the tile
  if (row_weight == nullptr && save_a == nullptr && n_out % 8 == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0) {
    // through LDS (free after the last slice), whole 16-byte pieces of whole
    // row segments; the tile leaves in passes of the rows the LDS holds
    constexpr int CPR = OC / 8;
    constexpr int FIT = 3 * A_STAGE / (OC * 2);                    // rows that fit the stages
    constexpr int PS = FIT / 16 < SUB ? FIT / 16 : SUB;            // sub-tiles per pass
    static_assert(PS >= 1, "the stages hold a sub-tile of outputs");
    auto chunk_of = [](int row, int col) { return (col / 8) ^ (((row & 15) << 1) & (CPR - 1)); };
#pragma unroll
    for (int p0 = 0; p0 < SUB; p0 += PS) {
      if (p0 >= active) break;
      __syncthreads();
#pragma unroll
      for (int i = p0; i < (p0 + PS < SUB ? p0 + PS : SUB); ++i) {
        if (i >= active) continue;
        const int rl = 16 * (i - p0) + l16;
#pragma unroll
        for (int t = 0; t < (GATEUP ? QP_NT / 2 : QP_NT); ++t) {
          const int col = GATEUP ? 32 * wave + 16 * t + 4 * lq : 64 * wave + 16 * t + 4 * lq;
          uint32_t pk[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            if (GATEUP)
              pk[h] = swiglu_pack2<ACT>(acc[i][t][2 * h], acc[i][t][2 * h + 1], acc[i][t + QP_NT / 2][2 * h],
                                        acc[i][t + QP_NT / 2][2 * h + 1]);
            else
              pk[h] = pack_half2<ACT>(acc[i][t][2 * h], acc[i][t][2 * h + 1]);
          }
          *reinterpret_cast<uint2*>(smem + rl * (OC * 2) + chunk_of(rl, col) * 16 + (col % 8) * 2) =
              make_uint2(pk[0], pk[1]);
        }
      }
      __syncthreads();
      const int rows = min(count - 16 * p0, 16 * PS);
      for (int c = tid; c < rows * CPR; c += QP_THREADS) {
        const int rl = c / CPR, q = c % CPR, col = n0 + q * 8;
        if (col < n_out)
          *reinterpret_cast<uint4*>(out + static_cast<int64_t>(r0 + 16 * p0 + rl) * n_out + col) =
              *reinterpret_cast<const uint4*>(smem + rl * (OC * 2) + chunk_of(rl, q * 8) * 16);
      }
    }
    return;
  }
  // row weights, saved copies or odd widths: direct stores
  const bool vec = n_out % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & 7) == 0;
  auto put = [&](uint16_t* base, int64_t at, int col, const float (&v)[4]) {
    if (vec) {
      *reinterpret_cast<uint2*>(base + at) = make_uint2(pack_half2<ACT>(v[0], v[1]), pack_half2<ACT>(v[2], v[3]));
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (col + u < n_out) base[at + u] = f32_to_half<ACT>(v[u]);
    }
  };
#pragma unroll
  for (int i = 0; i < SUB; ++i) {
    const int row = 16 * i + l16;
    if (row >= count) continue;
    const int64_t orow = static_cast<int64_t>(r0 + row) * n_out;
#pragma unroll
    for (int t = 0; t < (GATEUP ? QP_NT / 2 : QP_NT); ++t) {
      const int col = n0 + (GATEUP ? 32 * wave + 16 * t + 4 * lq : 64 * wave + 16 * t + 4 * lq);
      if (col >= n_out) continue;
      float a[4], c[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        a[u] = acc[i][t][u];
        c[u] = GATEUP ? acc[i][(t + QP_NT / 2) % QP_NT][u] : 0.0f;
      }
      if (GATEUP) {
        const uint32_t lo = swiglu_pack2<ACT>(a[0], a[1], c[0], c[1]);
        const uint32_t hi = swiglu_pack2<ACT>(a[2], a[3], c[2], c[3]);
        if (vec) {
          *reinterpret_cast<uint2*>(out + orow + col) = make_uint2(lo, hi);
        } else {
          const uint32_t w[2] = {lo, hi};
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (col + u < n_out) out[orow + col + u] = static_cast<uint16_t>(w[u / 2] >> (16 * (u % 2)));
        }
        if (save_a) {  // gate and up projections
          put(save_a, orow + col, col, a);
          put(save_b, orow + col, col, c);
        }
      } else {
        if (save_a) put(save_a, orow + col, col, a);  // the rows before their weight
        if (row_weight) {
          const float wgt = row_weight[r0 + row];
#pragma unroll
          for (int u = 0; u < 4; ++u) a[u] = round_act<ACT>(a[u]) * wgt;
        }
        put(out, orow + col, col, a);
      }
    }
  }
}

// A few rows against one quantised matrix: 16 SUB rows by 64 weight rows per
// workgroup, its four waves taking every fourth K slice each, with codes and
// activation operands straight in registers, requested one slice ahead, no LDS ring and no
// barrier in the K loop; the four partial tiles are added in wave order.
// Bound by the latency of a wave's chain of slices: with 256 weight rows per
// workgroup (the kernel above) 2048 x 7168 gives 28 workgroups of 16 or 32
// slices each, 24 to 34 us; here 112 workgroups of 4 or 8 slices per wave, 12
// us, which is the caller's own time per call (225 us on the general kernel).
template <int ACT, int WF, int SUB, int KS, bool RS>
__global__ __launch_bounds__(QP_THREADS, 2) void quant_split_kernel(const uint16_t* __restrict__ x, int rows,
                                                                    const MfW w, int n_w, int K,
                                                                    uint16_t* __restrict__ out, int n_tiles,
                                                                    int chunks) {
  constexpr int STEPS = KS / 32, DW = qp_dwords<WF, KS>();
  constexpr int ROWS = 16 * SUB, COLS = 16 * QP_NT;
  __shared__ __attribute__((aligned(16))) float part[4][ROWS * COLS];
  // the row chunks of a column tile on one XCD: its weights are fetched by one L2
  const int b = blockIdx.x, xcd = b % kXcds, j = b / kXcds;
  const int nt = j / chunks * kXcds + xcd, r0 = j % chunks * ROWS;
  if (nt >= n_tiles) return;
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const int l16 = lane % 16, lq = lane / 16;
  const int n0 = nt * COLS, KT = K / KS;
  const int piece = (WF == QW_U4 && KS == 128) ? lq : ((lq & 1) << 1 | (lq >> 1));
  const char* b_src[QP_NT];
  const float* s_src[QP_NT];
  float row_sc[QP_NT];
#pragma unroll
  for (int t = 0; t < QP_NT; ++t) {
    const int wrow = min(n0 + 16 * t + l16, n_w - 1);
    b_src[t] = w.w + wrow * w.row_bytes + piece * (4 * DW);
    s_src[t] = w.scales + static_cast<int64_t>(wrow) * w.groups;
    row_sc[t] = RS ? s_src[t][0] : 0.0f;
  }
  const uint16_t* a_src[SUB];
#pragma unroll
  for (int i = 0; i < SUB; ++i) a_src[i] = x + static_cast<int64_t>(min(r0 + 16 * i + l16, rows - 1)) * K + 8 * lq;
  const int step32 = KS == 128 ? lq : (lq & 1), group32 = w.group / 32;

  uint32_t raw[2][QP_NT][DW];
  float sc[2][QP_NT];
  bf16x8 xa[2][SUB][STEPS];
  auto load = [&](int kt, auto buf) {
    constexpr int B = decltype(buf)::value;
#pragma unroll
    for (int t = 0; t < QP_NT; ++t) load_codes<DW>(b_src[t] + kt * (16 * DW), raw[B][t]);
    if constexpr (!RS) {
      const int step = kt * STEPS + step32;
      const int idx = group32 == 1 ? step : step / group32;
#pragma unroll
      for (int t = 0; t < QP_NT; ++t) sc[B][t] = s_src[t][idx];
    }
#pragma unroll
    for (int i = 0; i < SUB; ++i)
#pragma unroll
      for (int s = 0; s < STEPS; ++s) xa[B][i][s] = *reinterpret_cast<const bf16x8*>(a_src[i] + kt * KS + 32 * s);
  };
  f32x4 acc[SUB][QP_NT];
#pragma unroll
  for (int i = 0; i < SUB; ++i)
#pragma unroll
    for (int t = 0; t < QP_NT; ++t) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto slice = [&](int kt, auto buf) {
    constexpr int B = decltype(buf)::value;
    load(min(kt + 4, KT - 1), std::integral_constant<int, 1 - B>{});  // past the end: the last slice again, unused
    uint32_t cw[QP_NT][DW];
    float cs[QP_NT], s4[QP_NT][STEPS];
#pragma unroll
    for (int t = 0; t < QP_NT; ++t) {
#pragma unroll
      for (int i = 0; i < DW; ++i) cw[t][i] = raw[B][t][i];
      cs[t] = RS ? row_sc[t] : sc[B][t];
    }
    exchange<WF, KS, RS>(cw, cs, s4);
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
#pragma unroll
      for (int t = 0; t < QP_NT; ++t) {
        const bf16x8 f = weight_operand<ACT, WF, DW>(cw[t], s, s4[t][s]);
#pragma unroll
        for (int i = 0; i < SUB; ++i) acc[i][t] = mfma_step<ACT>(f, xa[B][i][s], acc[i][t]);
      }
  };
  if (wave < KT) {
    load(wave, std::integral_constant<int, 0>{});
    for (int kt = wave; kt < KT; kt += 8) {
      slice(kt, std::integral_constant<int, 0>{});
      if (kt + 4 < KT) slice(kt + 4, std::integral_constant<int, 1>{});
    }
  }
  // a lane holds row l16, columns 4 lq .. + 3 of each tile: 16-byte chunk c of
  // row r at chunk c ^ (r & 15), so the 16 rows of a quarter hit all banks
#pragma unroll
  for (int i = 0; i < SUB; ++i)
#pragma unroll
    for (int t = 0; t < QP_NT; ++t) {
      const int r = 16 * i + l16, c = 4 * t + lq;
      *reinterpret_cast<f32x4*>(&part[wave][r * COLS + 4 * (c ^ l16)]) = acc[i][t];
    }
  __syncthreads();
  const bool vec = n_w % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & 7) == 0;
#pragma unroll
  for (int u = 0; u < ROWS * COLS / 4 / QP_THREADS; ++u) {
    const int at = tid + u * QP_THREADS, r = at / (COLS / 4), c = at % (COLS / 4);
    const int col = n0 + 4 * c, row = r0 + r;
    if (row >= rows || col >= n_w) continue;
    f32x4 v = *reinterpret_cast<const f32x4*>(&part[0][r * COLS + 4 * (c ^ (r & 15))]);
#pragma unroll
    for (int q = 1; q < 4; ++q) v += *reinterpret_cast<const f32x4*>(&part[q][r * COLS + 4 * (c ^ (r & 15))]);
    uint16_t* o = out + static_cast<int64_t>(row) * n_w + col;
    if (vec) {
      *reinterpret_cast<uint2*>(o) = make_uint2(pack_half2<ACT>(v[0], v[1]), pack_half2<ACT>(v[2], v[3]));
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (col + k < n_w) o[k] = f32_to_half<ACT>(v[k]);
    }
  }
}

template <int ACT, int WF, int SUB, int KS, bool RS>
int launch_split(const void* x, int64_t rows, const MfW& w, int64_t n_w, int64_t K, void* out, hipStream_t stream) {
  const int64_t n_tiles = ceil_div(n_w, 16 * QP_NT), chunks = ceil_div(rows, 16 * SUB);
  const int64_t grid = kXcds * ceil_div(n_tiles, kXcds) * chunks;
  if (grid > INT32_MAX) return set_error(QW_ERR_UNSUPPORTED, "quantised matrix grid too large");
  quant_split_kernel<ACT, WF, SUB, KS, RS><<<static_cast<unsigned>(grid), QP_THREADS, 0, stream>>>(
      static_cast<const uint16_t*>(x), static_cast<int>(rows), w, static_cast<int>(n_w), static_cast<int>(K),
      static_cast<uint16_t*>(out), static_cast<int>(n_tiles), static_cast<int>(chunks));
  QW_LAUNCH_CHECK("quant_split_kernel");
  return QW_OK;
}

template <int ACT, int WF>
int split_any(const void* x, int64_t rows, const MfW& w, int64_t n_w, int64_t K, void* out, hipStream_t stream) {
  auto go = [&](auto ks, auto rs) -> int {
    constexpr int KS = decltype(ks)::value;
    constexpr bool RS = decltype(rs)::value;
    return rows <= 16 ? launch_split<ACT, WF, 1, KS, RS>(x, rows, w, n_w, K, out, stream)
                      : launch_split<ACT, WF, 2, KS, RS>(x, rows, w, n_w, K, out, stream);
  };
  using K64 = std::integral_constant<int, 64>;
  if constexpr (WF == QW_U4)
    return K % 128 == 0 ? go(std::integral_constant<int, 128>{}, std::false_type{}) : go(K64{}, std::false_type{});
  else
    return w.groups == 1 ? go(K64{}, std::true_type{}) : go(K64{}, std::false_type{});
}

struct QpArgs {
  const void* x;
  const int32_t* row_index;
  const int32_t* offsets;
  int max_rows;
  MfW wa, wb;
  int n_w, K;
  const float* row_weight;
  void* out;
  int n_out, experts;
  int64_t row_cap, rows;  // the bound on an expert's rows, and what most experts hold
  void *save_a, *save_b;
};

template <int ACT, int WF, bool GATEUP, int SUB, int KS, bool RS>
int launch_t(const QpArgs& a, hipStream_t stream) {
  constexpr int MCH = 16 * SUB;
  const int n_tiles = static_cast<int>(ceil_div(GATEUP ? a.n_w : a.n_out, GATEUP ? QP_NB / 2 : QP_NB));
  int64_t grid;
  int m_chunks;
  if (a.experts >= kXcds) {
    // chunks of one XCD: its experts' slots at the row bound, or those its runs can hold
    const int run = loose_run(a.max_rows, a.experts, MCH);
    const int64_t slots = ceil_div(a.experts, kXcds) * ceil_div(a.row_cap, MCH);
    const int64_t found = loose_chunks(a.max_rows, a.experts, MCH, run);
    // Where the bound allows a chunk that few experts fill, the chunks are found
    // on the device too: as fixed slots, the rare ones started between empty
    // ones and ran into a last round of their own (int4 layer, T = 2500, 79
    // rows per expert, capacity 98, chunks of 96 rows: 566 us against 397).
    const bool tight = ceil_div(a.row_cap, MCH) == ceil_div(a.rows, MCH);
    const bool fixed = tight && slots <= ceil_div(a.max_rows, MCH) + ceil_div(a.experts, kXcds);
    m_chunks = fixed ? static_cast<int>(ceil_div(a.row_cap, MCH)) : -run;
    grid = static_cast<int64_t>(kXcds) * (fixed ? slots : found) * n_tiles;
  } else {
    m_chunks = static_cast<int>(ceil_div(a.row_cap, MCH));
    grid = static_cast<int64_t>(kXcds) * ceil_div(static_cast<int64_t>(a.experts) * n_tiles, kXcds) * m_chunks;
  }
  if (grid > INT32_MAX) return set_error(QW_ERR_UNSUPPORTED, "quantised MFMA grid too large");
  constexpr int LDS = 3 * MCH * KS * 2;
  const hipError_t attr = reserve_lds<ffn_quant_kernel<ACT, WF, GATEUP, SUB, KS, RS>>(LDS);
  if (attr != hipSuccess) return set_error(QW_ERR_HIP, "cannot reserve %d bytes of LDS: %s", LDS, hipGetErrorString(attr));
  ffn_quant_kernel<ACT, WF, GATEUP, SUB, KS, RS><<<static_cast<unsigned>(grid), QP_THREADS, LDS, stream>>>(
      static_cast<const uint16_t*>(a.x), a.row_index, a.offsets, a.max_rows, a.wa, a.wb, a.n_w, a.K, a.row_weight,
      static_cast<uint16_t*>(a.out), a.n_out, n_tiles, m_chunks, a.experts, static_cast<uint16_t*>(a.save_a),
      static_cast<uint16_t*>(a.save_b));
  QW_LAUNCH_CHECK(GATEUP ? "ffn_quant_kernel<gateup>" : "ffn_quant_kernel<down>");
  return QW_OK;
}

template <int ACT, int WF, bool GATEUP>
int launch_sub(int sub, const QpArgs& a, hipStream_t stream) {
  const bool rs = a.wa.groups == 1 && a.wb.groups == 1;
#define QW_QP(S)                                                                                           \
  if (sub == S) {                                                                                          \
    if constexpr (WF == QW_U4) {                                                                           \
      if (a.K % 128 == 0) return launch_t<ACT, WF, GATEUP, S, 128, false>(a, stream);                      \
      return launch_t<ACT, WF, GATEUP, S, 64, false>(a, stream);                                           \
    } else {                                                                                               \
      return rs ? launch_t<ACT, WF, GATEUP, S, 64, true>(a, stream)                                        \
                : launch_t<ACT, WF, GATEUP, S, 64, false>(a, stream);                                      \
    }                                                                                                      \
  }
  QW_QP(2)
  QW_QP(4)
  QW_QP(6)
#undef QW_QP
  return set_error(QW_ERR_UNSUPPORTED, "no quantised MFMA variant for %d sub-tiles", sub);
}

template <bool GATEUP>
int launch_any(int act, int wfmt, int sub, const QpArgs& a, hipStream_t stream) {
  if (act == QW_F16)
    return wfmt == QW_I8 ? launch_sub<QW_F16, QW_I8, GATEUP>(sub, a, stream)
                         : launch_sub<QW_F16, QW_U4, GATEUP>(sub, a, stream);
  return wfmt == QW_I8 ? launch_sub<QW_BF16, QW_I8, GATEUP>(sub, a, stream)
                       : launch_sub<QW_BF16, QW_U4, GATEUP>(sub, a, stream);
}

// 16-row sub-tiles per workgroup for experts of `rows` rows: the fewest chunks
// of at most 96 rows (what the registers hold beside the codes in flight),
// evenly filled.
int pick_sub(int64_t rows) {
  const int64_t chunks = std::max<int64_t>(1, ceil_div(rows, 96));
  for (int s : {2, 4, 6})
    if (16 * s * chunks >= rows) return s;
  return 6;
}

}  // namespace

int launch_ffn_quant(const FfnArgs& a, hipStream_t stream, bool* handled) {
  *handled = false;
  if (!is_half(a.act) || (a.wfmt != QW_I8 && a.wfmt != QW_U4) || !rows_on_16_bytes(a)) return QW_OK;
  if (!quant_fits(a.gate, a.wfmt) || !quant_fits(a.up, a.wfmt) || !quant_fits(a.down, a.wfmt)) return QW_OK;
  const int64_t cap = a.row_cap > 0 ? a.row_cap : a.max_rows;
  const int64_t rows = likely_rows(a, 2.0);
  const int sub = pick_sub(rows);
  const int D = static_cast<int>(a.d_model), F = static_cast<int>(a.d_ff), E = static_cast<int>(a.experts);
  const MfW g = mf_view(a.wfmt, a.gate), u = mf_view(a.wfmt, a.up), d = mf_view(a.wfmt, a.down);
  QpArgs q{a.x, a.row_index, a.offsets, static_cast<int>(a.max_rows), g, u, F, D, nullptr, a.hidden, F, E, cap, rows,
           a.save_gate, a.save_up};
  int st = launch_any<true>(a.act, a.wfmt, sub, q, stream);
  if (st) return st;
  q = QpArgs{a.hidden, nullptr, a.offsets, static_cast<int>(a.max_rows), d, d, D, F, a.row_weight, a.y, D, E, cap, rows,
             a.save_y, nullptr};
  st = launch_any<false>(a.act, a.wfmt, sub, q, stream);
  if (st) return st;
  *handled = true;
  return QW_OK;
}

int quant_matmul(const void* x, int act, const WView& w, int wfmt, int64_t E, const int32_t* offsets, int64_t rows,
                 int64_t row_cap, void* out, hipStream_t stream, bool* handled) {
  *handled = false;
  if (!is_half(act) || !quant_fits(w, wfmt) || reinterpret_cast<uintptr_t>(x) % 16 != 0) return QW_OK;
  // One matrix: the split kernel until its grid is 3.5 workgroups per compute
  // unit, from where its weights are dequantised too often (int4 2048 x 7168,
  // split against not: 12 / 34 us at 64 rows, 20 / 35 at 128, 37 / 35 at 256 =
  // 896 workgroups; 4096 x 1408: 49 / 65 us at 1023 = 704, 97 / 67 at 2048).
  if (offsets == nullptr && ceil_div(w.rows, 16 * QP_NT) * ceil_div(rows, rows <= 16 ? 16 : 32) <= 896) {
    const MfW m = mf_view(wfmt, w);
    const int st = act == QW_F16 ? (wfmt == QW_I8 ? split_any<QW_F16, QW_I8>(x, rows, m, w.rows, w.cols, out, stream)
                                                  : split_any<QW_F16, QW_U4>(x, rows, m, w.rows, w.cols, out, stream))
                                 : (wfmt == QW_I8 ? split_any<QW_BF16, QW_I8>(x, rows, m, w.rows, w.cols, out, stream)
                                                  : split_any<QW_BF16, QW_U4>(x, rows, m, w.rows, w.cols, out, stream));
    if (st == QW_OK) *handled = true;
    return st;
  }
  int sub = pick_sub(E > 1 ? std::min(row_cap, 2 * ceil_div(rows, E)) : rows);
  // a few matrices leave compute units idle in large chunks: smaller ones
  // while there are fewer than two workgroups per unit
  while (sub > 4 && E * ceil_div(w.rows, QP_NB) * ceil_div(row_cap, 16 * sub) < 512) sub -= 2;
  const MfW v = mf_view(wfmt, w);
  const QpArgs q{x, nullptr, offsets, static_cast<int>(rows), v, v, static_cast<int>(w.rows),
                 static_cast<int>(w.cols), nullptr, out, static_cast<int>(w.rows), static_cast<int>(E), row_cap,
                 row_cap, nullptr, nullptr};
  const int st = launch_any<false>(act, wfmt, sub, q, stream);
  if (st) return st;
  *handled = true;
  return QW_OK;
}

}  // namespace qw
