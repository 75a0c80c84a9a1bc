// Linear layers over many rows (prefill steps, mixed steps, the LM head of large batches):
//
//   y = epilogue( x W^T + b )      x [M, K], W [N, K] (nn.Linear layout), fp32 in, fp32 out
//
// as fp32 products on the bf16 matrix cores. Every fp32 operand is the exact sum of three
// bf16 numbers (8 + 8 + 8 significant bits: each the rounded rest of the ones before), and
//
//   x w = x0 w0 + (x0 w1 + x1 w0) + (x0 w2 + x1 w1 + x2 w0) + terms below 2^-24 |x w|
//
// so six bf16 products, accumulated in fp32 by the MFMA, give the product to fp32's own
// precision; the sum is a little more exact for taking 16 k per accumulation instead of 4: against
// float64, weights N(0, 0.02), rows N(0, 1): 4.2e-7 (K = 768) and 8.6e-7 (K = 3072; 3.1e-7 to 4.3e-7 in
// parts of K) relative where the fp32 MFMA GEMM of the library has 5.0e-7 and 9.9e-7. The fp32 MFMA peaks at 157
// TFLOP/s on this GPU; bf16 runs ~1,200 (what a large library product reaches here, power
// bound), a sixth of which is 200. The split costs no extra traffic: operands are read as
// fp32 and split on the way in, nothing is kept between calls.
//
// Infinities, NaN and overflow: the split of a non-finite number (or of one that rounds past
// the largest bf16) is NaN, so every output it touches comes out non-finite. Outputs whose
// accumulator is not finite are computed again with plain fp32 FMAs, which give them IEEE's
// value: the wave's lanes share one output's K (row_dot).
//
// Operands below 2^-110 lose bits to the limbs' smallest exponent (split_bf16.h): up to K 2^-133 times the largest
// operand of an output's row and column, which is below 2^-22 of an output of K 2^-111 times it. A wave
// whose accumulators are all between K 2^-79 and 2^32 in size stops there (operands above 2^32 show in some output of
// the tile unless all they meet is as tiny). Another one looks through the rows and columns of its tile for such
// operands and the largest ones, and computes the outputs below that bound again too: rows of 1e-36, say,
// which the limbs alone give to 5e-5. All other outputs keep their bits. What it costs ordinary inputs
// (us, without -> with): [256, 768, 3072] 18.2 -> 18.9, [1987, 2304, 768] 45.2 -> 46.0, the other sizes measured within
// 1 %; keeping the largest operands in the main loop instead took 2-8 %.
//
// Work split: a workgroup of WM waves covers 32 WM rows x 32 NB columns; wave w owns rows
// 32 w .. 32 w + 31 and all the columns, as NB accumulators of v_mfma_f32_32x32x16_bf16 (A = W,
// B = X^T: lane (i, g) = (lane % 32, lane / 32) supplies row i, k octet g of a 16-wide k half).
// Each wave reads and splits its own X rows straight into registers; W is read, split and
// written to LDS once per workgroup, double buffered, one barrier per 32 of K.
//  * 32x32x16 rather than 16x16x32: the split's VALU work (about four instructions per MFMA)
//    hides behind it, while beside 16x16x32 it adds to the MFMA time (two waves a SIMD, 4 subs
//    and 2 conversions per 32 cycles of MFMA: 35 cycles against 47).
//  * X in registers: LDS is the next bound (reads 128 B, writes 64 B a clock and CU; three
//    limbs are 6 B an element). With X in LDS too a 128 x 128 tile took 1.06 us per 32 of K,
//    0.63 us of it LDS; this way 1.00 us. A wave's X loads have one row per lane, which the
//    address unit takes at 16 B a clock; W's, four lanes a row, at 54, and W staged one row
//    per lane cost 5-6 us of a 29 us tile.
//  * W's fragments sit in LDS in the order the MFMA reads them, rows swizzled by the k octet, so that
//    consecutive lanes meet in no bank. Counters: 17-25 % of the LDS cycles are conflicts all the same (the
//    hardware takes a 16-byte access's lanes in other groups), with the LDS busy for 19-28 % of the time.
//  * A step's loads are issued two steps before they are split (one where the registers allow no
//    more): weights come from HBM in a model's step, and one step is shorter than their latency.
// Outputs of fewer than 160 tiles of 128 x 64 are computed in parts of K, a workgroup per tile and
// part, and summed in order (with bias and epilogue) by a second launch: no tile waits for another
// workgroup, and the partial sums live in the caller's workspace.
// Measured (GPU time, MI355X, weights evicted between calls) against the library's fp32 GEMM: 1,987
// rows, [N, K] = [2304, 768] / [3072, 768] / [768, 3072] / [768, 768]: 76 / 78 / 86 / 27 -> 45 / 51 /
// 67 / 20 us; 8,192 rows (operands resident): 221 / 280 / 266 / 85 -> 154 / 191 / 181 / 54 us (188-213
// TFLOP/s of fp32 products, 1,130-1,280 of bf16 ones; MFMA busy for 68 % of the cycles at 1.85 GHz: power bound). At
// 1,987 rows the MFMAs are busy for 38-47 %: one tile a CU, on 192-216 of 256 CUs.
//
// Reference semantics: nn.Linear (tokquay/model.py:62-63, :103-104), the tanh GELU (:107), the
// tied LM head (:180-181).

#include <float.h>

#include <type_traits>

#include "split_bf16.h"
#include "tq_internal.h"

namespace tq {
namespace {

constexpr int kStep = 32;              // k per pipeline step
constexpr int kXcds = 8;               // workgroup i is dispatched to XCD i % 8
constexpr int kBufferWord3 = 0x00020000;  // raw buffer descriptor: 32-bit format, no swizzle

constexpr float kTinyOutput = 0x1p-111f;   // x K x the largest operand: smaller outputs may have lost bits
constexpr float kLargeOperand = 0x1p32f;
enum Epilogue { kEpiBias = 0, kEpiGelu = 1 };

struct LinearArgs {
  float* y;
  int64_t y_stride;
  const float* x;
  int64_t x_stride;
  const float* w;
  const float* bias;  // may be null
  int32_t M, N, K;
  int32_t m_tiles, n_tiles;
  int32_t epilogue;
  int32_t vec;       // rows of y and bias can be accessed four floats at a time
  int32_t k_part;    // k a workgroup covers: K, or K / parts with blockIdx.y the part
  int32_t parts;
};

// v (tanh-form GELU): v / (1 + exp(-2u)) = 0.5 v (1 + tanh u), u = sqrt(2/pi) (v + 0.044715 v^3),
// without the cancellation of 1 + tanh u for negative u.
__device__ __forceinline__ float gelu(float v) {
  const float u2 = -2.f * 0.7978845608028654f * (v + 0.044715f * v * v * v);
  return v / (1.f + expf(u2));
}

__device__ __forceinline__ void load8(const __amdgpu_buffer_rsrc_t& d, floatx4 (&r)[2], uint32_t offset, int32_t k) {
  r[0] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(d, offset, k * 4, 0));
  r[1] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(d, offset + 16, k * 4, 0));
}

// sum_k x[k] w[k] in fp32, K in whole steps, by one wave: the lanes take four k at a time and their sums are added
// pairwise. Every lane returns the sum.
__device__ __forceinline__ float row_dot(const float* x, const float* w, int32_t K) {
  const int lane = threadIdx.x & (kWave - 1);
  float v = 0.f;
  for (int32_t k = 4 * lane; k < K; k += 4 * kWave) {
    const floatx4 xv = *reinterpret_cast<const floatx4*>(x + k), wv = *reinterpret_cast<const floatx4*>(w + k);
#pragma unroll
    for (int e = 0; e < 4; ++e) v = fmaf(xv[e], wv[e], v);
  }
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

// What a wave finds in `count` <= 32 rows of K values: eight rows at a time, eight lanes a row.
struct Scan {
  uint32_t loses;  // bit r: row r holds a value that loses bits
  float max;       // lane r: the largest |value| of row r
};
__device__ __forceinline__ Scan scan_rows(const float* rows, int64_t stride, int count, int32_t K) {
  const int lane = threadIdx.x & (kWave - 1);
  Scan found = {0, 0.f};
#pragma unroll 1
  for (int first = 0; first < count; first += 8) {
    const float* p = rows + min(first + lane / 8, count - 1) * stride + 4 * (lane % 8);
    bool loses = false;
    float m = 0.f;
#pragma unroll 4
    for (int32_t k = 0; k < K; k += 32) {
      const floatx4 v = *reinterpret_cast<const floatx4*>(p + k);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        loses |= loses_bits(v[e]);
        m = fmaxf(m, fabsf(v[e]));
      }
    }
#pragma unroll
    for (int off = 1; off < 8; off <<= 1) m = fmaxf(m, __shfl_xor(m, off));
    const float mine = __shfl(m, 8 * (lane - first) & (kWave - 1));
    if (lane >= first && lane < first + 8) found.max = mine;
    const uint64_t any = __builtin_amdgcn_ballot_w64(loses);
#pragma unroll
    for (int r = 0; r < 8; ++r)
      if (any >> 8 * r & 0xff) found.loses |= 1u << (first + r);
  }
  return found;
}

template <int WM, int NB, int DEPTH>
__global__ __launch_bounds__(kWave* WM, WM == 8 ? 1 : 2) void linear_kernel(const LinearArgs a) {
  constexpr int BM = 32 * WM, BN = 32 * NB;
  constexpr int kUnits = 2 * NB;                     // staging units: 16 rows of W each
  constexpr int kOwn = (kUnits + WM - 1) / WM;       // units a wave stages (the last ones may repeat)
  constexpr int kPad = 36;                           // row stride of the output transpose, conflict free
  struct Stage {
    uint32x4 w[2][NB][2][3][kWave];  // [buffer][column block][k half][limb][lane]
  };
  struct Out {
    float rows[WM][32][kPad];  // a 32 x 32 block of each wave
  };
  __shared__ union {
    Stage st;
    Out out;
  } s;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int i = lane & 31, g = lane >> 5;

  // Each XCD takes a contiguous run of tiles along the shorter of M and N, so that of the two
  // operands it reads the smaller one whole and about an eighth of the other.
  const int total = a.m_tiles * a.n_tiles;
  const int q = total / kXcds, rem = total % kXcds, xcd = blockIdx.x % kXcds;
  const int p = xcd * q + min(xcd, rem) + blockIdx.x / kXcds;
  const bool rows_first = a.M < a.N;
  const int minor = rows_first ? a.m_tiles : a.n_tiles;
  const int hi = p / minor, lo = p - hi * minor;
  const int m_tile = rows_first ? lo : hi, n_tile = rows_first ? hi : lo;
  const int m0 = m_tile * BM + 32 * wave, n0 = n_tile * BN;

  const int k_lo = blockIdx.y * a.k_part;
  // Descriptors on the wave's rows of X and the tile's rows of W: loads past the last row give 0.
  const int x_rows = max(0, min(32, a.M - m0)), w_rows = min(BN, a.N - n0);
  const __amdgpu_buffer_rsrc_t xd = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(a.x + (int64_t)min(m0, a.M - 1) * a.x_stride + k_lo), (short)0,
      x_rows > 0 ? (int32_t)(((x_rows - 1) * a.x_stride + a.k_part) * 4) : 0, kBufferWord3);
  const __amdgpu_buffer_rsrc_t wd =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.w + (int64_t)n0 * a.K + k_lo), (short)0,
                                        ((w_rows - 1) * a.K + a.k_part) * 4, kBufferWord3);
  const uint32_t x_off = (uint32_t)(i * a.x_stride + 8 * g) * 4u;  // row i, octet g of each k half
  // Staging: unit rows lane / 4, k octet lane % 4 (k half octet / 2).
  const int sr = lane >> 2, so = lane & 3;
  uint32_t w_off[kOwn];
  int w_unit[kOwn];
#pragma unroll
  for (int u = 0; u < kOwn; ++u) {
    w_unit[u] = min(wave + WM * u, kUnits - 1);  // a repeated unit stores the same values again
    w_off[u] = (uint32_t)((16 * w_unit[u] + sr) * a.K + 8 * so) * 4u;
  }
  // Slot of (row, octet) in a fragment: 32 (octet % 2) + (row ^ 4 octet).
  const int slot[2] = {32 * g + (i ^ (g << 2)), 32 * g + (i ^ ((2 + g) << 2))};

  floatx16 acc[NB];
#pragma unroll
  for (int n = 0; n < NB; ++n)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[n][r] = 0.f;
  // Operands as loaded, [step % DEPTH]: a step's loads are issued DEPTH steps before it is split.
  floatx4 xr[DEPTH][2][2], wr[DEPTH][kOwn][2];
  uint32x4 xl[2][2][3];           // [step parity][k half][limb]
  auto stage = [&](int buf, const floatx4(&raw)[2], int u) {
    uint32x4 l[3];
    split8(raw[0], raw[1], l);
    const int row = (16 * (w_unit[u] & 1) + sr) ^ (so << 2);
#pragma unroll
    for (int t = 0; t < 3; ++t) s.st.w[buf][w_unit[u] >> 1][so >> 1][t][32 * (so & 1) + row] = l[t];
  };

  // One step: the MFMAs of step parity CUR; between them the next step's operands are split
  // (W's into the other buffer) and the step after's loads (at k_next) are issued. LAST: nothing
  // to prepare. The regions (column block, k half) are fenced from each other so that every
  // region keeps its own share of the split work between its MFMAs.
  auto step = [&](auto cur, auto last, int32_t k_next) {
    constexpr int CUR = decltype(cur)::value;
    constexpr bool LAST = decltype(last)::value;
    constexpr int kSplits = kOwn + 2, kRegions = 2 * NB;
    constexpr int kRaw = DEPTH == 2 ? CUR ^ 1 : 0;  // where the next step's operands are
    bf16x8 w[2][3];
#pragma unroll
    for (int t = 0; t < 3; ++t) w[0][t] = __builtin_bit_cast(bf16x8, s.st.w[CUR][0][0][t][slot[0]]);
#pragma unroll
    for (int r = 0; r < kRegions; ++r) {
      if (r + 1 < kRegions) {
#pragma unroll
        for (int t = 0; t < 3; ++t)
          w[(r + 1) & 1][t] = __builtin_bit_cast(bf16x8, s.st.w[CUR][(r + 1) / 2][(r + 1) & 1][t][slot[(r + 1) & 1]]);
      }
      if constexpr (!LAST) {
#pragma unroll
        for (int u = r * kSplits / kRegions; u < (r + 1) * kSplits / kRegions; ++u) {
          if (u < kOwn) {
            stage(CUR ^ 1, wr[kRaw][u], u);
            load8(wd, wr[kRaw][u], w_off[u], k_next);
          } else {
            floatx4(&raw)[2] = xr[kRaw][u - kOwn];
            split8(raw[0], raw[1], xl[CUR ^ 1][u - kOwn]);
            load8(xd, raw, x_off + 64 * (u - kOwn), k_next);
          }
        }
      }
#pragma unroll
      for (int t = 0; t < 6; ++t)
        acc[r / 2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            w[r & 1][kLimbA[t]], __builtin_bit_cast(bf16x8, xl[CUR][r & 1][kLimbB[t]]), acc[r / 2], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (!LAST) __syncthreads();
  };

  const int steps = a.k_part / kStep;
  const int32_t k_end = (steps - 1) * kStep;
  auto load_step = [&](int at, int32_t k) {
#pragma unroll
    for (int u = 0; u < kOwn; ++u) load8(wd, wr[at][u], w_off[u], k);
#pragma unroll
    for (int h = 0; h < 2; ++h) load8(xd, xr[at][h], x_off + 64 * h, k);
  };
  load_step(0, 0);
  if constexpr (DEPTH == 2) load_step(1, min(kStep, k_end));
#pragma unroll
  for (int u = 0; u < kOwn; ++u) stage(0, wr[0][u], u);
#pragma unroll
  for (int h = 0; h < 2; ++h) split8(xr[0][h][0], xr[0][h][1], xl[0][h]);
  load_step(0, min(DEPTH * kStep, k_end));
  __syncthreads();
  using Even = std::integral_constant<int, 0>;
  using Odd = std::integral_constant<int, 1>;
  auto ahead = [&](int t) { return min((t + 1 + DEPTH) * kStep, k_end); };  // past the end: the last step again
  int st = 0;
  for (; st + 2 < steps; st += 2) {
    step(Even{}, std::false_type{}, ahead(st));
    step(Odd{}, std::false_type{}, ahead(st + 1));
  }
  if (st + 2 == steps) {
    step(Even{}, std::false_type{}, k_end);
    step(Odd{}, std::true_type{}, 0);
  } else {
    step(Even{}, std::true_type{}, 0);
  }

  // A part of K stores its plain partial sums (no bias, no epilogue) into its own [M, N] of y.
  float* y = a.y + (int64_t)blockIdx.y * a.M * a.N;
  auto finish = [&](float v) { return a.epilogue == kEpiGelu ? gelu(v) : v; };
  float least = FLT_MAX, most = 0.f;  // of the |accumulators| that are outputs; NaN if any is
  const auto note = [&](auto ragged) {
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        const float lo = fabsf(acc[n][r]), hi = fabsf(acc[n][r + 1]);
        if constexpr (decltype(ragged)::value) {
          const int c = n0 + 32 * n + 8 * (r / 4) + 4 * g + r % 4;
          least = min3(least, c < a.N ? lo : FLT_MAX, c + 1 < a.N ? hi : FLT_MAX);
        } else {
          least = min3(least, lo, hi);
        }
        most = max3(most, lo, hi);
      }
  };
  if (__builtin_expect(n0 + BN <= a.N, 1)) note(std::false_type{});  // uniform
  else note(std::true_type{});
  __syncthreads();  // the stage buffers become the output blocks
  // Each 32 x 32 block goes through the wave's own LDS rows, so that the stores cover whole
  // 128-byte runs of y (lane: row 8 t + lane / 8, columns 4 (lane % 8) ..).
  const int oc = 4 * (lane & 7);
#pragma unroll
  for (int n = 0; n < NB; ++n) {
    wave_lds_fence();  // after the reads of the block before
#pragma unroll
    for (int r = 0; r < 4; ++r)
      *reinterpret_cast<floatx4*>(&s.out.rows[wave][i][8 * r + 4 * g]) =
          floatx4{acc[n][4 * r], acc[n][4 * r + 1], acc[n][4 * r + 2], acc[n][4 * r + 3]};
    wave_lds_fence();
    const int c = n0 + 32 * n + oc;
    floatx4 b = {0.f, 0.f, 0.f, 0.f};
    if (a.bias != nullptr) {
      if (a.vec) {
        if (c < a.N) b = *reinterpret_cast<const floatx4*>(a.bias + c);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) b[e] = c + e < a.N ? a.bias[c + e] : 0.f;
      }
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int row = 8 * t + (lane >> 3);
      floatx4 v = *reinterpret_cast<const floatx4*>(&s.out.rows[wave][row][oc]);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = finish(v[e] + b[e]);
      if (m0 + row >= a.M) continue;
      float* yp = y + (int64_t)(m0 + row) * a.y_stride + c;
      if (a.vec) {
        if (c < a.N) *reinterpret_cast<floatx4*>(yp) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (c + e < a.N) yp[e] = v[e];
      }
    }
  }

  // Outputs to be computed again (see the top of the file), a 32 x 32 block at a time.
  const float tiny = kTinyOutput * (float)a.k_part;
  if (__builtin_amdgcn_ballot_w64(m0 + i < a.M && !(least >= tiny * kLargeOperand && most <= kLargeOperand)) == 0)
    return;
  __threadfence();   // after the stores above
  wave_lds_fence();  // and the reads of their block
  const float* x_rows_at = a.x + (int64_t)m0 * a.x_stride + k_lo;
  const Scan xs = scan_rows(x_rows_at, a.x_stride, x_rows, a.k_part);
  const float x_max = __shfl(xs.max, i);
#pragma unroll 1
  for (int n = 0; n < NB && n0 + 32 * n < a.N; ++n) {
    float* block = &s.out.rows[wave][i][4 * g];  // value r of the lane: + 8 (r / 4) + r % 4
#pragma unroll
    for (int b = 0; b < NB; ++b)
      if (b == n) {
#pragma unroll
        for (int r = 0; r < 16; ++r) block[8 * (r / 4) + r % 4] = acc[b][r];
      }
    const int first = n0 + 32 * n, cols = min(32, a.N - first);
    const float* w_rows_at = a.w + (int64_t)first * a.K + k_lo;
    bool any = false;  // a finite output of a row that is not zeros is extreme: the columns count too
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float v = fabsf(block[8 * (r / 4) + r % 4]);
      any |= (v < tiny * kLargeOperand || v > kLargeOperand) && v <= FLT_MAX && 8 * (r / 4) + 4 * g + r % 4 < cols;
    }
    Scan ws = {0, 0.f};
    if (__builtin_amdgcn_ballot_w64(any && x_max > 0.f) != 0) ws = scan_rows(w_rows_at, a.K, cols, a.k_part);
#pragma unroll 1
    for (int r = 0; r < 16; ++r) {
      const float v = block[8 * (r / 4) + r % 4];  // row i, column col(g) of the block
      const auto col = [&](int group) { return 8 * (r / 4) + 4 * group + r % 4; };
      const float largest = fmaxf(x_max, __shfl(ws.max, col(g)));
      const bool lost = ((xs.loses >> i | ws.loses >> col(g)) & 1) != 0 && fabsf(v) < tiny * largest;
      uint64_t todo = __builtin_amdgcn_ballot_w64((lost || !(fabsf(v) <= FLT_MAX)) && i < x_rows && col(g) < cols);
      while (todo != 0) {  // uniform
        const int from = __builtin_ctzll(todo);
        todo &= todo - 1;
        const int m = from & 31, c = col(from >> 5);
        const float dot = row_dot(x_rows_at + m * a.x_stride, w_rows_at + (int64_t)c * a.K, a.k_part);
        if (lane == from)
          y[(int64_t)(m0 + m) * a.y_stride + first + c] = finish(a.bias != nullptr ? dot + a.bias[first + c] : dot);
      }
    }
  }
}

template <int WM, int NB, int DEPTH>
void launch(LinearArgs a, hipStream_t s) {
  a.m_tiles = (a.M + 32 * WM - 1) / (32 * WM);
  a.n_tiles = (a.N + 32 * NB - 1) / (32 * NB);
  hipLaunchKernelGGL((linear_kernel<WM, NB, DEPTH>), dim3((unsigned)(a.m_tiles * a.n_tiles), (unsigned)a.parts),
                     dim3(kWave * WM), 0, s, a);
}

// y = epilogue( the parts' sums, added in order, + bias ): a float4 per thread.
__global__ __launch_bounds__(256) void linear_sum_kernel(const LinearArgs a, const float* partials) {
  const int64_t at = 4 * ((int64_t)blockIdx.x * 256 + threadIdx.x), size = (int64_t)a.M * a.N;
  if (at >= size) return;
  floatx4 v = *reinterpret_cast<const floatx4*>(partials + at);
#pragma unroll 4
  for (int p = 1; p < a.parts; ++p) v += *reinterpret_cast<const floatx4*>(partials + p * size + at);
  const int64_t m = at / a.N;
  const int32_t c = (int32_t)(at - m * a.N);
  if (a.bias != nullptr) {  // any alignment
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] += a.bias[c + e];
  }
  if (a.epilogue == kEpiGelu) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = gelu(v[e]);
  }
  *reinterpret_cast<floatx4*>(a.y + m * a.y_stride + c) = v;
}

// Parts K is split into where the output alone gives too few of the 256 CUs a 128 x 64 tile: the
// most that keep the parts equal, at least four steps long and on a CU each. 1: no split.
constexpr int kSplitTiles = 160;
int split_parts(int64_t M, int64_t N, int64_t K) {
  constexpr int kCus = 256;
  const int64_t tiles = ((M + 127) / 128) * ((N + 63) / 64), steps = K / kStep;
  if (tiles >= kSplitTiles || N % 4 != 0) return 1;
  int parts = 1;
  for (int p = 2; p * tiles <= kCus && 4 * p <= steps; ++p)
    if (steps % p == 0) parts = p;
  return parts;
}

// Tile shapes and what one tile takes per 32 of K alone on a CU (ns, measured at K = 3072). A CU
// gains nothing from a second resident tile (LDS and the matrix cores are busy already), so a
// launch takes ceil(tiles / 256) of them in a row: the shape with the least rounds x time wins.
// (E.g. 1,987 rows x 2,304: 128 x 64 tiles need three rounds, 52 us; 256 x 96 one, 43 us.)
struct TileShape {
  int wm, nb;
  int step_ns;
};
constexpr TileShape kShapes[] = {{4, 1, 575}, {4, 2, 630}, {4, 3, 885}, {4, 4, 1000}, {8, 3, 1235}, {8, 4, 1630}};

const TileShape& choose_shape(int64_t M, int64_t N) {
  constexpr int64_t kCus = 256;
  const TileShape* best = nullptr;
  int64_t best_ns = 0;
  for (const TileShape& t : kShapes) {
    const int64_t tiles = ((M + 32 * t.wm - 1) / (32 * t.wm)) * ((N + 32 * t.nb - 1) / (32 * t.nb));
    const int64_t ns = (tiles + kCus - 1) / kCus * t.step_ns;
    if (best == nullptr || ns < best_ns) best = &t, best_ns = ns;
  }
  return *best;
}

}  // namespace
}  // namespace tq

extern "C" size_t tq_linear_workspace_size(int32_t M, int32_t N, int32_t K) {
  using namespace tq;
  if (M < 1 || N < 1 || K < 1 || K % kStep != 0) return 0;
  const int parts = split_parts(M, N, K);
  return parts > 1 ? (size_t)parts * M * N * 4 : 0;
}

extern "C" tq_status tq_linear(float* y, int64_t y_stride, const float* x, int64_t x_stride, int32_t M, const float* w,
                               const float* bias, int32_t N, int32_t K, int32_t epilogue, void* workspace,
                               size_t workspace_bytes, void* stream) {
  using namespace tq;
  if (M < 0 || N < 1 || K < 1 || epilogue < 0 || epilogue > 1) return TQ_ERR_INVALID_ARGUMENT;
  // 32-bit offsets inside a tile; K in whole steps.
  if (K % kStep != 0 || (int64_t)K * 4 * 256 > 0x7fffffffLL || x_stride * 4 * 256 > 0x7fffffffLL)
    return TQ_ERR_UNSUPPORTED;
  if (M == 0) return TQ_OK;
  if (y == nullptr || x == nullptr || w == nullptr) return TQ_ERR_INVALID_ARGUMENT;
  if (x_stride < K || y_stride < N) return TQ_ERR_INVALID_ARGUMENT;
  if (((uintptr_t)x | (uintptr_t)w) % 16 != 0 || x_stride % 4 != 0) return TQ_ERR_INVALID_ARGUMENT;
  if (((int64_t)M + 127) / 128 * (((int64_t)N + 31) / 32) > 0x7fffffffLL) return TQ_ERR_UNSUPPORTED;
  LinearArgs a = {};
  a.y = y;
  a.y_stride = y_stride;
  a.x = x;
  a.x_stride = x_stride;
  a.w = w;
  a.bias = bias;
  a.M = M;
  a.N = N;
  a.K = K;
  a.epilogue = epilogue;
  const bool vec_y = N % 4 == 0 && y_stride % 4 == 0 && (uintptr_t)y % 16 == 0;
  a.vec = vec_y && (uintptr_t)bias % 16 == 0;
  a.k_part = K;
  a.parts = 1;
  hipStream_t s = (hipStream_t)stream;
  // The sum writes whole float4s; an unaligned bias alone does not need the split's workspace.
  const int parts = vec_y && (a.vec || workspace != nullptr) ? split_parts(M, N, K) : 1;
  if (parts > 1) {
    if (workspace == nullptr || workspace_bytes < tq_linear_workspace_size(M, N, K) || (uintptr_t)workspace % 16 != 0)
      return TQ_ERR_WORKSPACE;
    LinearArgs part = a;
    part.y = static_cast<float*>(workspace);
    part.y_stride = N;
    part.bias = nullptr;
    part.vec = 1;
    part.epilogue = kEpiBias;
    part.k_part = K / parts;
    part.parts = a.parts = parts;
    launch<4, 2, 2>(part, s);
    const int64_t groups = ((int64_t)M * N / 4 + 255) / 256;
    hipLaunchKernelGGL(linear_sum_kernel, dim3((unsigned)groups), dim3(256), 0, s, a,
                       static_cast<const float*>(workspace));
    return check_launch();
  }
  const TileShape& t = choose_shape(M, N);
  switch (t.wm * 10 + t.nb) {
    case 41: launch<4, 1, 2>(a, s); break;
    case 42: launch<4, 2, 2>(a, s); break;
    case 43: launch<4, 3, 2>(a, s); break;
    case 44: launch<4, 4, 1>(a, s); break;
    case 83: launch<8, 3, 2>(a, s); break;
    default: launch<8, 4, 2>(a, s); break;
  }
  return check_launch();
}
