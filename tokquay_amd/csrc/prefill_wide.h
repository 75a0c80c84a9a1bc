// Causal prefill attention for launches with many query rows, on the bf16 matrix cores at fp32
// precision (three bf16 limbs per operand, six products: linear.hip).
//
// A workgroup takes 128 consecutive queries of one (sequence, head), 32 per wave, and walks the
// keys 32 at a time. The K and V tiles are read and split into limbs once per workgroup and
// shared through LDS (double buffered, one barrier per tile); per wave and tile
//
//   S^T[key][query]  = K[key][:] . Q[query][:]         4 dim steps of 16 x 6 limb products
//   O^T[dim][query] += V^T[dim][key] P^T[key][query]   2 key steps of 16 x 2 dim blocks x 6
//
// on v_mfma_f32_32x32x16_bf16: 48 MFMAs of 32 cycles where the fp32 MFMAs of the 16-row kernels
// take 128 of 32. As there, the transposed scores leave the probabilities where the PV product
// wants them: lane (q, g) = (lane % 32, lane / 32) holds query q and keys 8 (r / 4) + 4 g + r % 4,
// r = 0..15, in S^T's accumulator; r = 8 h .. 8 h + 7 are the keys key step h takes from lane group
// g, in that order, and V is staged in that order (eight keys of one dim per lane).
//
// Staging, per wave: 8 keys of K (lane: key lane / 8, dim octet lane % 8, so four lanes share a
// 128-byte line: with a key row per lane the address unit takes one lane a clock) and the 8 keys
// of V that one (key step, lane group) reads (lane = dim, one 256-byte row per load). Keys past the
// workgroup's range and bad block ids read as zeros (descriptor sizes).
//
// The tiles are pipelined so that the scores of tile t + 1 run beside the softmax of tile t and
// the staging beside the PV product. A 128-query workgroup alone on a CU takes 1.5 us per tile
// (0.64 us of it MFMA); two per CU reach 201 TFLOP/s of fp32 products (2 x 8,192 rows), which is the
// rate a large bf16 library product reaches here, a sixth each (MFMA busy for 66 % of the cycles at 1.4 GHz: power
// bound; 44 % at 1.8 GHz for 32 prompts of 256-1,023 rows). Three per CU (168 VGPRs) spill and
// ran 10 % slower.
//
// The softmax is the 16-row kernels' (log2 units, lazy maximum). Queries whose result is not finite are
// computed again from the fp32 values (limbs of infinities and NaN are NaN, which would also reach queries
// that must not see them), and so are those that values of V below 2^-110 cost precision: each is off by up to 2^-134
// (split_bf16.h), as is each probability, which is below 2^-22 of an output of 2^-112 (keys max |v| + 1). A wave with an
// output below keys 2^-80 or above 2^32 looks through its V for such values and the largest one. All other
// queries keep their bits. Queries and keys: a score is off by up to 64 x 2^-133 of the larger operand, under
// 2^-20 up to 2^107. (Largest |K| and |V| kept in the loop, for outputs of every size, took 2-6 %.)
#pragma once

#include <float.h>

#include "prefill_args.h"
#include "split_bf16.h"

namespace tq {
namespace {

constexpr int kWideWaves = 4;
constexpr int kWideRows = 32 * kWideWaves;  // queries of a workgroup
constexpr int kWideKeys = 32;               // keys of a tile

// Causal attention of query `row` (position qpos) of one head in plain fp32, by one wave: lane = dim.
template <int BS>
__device__ __forceinline__ void prefill_plain_row(const PrefillArgs& a, const int32_t* bt, const float* head_base, int row,
                                               int qpos, int h) {
  const int lane = threadIdx.x & (kWave - 1);
  const float q = a.q[(int64_t)row * a.q_stride + h * kHeadDim + lane] * (a.scale * kLog2e);
  float m = -FLT_MAX, l = 0.f, o = 0.f;
  for (int key = 0; key <= qpos; ++key) {
    const int32_t blk = bt[key / BS];
    const bool ok = (uint32_t)blk < (uint32_t)a.num_blocks;  // bad ids are reported by the main loop
    const float* kp = head_base + (int64_t)(ok ? blk : 0) * a.block_stride + (key % BS) * kHeadDim + lane;
    float s = q * (ok ? kp[0] : 0.f);
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) s += __shfl_xor(s, off);
    const float mn = max2(m, s);
    const float c = __builtin_amdgcn_exp2f(m - mn), p = __builtin_amdgcn_exp2f(s - mn);
    l = fmaf(l, c, p);
    o = fmaf(o, c, p * (ok ? kp[a.kv_stride] : 0.f));
    m = mn;
  }
  a.out[(int64_t)row * a.out_stride + h * kHeadDim + lane] = o / l;
}

// Whether the first n keys' V of one head hold a value that loses bits, and the largest finite |v|. By one wave.
template <int BS>
__device__ __forceinline__ bool values_lose_bits(const PrefillArgs& a, const int32_t* bt, const float* head_base, int n,
                                                 float& largest) {
  const int lane = threadIdx.x & (kWave - 1);
  bool loses = false;
  float m = 0.f;
#pragma unroll 4
  for (int key = lane >> 4; key < n; key += 4) {  // 16 lanes a row
    const int32_t blk = bt[key / BS];
    if ((uint32_t)blk >= (uint32_t)a.num_blocks) continue;
    const floatx4 v = *reinterpret_cast<const floatx4*>(head_base + (int64_t)blk * a.block_stride + a.kv_stride +
                                                        (key % BS) * kHeadDim + 4 * (lane & 15));
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      loses |= loses_bits(v[e]);
      m = fabsf(v[e]) <= FLT_MAX ? fmaxf(m, fabsf(v[e])) : m;
    }
  }
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  largest = m;
  return __builtin_amdgcn_ballot_w64(loses) != 0;
}

template <int BS>
__global__ __launch_bounds__(kWave* kWideWaves, 2) void prefill_wide_kernel(const PrefillArgs a) {
  static_assert(BS == 16 || BS == 32, "a wave's staged keys lie in one block");
  __shared__ uint32x4 s_k[2][4][3][kWave];     // [buffer][dim step][limb][slot]
  __shared__ uint32x4 s_v[2][2][2][3][kWave];  // [buffer][dim block][key step][limb][slot]
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  int qt, h, b;
  if (!tile_of(a, blockIdx.x, qt, h, b)) return;  // padding workgroup (uniform)
  if (a.seq_order != nullptr) {
    const int sb = a.seq_order[b];
    if ((uint32_t)sb >= (uint32_t)a.num_seqs) {
      if (qt == 0 && h == 0 && threadIdx.x == 0) flag_error(a.d_error, TQ_DEVERR_ORDER);
      return;
    }
    b = sb;
  }
  // Uniform by construction; readfirstlane keeps what follows (loop bounds, descriptors) scalar.
  const int row0 = __builtin_amdgcn_readfirstlane(a.cu_q[b]);
  const int nq = __builtin_amdgcn_readfirstlane(a.cu_q[b + 1]) - row0;
  const int wg_q0 = qt * kWideRows;
  if (wg_q0 >= nq) return;
  const int start = __builtin_amdgcn_readfirstlane(a.q_start[b]);
  if (row0 < 0 || row0 + nq > a.num_q_rows || start < 0 || (int64_t)start + nq > (int64_t)a.max_blocks * BS) {
    if (qt == 0 && h == 0 && lane == 0) flag_error(a.d_error, TQ_DEVERR_LENGTH);
    return;
  }
  const int i = lane & 31, g = lane >> 5;
  const int q0 = wg_q0 + 32 * wave;  // the wave's first query
  const int rows = min(32, nq - q0);  // its queries (none: the wave only stages)
  const int qpos = start + min(q0 + i, nq - 1);
  const int qpos_lo = start + q0, qpos_hi = start + q0 + rows - 1;
  const int kend = start + min(wg_q0 + kWideRows, nq);  // keys the workgroup can see: [0, kend)
  const int tiles = (kend + kWideKeys - 1) / kWideKeys;

  const int32_t* bt = a.block_tables + (int64_t)b * a.bt_stride;
  const float* head_base = a.pool_layer + (int64_t)h * a.head_stride;

  // Q limbs: B operand of dim step ds, octet 2 ds + g of query i, pre-scaled into log2 units.
  uint32x4 ql[4][3];
  {
    const float qscale = a.scale * kLog2e;
    const float* qp = a.q + (int64_t)(row0 + min(q0 + i, nq - 1)) * a.q_stride + h * kHeadDim + 8 * g;
#pragma unroll
    for (int ds = 0; ds < 4; ++ds) {
      const floatx4 lo = *reinterpret_cast<const floatx4*>(qp + 16 * ds) * qscale;
      const floatx4 hi = *reinterpret_cast<const floatx4*>(qp + 16 * ds + 4) * qscale;
      split8(lo, hi, ql[ds]);
    }
  }

  // The staged keys' block: entry (kt + 16 (wave / 2)) / BS; 64 entries at a time sit one per lane.
  int tb_base = -1;
  int32_t tb_id = 0;
  auto block_of = [&](int t) {  // -1: past the range, or a bad id
    const int ti = (t * kWideKeys + 16 * (wave >> 1)) / BS;
    if ((ti & ~63) != tb_base) {  // wave-uniform
      tb_base = ti & ~63;
      const int nblk = (kend + BS - 1) / BS;
      tb_id = -1;
      if (tb_base + lane < nblk) {
        const int32_t id = bt[tb_base + lane];
        if ((uint32_t)id < (uint32_t)a.num_blocks) tb_id = id;
        else flag_error(a.d_error, TQ_DEVERR_BLOCK_ID);
      }
    }
    return __builtin_amdgcn_readlane(tb_id, ti - tb_base);
  };
  // The wave's share of key tile t as loaded, t's block id given. K: rows 8 wave .. + 7 of the tile;
  // V: rows v0 .. + 3 and v0 + 8 .. + 11, v0 = 16 (wave / 2) + 4 (wave % 2).
  constexpr int kRowBytes = kHeadDim * 4;
  floatx4 kraw[2];
  float vraw[8];
  auto fetch_k = [&](int t, int32_t blk) {
    const int first = t * kWideKeys + 8 * wave;
    const int n = __builtin_amdgcn_readfirstlane(blk < 0 ? 0 : max(0, min(8, kend - first)));  // no v_med3
    const __amdgpu_buffer_rsrc_t d = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(head_base + (int64_t)max(blk, 0) * a.block_stride + (first % BS) * kHeadDim), (short)0,
        n * kRowBytes, kBufferWord3);
#pragma unroll
    for (int c = 0; c < 2; ++c)
      kraw[c] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(d, (uint32_t)(lane * 32 + 16 * c), 0, 0));
  };
  auto fetch_v = [&](int t, int32_t blk) {
    const int first = t * kWideKeys + 16 * (wave >> 1) + 4 * (wave & 1);
    const int n = __builtin_amdgcn_readfirstlane(blk < 0 ? 0 : max(0, min(12, kend - first)));
    const __amdgpu_buffer_rsrc_t d = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(head_base + (int64_t)max(blk, 0) * a.block_stride + a.kv_stride + (first % BS) * kHeadDim),
        (short)0, n * kRowBytes, kBufferWord3);
#pragma unroll
    for (int s = 0; s < 8; ++s)
      vraw[s] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
          d, (uint32_t)(lane * 4 + (s < 4 ? s : s + 4) * kRowBytes), 0, 0));
  };
  // Slots: K (key, octet o of dims) at 32 (o % 2) + (key ^ 2 o) of dim step o / 2; V in lane order.
  auto stage_k = [&](int buf) {
    uint32x4 l[3];
    split8(kraw[0], kraw[1], l);
    const int key = 8 * wave + (lane >> 3), o = lane & 7;
#pragma unroll
    for (int t = 0; t < 3; ++t) s_k[buf][o >> 1][t][32 * (o & 1) + (key ^ (2 * o))] = l[t];
  };
  auto stage_v = [&](int buf) {
    uint32x4 l[3];
    split8(floatx4{vraw[0], vraw[1], vraw[2], vraw[3]}, floatx4{vraw[4], vraw[5], vraw[6], vraw[7]}, l);
#pragma unroll
    for (int t = 0; t < 3; ++t) s_v[buf][lane >> 5][wave >> 1][t][32 * (wave & 1) + (lane & 31)] = l[t];
  };

  floatx16 o[2], st;
#pragma unroll
  for (int r = 0; r < 16; ++r) o[0][r] = o[1][r] = st[r] = 0.f;
  float m = -FLT_MAX, mthr = -FLT_MAX + kSlack, l = 0.f;

  auto read_k = [&](bf16x8 (&kf)[3], int buf, int ds) {
    const int oc = 2 * ds + g;
#pragma unroll
    for (int u = 0; u < 3; ++u) kf[u] = __builtin_bit_cast(bf16x8, s_k[buf][ds][u][32 * g + (i ^ (2 * oc))]);
  };
  auto scores = [&](floatx16& acc, const bf16x8 (&kf)[3], int ds) {
#pragma unroll
    for (int u = 0; u < 6; ++u)
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[kLimbA[u]], __builtin_bit_cast(bf16x8, ql[ds][kLimbB[u]]), acc,
                                                    0, 0, 0);
  };

  // Pipeline: iteration t has S^T of tile t in st, K of t + 1 and V of t in LDS, K of t + 2 and V of
  // t + 1 in registers. The score products of tile t + 1 run beside the softmax of tile t (the VALU
  // work of one hides behind the MFMAs of the other), the staging beside the PV products.
  // Tiles past the end are the last one again.
  const int last = tiles - 1;
  int32_t blk = block_of(0);
  fetch_k(0, blk);
  fetch_v(0, blk);
  stage_k(0);
  stage_v(0);
  blk = block_of(min(1, last));
  fetch_k(min(1, last), blk);
  fetch_v(min(1, last), blk);
  __syncthreads();
  if (rows > 0) {
    bf16x8 kf[3];
#pragma unroll
    for (int ds = 0; ds < 4; ++ds) {
      read_k(kf, 0, ds);
      scores(st, kf, ds);
    }
  }
  stage_k(1);
  blk = block_of(min(2, last));
  fetch_k(min(2, last), blk);
  __syncthreads();
  for (int t = 0; t < tiles; ++t) {
    const int vbuf = t & 1, kbuf = vbuf ^ 1, kt = t * kWideKeys;
    const int32_t v_blk = blk;  // block of tile t + 2, for its V; K goes on to t + 3
    blk = block_of(min(t + 3, last));
    if (rows > 0 && kt <= qpos_hi) {  // uniform: some query of the wave sees the tile
      bf16x8 kf[2][3];
      read_k(kf[0], kbuf, 0);
      if (kt + kWideKeys - 1 > qpos_lo) {  // uniform: the tile crosses the wave's diagonal
#pragma unroll
        for (int r = 0; r < 16; ++r) st[r] = kt + 8 * (r / 4) + 4 * g + r % 4 <= qpos ? st[r] : -INFINITY;
      }
      float lmax = max4(st[0], st[1], st[2], st[3]);
#pragma unroll
      for (int r = 4; r < 16; r += 4) lmax = max2(lmax, max4(st[r], st[r + 1], st[r + 2], st[r + 3]));
      if (__builtin_amdgcn_ballot_w64(lmax > mthr) != 0) {
        const auto other = __builtin_amdgcn_permlane32_swap(__float_as_uint(lmax), __float_as_uint(lmax), false, false);
        const float tmax = max2(__uint_as_float(other[0]), __uint_as_float(other[1]));
        const bool grow = tmax > mthr;
        const float mn = grow ? tmax : m;
        const float corr = grow ? __builtin_amdgcn_exp2f(m - mn) : 1.f;
        l *= corr;
        o[0] *= corr;
        o[1] *= corr;
        m = mn;
        mthr = mn + kSlack;
      }
      floatx16 sn;
#pragma unroll
      for (int r = 0; r < 16; ++r) sn[r] = 0.f;
      uint32x4 pl[2][3];
      bf16x8 vf[2][3];
      // Dim step ds of tile t + 1's scores beside a quarter of tile t's probabilities.
      float p[8];
#pragma unroll
      for (int ds = 0; ds < 4; ++ds) {
        if (ds < 3) read_k(kf[(ds + 1) & 1], kbuf, ds + 1);
        if (ds == 3) {
#pragma unroll
          for (int u = 0; u < 3; ++u) vf[0][u] = __builtin_bit_cast(bf16x8, s_v[vbuf][0][0][u][lane]);
        }
        scores(sn, kf[ds & 1], ds);
        if (ds % 2 == 0) {
#pragma unroll
          for (int r = 0; r < 8; ++r) p[r] = __builtin_amdgcn_exp2f(st[4 * ds + r] - m);
          l += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
        } else {
          split8(floatx4{p[0], p[1], p[2], p[3]}, floatx4{p[4], p[5], p[6], p[7]}, pl[ds / 2]);
        }
#pragma unroll
        for (int u = 0; u < 6; ++u) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x402, 8, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {  // key step r / 2, dim block r % 2
        if (r < 3) {
#pragma unroll
          for (int u = 0; u < 3; ++u)
            vf[(r + 1) & 1][u] = __builtin_bit_cast(bf16x8, s_v[vbuf][(r + 1) & 1][(r + 1) >> 1][u][lane]);
        }
        if (r == 1) stage_k(vbuf);       // K of tile t + 2 over tile t's
        if (r == 2) stage_v(vbuf ^ 1);   // V of tile t + 1
#pragma unroll
        for (int u = 0; u < 6; ++u)
          o[r & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              vf[r & 1][kLimbA[u]], __builtin_bit_cast(bf16x8, pl[r >> 1][kLimbB[u]]), o[r & 1], 0, 0, 0);
        if (r == 1 || r == 2) {
#pragma unroll
          for (int u = 0; u < 6; ++u) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      st = sn;
    } else {
      stage_k(vbuf);
      stage_v(vbuf ^ 1);
    }
    fetch_k(min(t + 3, last), blk);
    fetch_v(min(t + 2, last), v_blk);
    __syncthreads();
  }
  if (rows <= 0) return;

  const auto other = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
  l = __uint_as_float(other[0]) + __uint_as_float(other[1]);
  float least = FLT_MAX, most = l;  // of the query's |sums| in this lane; NaN if any is
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    least = min3(least, fabsf(o[0][r]), fabsf(o[1][r]));
    most = max3(most, fabsf(o[0][r]), fabsf(o[1][r]));
  }
  bool redo = !(most <= FLT_MAX);
  // Uniform: whether values may have lost bits (see the top of the file).
  if (__builtin_amdgcn_ballot_w64(!redo && (least < (float)kend * 0x1p-80f || most > 0x1p32f)) != 0) {
    float vmax;
    if (values_lose_bits<BS>(a, bt, head_base, kend, vmax))
      redo |= least < 0x1p-112f * fmaf((float)kend, vmax, l);
  }
  // Lanes i and i + 32 hold the two dim blocks of query i.
  const uint64_t lanes = __builtin_amdgcn_ballot_w64(redo && i < rows);
  uint32_t again = (uint32_t)lanes | (uint32_t)(lanes >> 32);  // uniform: queries to compute again
  if (i < rows && !(again >> i & 1)) {
    const float inv = 1.f / l;
    float* op = a.out + (int64_t)(row0 + q0 + i) * a.out_stride + h * kHeadDim;
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        *reinterpret_cast<floatx4*>(op + 32 * d + 8 * r + 4 * g) =
            floatx4{o[d][4 * r], o[d][4 * r + 1], o[d][4 * r + 2], o[d][4 * r + 3]} * inv;
  }
  while (again != 0) {
    const int r = __builtin_ctz(again);
    again &= again - 1;
    prefill_plain_row<BS>(a, bt, head_base, row0 + q0 + r, start + q0 + r, h);
  }
}

}  // namespace
}  // namespace tq
