// What the prefill kernels share: their arguments, the dispatch order of their tiles, the maxima
// of their online softmax.
#pragma once

#include "tq_internal.h"

namespace tq {
namespace {

constexpr int kTile = 16;  // queries per tile and keys per step of the 16-row kernels
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kSlack = 8.f;  // log2 units a stale running maximum may trail a score by

struct PrefillArgs {
  float* out;
  int64_t out_stride;
  const float* q;
  int64_t q_stride;
  const float* pool_layer;
  int64_t block_stride;
  int64_t kv_stride;
  int64_t head_stride;
  const int32_t* block_tables;
  int64_t bt_stride;
  const int32_t* cu_q;
  const int32_t* q_start;
  const int32_t* seq_order;  // dispatch rank -> sequence, or nullptr for the natural order
  int32_t* d_error;
  float scale;
  int32_t num_blocks;
  int32_t num_heads;
  int32_t block_size;
  int32_t max_blocks;
  int32_t num_q_rows;
  int32_t max_query_len;
  int32_t qtiles;     // query tiles per (sequence, head)
  int32_t num_seqs;
  int32_t groups;     // num_heads * num_seqs
  int32_t total;      // workgroups: 8 XCDs x the most groups on one XCD x qtiles
};

constexpr int kXcds = 8;      // MI355X: workgroup i is dispatched to XCD i % 8
// Word 3 of a raw (untyped) buffer descriptor on gfx9-family GPUs: data format 32 bits (a
// nonzero format makes the loads valid), no swizzle, no typed conversion.
constexpr int kBufferWord3 = 0x00020000;
constexpr int kRound = 64;    // dispatches per XCD taken as one round (two per CU of its 32)

// Maps the dispatch index to a work tile. Workgroup p runs on XCD p % 8 (checked
// on MI355X with the XCC_ID register), and the XCD hands its workgroups to its 32
// CUs round robin. The (sequence, head) groups are dealt out whole, group g to XCD
// g % 8, so all query tiles of a group share one L2 for their K/V reads and the
// heads of a long sequence spread over all eight XCDs; an XCD with one group fewer
// than the most gets padding workgroups that exit at once. Inside an XCD the tiles
// go out by cost (query tile index, descending across its G groups) and the rounds
// of kRound dispatches snake: round k even takes cost ranks k kRound .. k kRound +
// kRound - 1 in order, odd in reverse, so the tiles a CU receives over two rounds
// add up to about the same number of key tiles (measured on 256-token chunks of 4
// prompts: 15.1 / 24.9 / 34.5 -> 11.5 / 21.5 / 31.4 us at starts 0 / 256 / 512
// against contiguous runs with the last query tiles first; rounds of 32 or 128 do
// about as well, 16 worse; dealing contiguous runs of groups instead of every
// eighth group left a 3-prompt chunk with one long prompt 45 % slower). Returns
// false for a padding workgroup. `p` is the workgroup's index among the launch's prefill
// workgroups, a multiple of 8 dispatches after the first (so p % 8 is still its XCD). The
// sequence b it returns is a dispatch rank; a.seq_order maps it to the sequence itself.
__device__ __forceinline__ bool tile_of(const PrefillArgs& a, int p, int& qt, int& h, int& b) {
  const int xcd = p % kXcds, local = p / kXcds;
  const int G = (a.groups - xcd + kXcds - 1) / kXcds;  // groups xcd, xcd + 8, ... on this XCD
  const int n = G * a.qtiles;
  if (local >= n) return false;
  const int k = local / kRound, c = local - k * kRound;
  const int m = min(kRound, n - k * kRound);  // size of this round
  const int rank = k * kRound + ((k & 1) ? m - 1 - c : c);
  qt = a.qtiles - 1 - rank / G;
  const int seq_head = xcd + kXcds * (rank % G);
  h = seq_head % a.num_heads;
  b = seq_head / a.num_heads;
  return true;
}

// Maxima are IEEE maximum (v_maximum3_f32 / v_maximum_f32): unlike fmaxf they need no
// canonicalization of their operands, and a NaN score propagates instead of being dropped.
__device__ __forceinline__ float max2(float a, float b) { return __builtin_elementwise_maximum(a, b); }
__device__ __forceinline__ float max4(float a, float b, float c, float d) { return max2(max2(a, b), max2(c, d)); }

}  // namespace
}  // namespace tq
