// What the decode rows' kernels and the packed-prefill entry share: the arguments
// and partition of a row, wave reductions, and the merge of its split partials.
#pragma once

#include "common.h"

namespace vrh {

constexpr int kMaxSplits = 16;

struct DecodeArgs {
  void* out;
  const void* q;
  const void* k;
  const void* v;
  const int32_t* tables;
  const int32_t* lengths;
  float* part_ml;   // [rows, q_heads, kMaxSplits, 2]
  float* part_acc;  // [rows, q_heads, kMaxSplits, head_dim]
  int64_t q_row, q_head, o_row, o_head;
  int64_t k_block, k_token, k_head;
  int64_t v_block, v_token, v_head;
  int64_t table_stride;
  int64_t row_base;
  int64_t rows;      // rows of the whole call (the launch may cover a chunk)
  // A head's row of K or V is not a whole number of 128-byte cache lines, so
  // neighbouring heads (other waves) share lines: every page is then read
  // with cache-allocating loads.
  int32_t line_shared;
  // Packed-prefill expansion (null for decode): row r is query i of sequence
  // s with cu_q[s] <= r < cu_q[s+1]; it reads table row s with causal length
  // lengths[s] - q_len(s) + i + 1.
  // expand_e > 0: row r is query r % E of sequence r / E, and only sequences
  // with q_len <= E are processed here (the others belong to the MFMA kernel).
  const int32_t* cu_q;
  int32_t num_seqs;
  int32_t expand_e;
  int32_t unit_group;  // waves (or workgroups) of one kv head, split and row
  int32_t q_heads, group, head_dim, block_size, bs_shift, window, min_bps, table_width;
  int32_t long_bps;   // pages of the shortest split of other rows
  int32_t short_pages;  // longest row (pages) cut into splits of min_bps
  int32_t min_part;   // pages of the shortest part of a split
  int32_t max_parts;  // most parts of a split
  int32_t part_unit;  // pages of a chunk: parts are whole multiples
  float scale_log2;
};

struct Partition {
  int start;    // first visible token
  int first;    // first page
  int pages;    // pages touched
  int bps;      // pages per split
  int nsplit;
};

__device__ __forceinline__ Partition partition(int n, const DecodeArgs& a) {
  Partition p;
  p.start = (a.window > 0 && n > a.window) ? n - a.window : 0;
  if (a.bs_shift >= 0) {
    p.first = p.start >> a.bs_shift;
    p.pages = ((n + a.block_size - 1) >> a.bs_shift) - p.first;
  } else {
    p.first = p.start / a.block_size;
    p.pages = (n + a.block_size - 1) / a.block_size - p.first;
  }
  const int least = p.pages > a.long_bps && p.pages <= a.short_pages ? a.min_bps : a.long_bps;
  p.bps = max(least, ceil_div(p.pages, kMaxSplits));
  p.nsplit = ceil_div(p.pages, p.bps);
  return p;
}

// Pages per part of a split (the whole split: one part). A split of up to two
// shortest parts is not cut: folding costs launches that run parts in turn 4-8 % at
// two parts (6 rows of 2300-3000 tokens, 32 over 8 heads, 27.2 against 25.6 us) and
// gains lone rows little (19.8 against 21.5; tables of up to 4096 tokens then have no
// parts at all). Parts are whole chunks, so that only a split's last one has a chunk
// that is not full (3 rows of 18000-22500 tokens 97.9 us without, 94.2 with).
__device__ __forceinline__ int part_pages(const Partition& p, const DecodeArgs& a) {
  if (p.bps <= 2 * a.min_part) return p.bps;
  const int even = ceil_div(p.bps, a.max_parts);
  return max(a.min_part, ceil_div(even, a.part_unit) * a.part_unit);
}

__device__ __forceinline__ int clamp_length(int n, const DecodeArgs& a) {
  // A length beyond the table would read past the row's page ids.
  const int64_t cap = (int64_t)a.table_width * a.block_size;
  if (n < 0) return 0;
  return (int64_t)n > cap ? (int)cap : n;
}

// Visible length, table row and query/output row of work row `row`
// (decode: itself); -1 when the row is not handled by this launch.
__device__ __forceinline__ int row_length(int64_t row, const DecodeArgs& a, int64_t* table_row,
                                          int64_t* query_row) {
  if (a.cu_q == nullptr) {
    *table_row = row;
    *query_row = row;
    return clamp_length(a.lengths[row], a);
  }
  int seq, i;
  if (a.expand_e > 0) {
    seq = (int)(row / a.expand_e);
    i = (int)(row - (int64_t)seq * a.expand_e);
  } else {
    // Rows outside [cu_q[0], cu_q[num_seqs]) (padding of a bucketed q) belong
    // to no sequence.
    if (row < a.cu_q[0] || row >= a.cu_q[a.num_seqs]) return -1;
    int lo = 0, hi = a.num_seqs - 1;  // last s with cu_q[s] <= row
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (a.cu_q[mid] <= row) lo = mid; else hi = mid - 1;
    }
    seq = lo;
    i = (int)(row - a.cu_q[lo]);
  }
  const int q_len = a.cu_q[seq + 1] - a.cu_q[seq];
  if (i < 0 || i >= q_len || (a.expand_e > 0 && q_len > a.expand_e)) return -1;
  *table_row = seq;
  *query_row = a.cu_q[seq] + i;
  return clamp_length(a.lengths[seq] - q_len + i + 1, a);
}

// Maximum of an int over the wave: DPP within rows of 16 lanes, then the 4
// row results through scalar reads (no LDS traffic).
__device__ __forceinline__ int wave_max_i(int x) {
  x = max(x, __builtin_amdgcn_update_dpp(0, x, kDppQuadXor1, 0xF, 0xF, false));
  x = max(x, __builtin_amdgcn_update_dpp(0, x, kDppQuadXor2, 0xF, 0xF, false));
  x = max(x, __builtin_amdgcn_update_dpp(0, x, kDppRowHalfMirror, 0xF, 0xF, false));
  x = max(x, __builtin_amdgcn_update_dpp(0, x, kDppRowMirror, 0xF, 0xF, false));
  return max(max(__builtin_amdgcn_readlane(x, 0), __builtin_amdgcn_readlane(x, 16)),
             max(__builtin_amdgcn_readlane(x, 32), __builtin_amdgcn_readlane(x, 48)));
}

// Sum of an int over the wave, likewise.
__device__ __forceinline__ int wave_sum_i(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, kDppQuadXor1, 0xF, 0xF, false);
  x += __builtin_amdgcn_update_dpp(0, x, kDppQuadXor2, 0xF, 0xF, false);
  x += __builtin_amdgcn_update_dpp(0, x, kDppRowHalfMirror, 0xF, 0xF, false);
  x += __builtin_amdgcn_update_dpp(0, x, kDppRowMirror, 0xF, 0xF, false);
  return __builtin_amdgcn_readlane(x, 0) + __builtin_amdgcn_readlane(x, 16) +
         __builtin_amdgcn_readlane(x, 32) + __builtin_amdgcn_readlane(x, 48);
}

// Log-sum-exp merge of one (row, q head)'s split partials by one wave, for
// head dims [d0, d0 + 64 * ND): lane s holds split s's weight; each lane owns
// ND dims and issues the loads of all splits at once, then combines them in
// split order.
template <typename T, int ND>
__device__ __forceinline__ void merge_partials(const DecodeArgs& a, int64_t row, int head,
                                               int64_t qrow, int nsplit, int lane, int d0) {
  const int64_t idx0 = (row * a.q_heads + head) * kMaxSplits;
  const bool live = lane < nsplit;
  const float mi = live ? a.part_ml[(idx0 + lane) * 2 + 0] : -INFINITY;
  const float li = live ? a.part_ml[(idx0 + lane) * 2 + 1] : 0.f;
  const float M = wave_max(mi);
  const float wi = live ? fast_exp2(mi - M) : 0.f;
  const float L = wave_sum(wi * li);
  const float inv = fast_rcp(fmaxf(L, 1e-30f));
  const float* part = a.part_acc + idx0 * a.head_dim;
  float acc[ND];
#pragma unroll
  for (int e = 0; e < ND; ++e) acc[e] = 0.f;
  float v[kMaxSplits][ND];
#pragma unroll
  for (int j = 0; j < kMaxSplits; ++j)
#pragma unroll
    for (int e = 0; e < ND; ++e) {
      const int d = d0 + lane + 64 * e;
      v[j][e] = (j < nsplit && d < a.head_dim) ? part[(int64_t)j * a.head_dim + d] : 0.f;
    }
#pragma unroll
  for (int j = 0; j < kMaxSplits; ++j) {
    const float w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wi), j));
#pragma unroll
    for (int e = 0; e < ND; ++e) acc[e] = fmaf(w, v[j][e], acc[e]);
  }
  T* out = reinterpret_cast<T*>(a.out) + qrow * a.o_row + (int64_t)head * a.o_head;
#pragma unroll
  for (int e = 0; e < ND; ++e) {
    const int d = d0 + lane + 64 * e;
    if (d < a.head_dim) out[d] = from_f32<T>(acc[e] * inv);
  }
}

// The merge of four (row, q head) pairs by a workgroup of 4 waves: heads
// 4 * head4 .. + 3 of one row.
template <typename T, int ND>
__device__ __forceinline__ void decode_merge(const DecodeArgs& a, int head4, int64_t row) {
  const int lane = threadIdx.x & 63;
  const int head = head4 * 4 + (threadIdx.x >> 6);
  if (head >= a.q_heads) return;
  int64_t trow, qrow;
  const int n = row_length(row, a, &trow, &qrow);
  if (n <= 0) return;
  const Partition P = partition(n, a);
  if (P.nsplit <= 1) return;
  merge_partials<T, ND>(a, row, head, qrow, P.nsplit, lane, 0);
}

}  // namespace vrh

// Decode rows over a paged cache (paged_decode.hip). With `later` (rows that fit one
// launch) the merge of the split partials is left to the caller: *later_blocks
// workgroups of 4 waves, block b running decode_merge of heads 4 * (b % ceil(q_heads
// / 4)) of row b / ceil(q_heads / 4); untouched when no row can have a second split.
int vrh_decode_rows(int dtype, void* out, const void* q, const void* key_cache,
                    const void* value_cache, const int32_t* block_tables,
                    const int32_t* context_lengths, const int32_t* cu_q, int32_t num_seqs,
                    int32_t expand_e, int64_t rows, int32_t q_heads, int32_t kv_heads,
                    int32_t head_dim, int32_t block_size, int32_t table_width,
                    int64_t table_stride, int64_t q_row_stride, int64_t q_head_stride,
                    int64_t out_row_stride, int64_t out_head_stride, int64_t k_block_stride,
                    int64_t k_token_stride, int64_t k_head_stride, int64_t v_block_stride,
                    int64_t v_token_stride, int64_t v_head_stride, int32_t window,
                    void* workspace, size_t workspace_bytes, hipStream_t s, const char* who,
                    vrh::DecodeArgs* later = nullptr, unsigned* later_blocks = nullptr);
