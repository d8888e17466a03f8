// Row lengths and segment lookup shared by the decode kernels (decode.hip, decode_mfma.hip).
#pragma once
#include "kernels.h"

namespace orin {

// Segment s with cu[s] <= row < cu[s+1] (binary search over n_seg segments).
__device__ __forceinline__ int find_segment(const int* cu, int n_seg, int row) {
  int lo = 0, hi = n_seg - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (cu[mid] <= row) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// Number of keys row `row` attends to.  A device-side length (gpu pos, context_lens) longer
// than the launch was sized for (len_cap, from the host's max_context_len / max_seq_len) is
// an argument error that the host cannot see; the kernels then write NaN for that row
// rather than attend over a truncated prefix.
__device__ __forceinline__ int row_len(const DecodeArgs& a, int row) {
  if (a.cu_seqlens) {
    const int s = find_segment(a.cu_seqlens, a.n_seg, row);
    return a.cu_seqlens[s + 1] - a.cu_seqlens[s];
  }
  if (a.lens) return a.lens[row] + a.len_add;
  return a.len_base + row * a.len_step;
}

// Tokens per split of a single-sequence decode over `len` rows, at most 2^splits_log2 splits.
// The splits follow the row's actual length, which only the device knows when the position is
// there, so that a launch sized for a long cache spreads a short row over the chip too: one CU
// streams about 36 GB/s, and 1338 rows of 8 kv heads (fp16, d 128, cache of 4096) take 7.4 us as
// 64-token splits, 8.6 as 128, 10.3 as 256 (merge included).  Up to 128 rows one split is kept:
// its launch needs no merge.
__host__ __device__ inline int single_row_split_tokens(int len, int splits_log2) {
  if (len <= 128) return 128;
  const int st = (((len + (1 << splits_log2) - 1) >> splits_log2) + 15) & ~15;
  return st < 32 ? 32 : st;
}

// Split size of a row of `len` tokens.
__device__ __forceinline__ int row_split_tokens(const DecodeArgs& a, int len) {
  return a.dyn_splits_log2 >= 0 ? single_row_split_tokens(len, a.dyn_splits_log2) : a.split_tokens;
}

}  // namespace orin
