// Rows sorted by type, cut into chunks of one type each (segment_mm.hip, pair_attn.hip).
#pragma once

#include "common.h"

namespace ga {

// Which chunk of which type does this workgroup own?  chunks(t) =
// ceil(rows_t / chunk_rows); workgroup id -> (t, first row, end row).
__device__ __forceinline__ bool locate_chunk(const int32_t *__restrict__ tp,
                                             int n_types, int chunk_rows, int target,
                                             int &type, int &row0, int &row1) {
  __shared__ int scan[kBlock];
  __shared__ int found[3];
  if (!tp) {               // one type; the caller passes the row count as n_types
    type = 0;
    if ((int64_t)target * chunk_rows >= n_types) return false;
    row0 = target * chunk_rows;
    row1 = min(n_types, row0 + chunk_rows);
    return true;
  }
  if (threadIdx.x == 0) found[0] = -1;
  int base = 0;
  for (int t0 = 0; t0 < n_types; t0 += kBlock) {
    const int t = t0 + threadIdx.x;
    int p0 = 0, p1 = 0, cnt = 0;
    if (t < n_types) {
      p0 = tp[t];
      p1 = tp[t + 1];
      cnt = (p1 - p0 + chunk_rows - 1) / chunk_rows;
    }
    __syncthreads();
    scan[threadIdx.x] = cnt;
    __syncthreads();
    for (int off = 1; off < kBlock; off <<= 1) {
      const int add = threadIdx.x >= off ? scan[threadIdx.x - off] : 0;
      __syncthreads();
      scan[threadIdx.x] += add;
      __syncthreads();
    }
    const int incl = base + scan[threadIdx.x];
    const int excl = incl - cnt;
    if (cnt > 0 && target >= excl && target < incl) {
      found[0] = t;
      found[1] = p0 + (target - excl) * chunk_rows;
      found[2] = p1;
    }
    base += scan[kBlock - 1];
    if (base > target) break;   // uniform: every thread sees the same totals
  }
  __syncthreads();
  type = found[0];
  if (type < 0) return false;
  row0 = found[1];
  row1 = min(found[2], row0 + chunk_rows);
  return true;
}

}  // namespace ga
