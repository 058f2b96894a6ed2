// Rows sorted by type, cut into chunks of one type each (segment_mm.hip, pair_attn.hip).
#pragma once

#include "common.h"

namespace ga {

// Which chunk of which type does this workgroup own?  chunks(t) =
// ceil(rows_t / chunk_rows); workgroup id -> (t, first row, end row).  Every wavefront finds
// it by itself, 64 types at a time with a prefix sum in registers: it stands in front of
// everything a workgroup does.  As a scan over the workgroup, with two barriers per step, it
// took 5 % of short workgroups (30,500 tiles of the pair attention, 51 types: 709 -> 674 us).
__device__ __forceinline__ bool locate_chunk(const int32_t *__restrict__ tp,
                                             int n_types, int chunk_rows, int target,
                                             int &type, int &row0, int &row1) {
  if (!tp) {               // one type; the caller passes the row count as n_types
    type = 0;
    if ((int64_t)target * chunk_rows >= n_types) return false;
    row0 = target * chunk_rows;
    row1 = min(n_types, row0 + chunk_rows);
    return true;
  }
  const int lane = threadIdx.x & (kWave - 1);
  int base = 0;            // chunks of the types before t0
  for (int t0 = 0; t0 < n_types; t0 += kWave) {
    const int t = t0 + lane;
    int p0 = 0, p1 = 0, cnt = 0;
    if (t < n_types) {
      p0 = tp[t];
      p1 = tp[t + 1];
      cnt = (p1 - p0 + chunk_rows - 1) / chunk_rows;
    }
    int incl = cnt;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const int add = __shfl_up(incl, off);
      if (lane >= off) incl += add;
    }
    incl += base;
    // the first type whose chunks reach past the target
    const uint64_t past = __ballot(incl > target);
    if (past) {
      const int at = __ffsll((long long)past) - 1;
      const int first = __builtin_amdgcn_readlane(p0, at);
      const int in_type = target - __builtin_amdgcn_readlane(incl - cnt, at);
      type = t0 + at;
      row0 = first + in_type * chunk_rows;
      row1 = min(__builtin_amdgcn_readlane(p1, at), row0 + chunk_rows);
      return true;
    }
    base = __builtin_amdgcn_readlane(incl, kWave - 1);
  }
  return false;
}

}  // namespace ga
