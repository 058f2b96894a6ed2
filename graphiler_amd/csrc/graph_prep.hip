// Graph preparation on the device: stable grouping of an edge list by one
// endpoint (or of items by type) into pointer / neighbour / edge-id columns,
// the layout python/graphiler/utils/setup.py:116-146 builds on the host with a
// Python prefix-sum loop and DGL's in_edges / out_edges.
//
// Order contract (what the operators rely on): slots of one key are contiguous,
// keys ascend, and inside a key the edge ids ascend, i.e. a STABLE sort of the
// edge ids by key.  Steps, all on the caller's stream:
//   1. narrow the int64 keys to int32 and check their range,
//   2. stable LSD radix sort of (key, edge id) pairs over the bits the keys
//      use (the counting passes below; above 16 M edges the rocPRIM device radix
//      sort, a library sort like a library GEMM),
//   3. pointer[v] = first slot whose key is >= v, by binary search in the sorted
//      keys (no counting with atomics: a hub node of a power-law graph would
//      serialise tens of thousands of them on one address),
//   4. gather the other endpoint through the sorted edge ids.
#include "common.h"

#include <cstring>

#include <rocprim/device/device_radix_sort.hpp>

namespace ga {
namespace {

__global__ __launch_bounds__(kBlock) void prep_keys_kernel(
    const int64_t *__restrict__ key, int64_t n_keys, int64_t n_items,
    int32_t *__restrict__ key32, int32_t *__restrict__ ids,
    int32_t *__restrict__ status) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n_items) return;
  int64_t k = key[i];
  if (k < 0 || k >= n_keys) {
    *status = 1;          // every writer stores the same value
    k = 0;                // keeps the remaining steps inside their arrays
  }
  key32[i] = (int32_t)k;
  ids[i] = (int32_t)i;
}

// first index with key_sorted[index] >= v
template <typename K>
__device__ __forceinline__ int64_t first_not_below(const K *__restrict__ key_sorted, int64_t n_items,
                                                   int64_t v) {
  int64_t lo = 0, hi = n_items;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if ((int64_t)key_sorted[mid] < v) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// pointer[v] = number of items with key < v, v in [0, n_keys]
template <typename K>
__global__ __launch_bounds__(kBlock) void pointer_kernel(
    const K *__restrict__ key_sorted, int64_t n_keys, int64_t n_items,
    int32_t *__restrict__ pointer) {
  const int64_t v = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (v > n_keys) return;
  pointer[v] = (int32_t)first_not_below(key_sorted, n_items, v);
}

__global__ __launch_bounds__(kBlock) void gather_other_kernel(
    const int64_t *__restrict__ other, const int32_t *__restrict__ ids,
    int64_t n_items, int32_t *__restrict__ nbr) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n_items) return;
  nbr[i] = (int32_t)other[ids[i]];
}

__global__ __launch_bounds__(kBlock) void fill_zero_kernel(int32_t *p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) p[i] = 0;
}

__global__ __launch_bounds__(kBlock) void group_zero_kernel(uint4 *p, int64_t n, int32_t *a, int32_t *b) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) p[i] = make_uint4(0u, 0u, 0u, 0u);
  if (i == 0) *a = *b = 0;
}

// Pointer of items that are already sorted by key: item i writes the entries of the keys
// after its predecessor's up to its own, the last item those after its own as well.  No
// sort, no search: every key is read once (672,884 keys: a stable sort and the comparison
// behind it took 185 us of launches and two waits).  status[0]: a key outside [0, n_keys),
// status[1]: a key below its predecessor; nothing is written for such an item.  A lane writes
// a gap between two keys alone, so there are at most kSerialKeys of them; above, WRITE is
// false and pointer_kernel searches every entry.
constexpr int64_t kSerialKeys = 4096;
template <bool WRITE>
__global__ __launch_bounds__(kBlock) void sorted_pointer_kernel(
    const int64_t *__restrict__ key, int64_t n_keys, int64_t n_items,
    int32_t *__restrict__ pointer, int32_t *__restrict__ status) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (WRITE && n_items == 0 && i <= n_keys) pointer[i] = 0;
  if (i >= n_items) return;
  const int64_t k = key[i], before = i > 0 ? key[i - 1] : -1;
  const bool outside = k < 0 || k >= n_keys, unsorted = i > 0 && k < before;
  if (outside) status[0] = 1;       // every writer stores the same value
  if (unsorted) status[1] = 1;
  if (!WRITE || outside || unsorted) return;
  for (int64_t v = before < -1 ? 0 : before + 1; v <= k; ++v) pointer[v] = (int32_t)i;
  if (i == n_items - 1)
    for (int64_t v = k + 1; v <= n_keys; ++v) pointer[v] = (int32_t)n_items;
}

// ---- slots ordered by classes of their sources ---------------------------------
// A stable partition of the in-adjacency's slots into up to kMaxClasses classes of source
// nodes: every wavefront counts the classes of kPartSlots consecutive slots (ballots),
// one workgroup turns the counts into positions, every wavefront writes its slots.  A
// class is made of blocks of kClassRows node ids, so that the rows of a class spread over
// all memory channels (with src % classes every class of 256-byte rows lies in two of
// sixteen), and the blocks are dealt by a multiplicative hash, so that popular ids, which
// graph generators and loaders put side by side, meet all classes.
constexpr int kMaxClasses = 8;
constexpr int kPartSlots = 4096;
constexpr int kClassRowsShift = 6;
__device__ __forceinline__ int source_class(int32_t src, int class_shift) {
  return (int)((((uint32_t)src >> kClassRowsShift) * 0x9E3779B1u) >> (32 - class_shift));
}

__global__ __launch_bounds__(kBlock) void class_count_kernel(
    const int32_t *__restrict__ nbr, int64_t n_edges, int class_shift, int64_t n_units,
    int32_t *__restrict__ counts) {
  const int64_t unit = (int64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
  if (unit >= n_units) return;
  const int lane = threadIdx.x & (kWave - 1);
  int n[kMaxClasses] = {};
  for (int i = 0; i < kPartSlots; i += kWave) {
    const int64_t j = unit * kPartSlots + i + lane;
    const int c = j < n_edges ? source_class(nbr[j], class_shift) : -1;
#pragma unroll
    for (int k = 0; k < kMaxClasses; ++k) n[k] += __popcll(__ballot(c == k));
  }
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < kMaxClasses; ++k)
      if (k >> class_shift == 0) counts[k * n_units + unit] = n[k];
  }
}

// counts <- their exclusive prefix sums, in place, by one workgroup
__global__ __launch_bounds__(1024) void class_scan_kernel(int32_t *__restrict__ counts, int64_t n) {
  __shared__ int32_t wave_sum[1024 / kWave];
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  int32_t before = 0;                    // all items of earlier rounds
  for (int64_t base = 0; base < n; base += 1024) {
    const int64_t i = base + threadIdx.x;
    const int32_t v = i < n ? counts[i] : 0;
    int32_t incl = v;
    for (int off = 1; off < kWave; off <<= 1) {
      const int32_t o = __shfl_up(incl, off);
      if (lane >= off) incl += o;
    }
    if (lane == kWave - 1) wave_sum[wave] = incl;
    __syncthreads();
    int32_t in_front = before, all = 0;
    for (int w = 0; w < 1024 / kWave; ++w) {
      if (w < wave) in_front += wave_sum[w];
      all += wave_sum[w];
    }
    if (i < n) counts[i] = in_front + incl - v;
    before += all;
    __syncthreads();
  }
}

__global__ __launch_bounds__(kBlock) void class_scatter_kernel(
    const int32_t *__restrict__ row_of_slot, const int32_t *__restrict__ nbr, int64_t n_rows,
    int64_t n_edges, int class_shift, int64_t n_units, const int32_t *__restrict__ first,
    int32_t *__restrict__ rows_out, int32_t *__restrict__ nbr_out) {
  const int64_t unit = (int64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
  if (unit >= n_units) return;
  const int lane = threadIdx.x & (kWave - 1);
  const uint64_t below = ((uint64_t)1 << lane) - 1;
  int32_t pos[kMaxClasses];
#pragma unroll
  for (int k = 0; k < kMaxClasses; ++k)
    pos[k] = k >> class_shift == 0 ? first[k * n_units + unit] : 0;
  for (int i = 0; i < kPartSlots; i += kWave) {
    const int64_t j = unit * kPartSlots + i + lane;
    int32_t src = 0, row = 0;
    int c = -1;
    if (j < n_edges) {
      src = nbr[j];
      row = row_of_slot[j];
      c = source_class(src, class_shift);
    }
    int32_t p = 0;
#pragma unroll
    for (int k = 0; k < kMaxClasses; ++k) {
      const uint64_t m = __ballot(c == k);
      if (c == k) p = pos[k] + __popcll(m & below);
      pos[k] += __popcll(m);
    }
    if (c >= 0) {
      rows_out[p] = (int32_t)(c * n_rows + row);
      nbr_out[p] = src;
    }
  }
}

// Row lengths as fp32, at least `least`: the degrees a layer's norm is made of, one launch
// instead of a subtraction, a conversion and a clamp (5 us each on 2,708 nodes, host included).
__global__ __launch_bounds__(kBlock) void row_lengths_kernel(
    const int32_t *__restrict__ pointer, int64_t n_rows, float least, float *__restrict__ out) {
  const int64_t v = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (v < n_rows) out[v] = fmaxf((float)(pointer[v + 1] - pointer[v]), least);
}

// Rows and their items by the power of two below a row's length: integers, so the order in
// which the workgroups add them does not matter.
__global__ __launch_bounds__(kBlock) void degree_buckets_kernel(
    const int32_t *__restrict__ pointer, int64_t n_rows, unsigned long long *__restrict__ buckets) {
  __shared__ unsigned long long all[2 * GA_DEGREE_BUCKETS];
  if (threadIdx.x < 2 * GA_DEGREE_BUCKETS) all[threadIdx.x] = 0;
  __syncthreads();
  for (int64_t v = (int64_t)blockIdx.x * kBlock + threadIdx.x; v < n_rows;
       v += (int64_t)gridDim.x * kBlock) {
    const int32_t d = pointer[v + 1] - pointer[v];
    if (d <= 0) continue;
    const int b = 31 - __clz(d);
    atomicAdd(&all[b], 1ull);
    atomicAdd(&all[GA_DEGREE_BUCKETS + b], (unsigned long long)d);
  }
  __syncthreads();
  if (threadIdx.x < 2 * GA_DEGREE_BUCKETS && all[threadIdx.x])
    atomicAdd(&buckets[threadIdx.x], all[threadIdx.x]);
}

// ---- stable grouping by counting: up to two keys (both endpoints) in the same launches ------
// LSD radix passes of up to kDigitBits bits, two launches each.  A workgroup owns a tile of
// consecutive items.  group_count_kernel counts its digits and adds them to the counts of its
// span of workgroups; group_scatter_kernel finds where its items of a digit go from the counts
// of the spans and of the workgroups of its own span, ranks its items (ballots inside a
// wavefront, the wavefronts' counts in LDS), orders them in LDS, so that the items of a digit
// leave side by side (without that 110 instead of 72 us below), and moves them; the last pass
// gathers the other endpoint as well.  Integers throughout: the order of the atomic additions
// does not matter.
// Small lists are bound by launches that wait for one another: six for two passes over both
// keys, where the merge sort that the library takes below a million items is 23 a key.  Large
// ones by the traffic of the passes, of which a digit of ten bits saves one.  Both keys,
// library sort -> here, us: 12,000 edges 66 -> 29, 200,000 140 -> 41, 672,884 321 -> 69,
// 1 M 361 -> 91, 2 M 321 -> 172, 4 M 460 -> 411, 11.6 M 1175 -> 1029, 24 M 2416 -> 2220,
// 62 M 5835 -> 6245.
constexpr int kDigitBits = 10;
constexpr int kMaxBins = 1 << kDigitBits;
constexpr int kGroupThreads = 512;
constexpr int kGroupWaves = kGroupThreads / kWave;
// Items of a thread: four where eight leave the chip idle (200,000 items 41 : 50 us, 672,884
// 68 : 72, 1 M 105 : 91; sixteen are slower up to 2 M and equal above).
constexpr int64_t kShortTileItems = 700'000;
// Above it the library's sort: twice the scratch is not worth the last 8 % at 24 M.
constexpr int64_t kCountingItems = 16 << 20;

struct GroupSide {
  const int64_t *key, *other;
  int32_t *pointer, *nbr, *eid, *status;
  uint2 *pairs[2];                // (key, item) between passes
  int32_t *key_sorted, *counts, *spans;
};
struct GroupArgs {
  GroupSide side[2];
  int64_t n_keys, n_items;
  int shift, bits, span_shift, n_spans, pass;
  bool first, last;
};

// The key of an item in pass `pass`; out of range (first pass only): 0 and the status is set,
// which keeps the remaining steps inside their arrays.
__device__ __forceinline__ uint2 group_item(const GroupArgs &A, const GroupSide &S, int64_t i) {
  if (!A.first) return S.pairs[(A.pass - 1) & 1][i];
  const int64_t k = S.key[i];
  if (k < 0 || k >= A.n_keys) {
    *S.status = 1;                // every writer stores the same value
    return make_uint2(0u, (uint32_t)i);
  }
  return make_uint2((uint32_t)k, (uint32_t)i);
}

template <int ROUNDS>
__global__ __launch_bounds__(kGroupThreads) void group_count_kernel(GroupArgs A) {
  __shared__ int32_t hist[kMaxBins];
  const GroupSide &S = A.side[blockIdx.y];
  const int bins = 1 << A.bits;
  for (int b = threadIdx.x; b < bins; b += kGroupThreads) hist[b] = 0;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * (ROUNDS * kGroupThreads);
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    const int64_t i = base + r * kGroupThreads + threadIdx.x;
    if (i < A.n_items) atomicAdd(&hist[(group_item(A, S, i).x >> A.shift) & (bins - 1)], 1);
  }
  __syncthreads();
  int32_t *span = S.spans + ((int64_t)A.pass * A.n_spans + (blockIdx.x >> A.span_shift)) * kMaxBins;
  for (int b = threadIdx.x; b < bins; b += kGroupThreads) {
    S.counts[(int64_t)blockIdx.x * bins + b] = hist[b];
    if (hist[b]) atomicAdd(&span[b], hist[b]);
  }
}

template <int ROUNDS>
__global__ __launch_bounds__(kGroupThreads) void group_scatter_kernel(GroupArgs A) {
  constexpr int kPer = kMaxBins / kGroupThreads;
  __shared__ int32_t place[kGroupWaves][kMaxBins], away[kMaxBins];
  __shared__ uint2 ordered[ROUNDS * kGroupThreads];
  __shared__ int2 wave_sum[kPer][kGroupWaves];
  const GroupSide &S = A.side[blockIdx.y];
  const int bins = 1 << A.bits;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  for (int b = lane; b < bins; b += kWave) place[wave][b] = 0;
  // my items: ROUNDS times 64 consecutive ones per wavefront
  uint2 item[ROUNDS];
  const int64_t base = (int64_t)blockIdx.x * (ROUNDS * kGroupThreads) + wave * (kWave * ROUNDS) + lane;
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    const int64_t i = base + r * kWave;
    item[r] = i < A.n_items ? group_item(A, S, i) : make_uint2(0u, 0u);
  }
  // items before mine of every digit: thread t has the digits t and t + kGroupThreads
  int32_t before[kPer], total[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    before[k] = total[k] = 0;
    const int b = threadIdx.x + k * kGroupThreads;
    if (b < bins) {
      const int my_span = blockIdx.x >> A.span_shift;
      const int32_t *span = S.spans + (int64_t)A.pass * A.n_spans * kMaxBins + b;
#pragma unroll 8
      for (int g = 0; g < A.n_spans; ++g) {
        const int32_t c = span[(int64_t)g * kMaxBins];
        total[k] += c;
        before[k] += g < my_span ? c : 0;
      }
#pragma unroll 8
      for (int g = my_span << A.span_shift; g < (int)blockIdx.x; ++g)
        before[k] += S.counts[(int64_t)g * bins + b];
    }
  }
  // ranks: items of my wavefront with the same digit in front of each
  const uint64_t below = ((uint64_t)1 << lane) - 1;
  uint32_t rank[ROUNDS];
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    const bool live = base + r * kWave < A.n_items;
    const int digit = (item[r].x >> A.shift) & (bins - 1);
    uint64_t same = __ballot(live);
    for (int b = 0; b < A.bits; ++b) {
      const uint64_t set = __ballot(digit >> b & 1);
      same &= digit >> b & 1 ? set : ~set;
    }
    const int32_t seen = place[wave][digit];
    rank[r] = seen + __popcll(same & below);
    if (live && (same >> lane >> 1) == 0) place[wave][digit] = seen + __popcll(same);
  }
  __syncthreads();
  // the workgroup's items in the order they leave in: first place of every digit in it and of
  // every wavefront's items of it, and how far from there the digit's items lie in the result
  int32_t carry = 0, local_carry = 0;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int b = threadIdx.x + k * kGroupThreads;
    int32_t local = 0;
    if (b < bins)
      for (int w = 0; w < kGroupWaves; ++w) local += place[w][b];
    int32_t incl = total[k], local_incl = local;
    for (int off = 1; off < kWave; off <<= 1) {
      const int32_t o = __shfl_up(incl, off), l = __shfl_up(local_incl, off);
      if (lane >= off) { incl += o; local_incl += l; }
    }
    if (lane == kWave - 1) wave_sum[k][wave] = make_int2(incl, local_incl);
    __syncthreads();
    int32_t at = carry + incl - total[k] + before[k], local_at = local_carry + local_incl - local;
    for (int w = 0; w < kGroupWaves; ++w) {
      const int2 c = wave_sum[k][w];
      if (w < wave) { at += c.x; local_at += c.y; }
      carry += c.x;
      local_carry += c.y;
    }
    if (b < bins) {
      away[b] = at - local_at;
      for (int w = 0; w < kGroupWaves; ++w) {
        const int32_t c = place[w][b];
        place[w][b] = local_at;
        local_at += c;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r)
    if (base + r * kWave < A.n_items)
      ordered[place[wave][(item[r].x >> A.shift) & (bins - 1)] + rank[r]] = item[r];
  __syncthreads();
  const int64_t left = A.n_items - (int64_t)blockIdx.x * (ROUNDS * kGroupThreads);
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    const int i = r * kGroupThreads + threadIdx.x;
    if (i >= left) break;
    const uint2 v = ordered[i];
    const int64_t p = i + away[(v.x >> A.shift) & (bins - 1)];
    if (A.last) {
      S.key_sorted[p] = (int32_t)v.x;
      S.eid[p] = (int32_t)v.y;
      if (S.nbr) S.nbr[p] = (int32_t)S.other[v.y];
    } else {
      S.pairs[A.pass & 1][p] = v;
    }
  }
}

__global__ __launch_bounds__(kBlock) void group_pointer_kernel(GroupArgs A) {
  const GroupSide &S = A.side[blockIdx.y];
  const int64_t v = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (v > A.n_keys) return;
  S.pointer[v] = (int32_t)first_not_below(S.key_sorted, A.n_items, v);
}

inline size_t round_up(size_t v) { return (v + 255) & ~(size_t)255; }

struct PrepLayout {
  bool counting;                              // the kernels above, else the library's sort
  size_t zeroed, zeroed_bytes;                // the spans' counts of all passes, both sides
  size_t pairs[2], counts;                    // per side, at side * side_bytes
  size_t key32, key_sorted, ids, temp, side_bytes, total;
  size_t temp_bytes;
  int bits, passes, rounds, blocks, span_shift, spans;
};

int end_bit_for(int64_t n_keys) {
  int bits = 1;
  while (bits < 31 && ((int64_t)1 << bits) < n_keys) ++bits;
  return bits;
}

// Sizes only; nothing is launched (rocPRIM's calls with a null temporary
// buffer just report what they need).
int prep_layout(int64_t n_keys, int64_t n_items, int sides, PrepLayout &L) {
  L.counting = n_items <= kCountingItems;
  L.bits = end_bit_for(n_keys);
  L.passes = (L.bits + kDigitBits - 1) / kDigitBits;
  L.rounds = n_items <= kShortTileItems ? 4 : 8;
  const int64_t tile = (int64_t)L.rounds * kGroupThreads;
  L.blocks = (int)((n_items + tile - 1) / tile);
  L.span_shift = 0;
  while ((1 << 2 * L.span_shift) < L.blocks) ++L.span_shift;
  L.spans = (L.blocks + (1 << L.span_shift) - 1) >> L.span_shift;
  L.temp_bytes = 0;
  size_t off = 0;
  L.zeroed = 0;
  L.zeroed_bytes = L.counting ? (size_t)sides * L.passes * L.spans * kMaxBins * 4 : 0;
  off += round_up(L.zeroed_bytes);
  const size_t start = off;
  if (L.counting) {
    for (int k = 0; k < 2; ++k) {
      L.pairs[k] = off;
      off += L.passes > k + 1 ? round_up((size_t)n_items * 8) : 0;
    }
    L.counts = off;      off += round_up((size_t)L.blocks * kMaxBins * 4);
    L.key_sorted = off;  off += round_up((size_t)n_items * 4);
    L.side_bytes = off - start;
    L.total = start + (size_t)sides * L.side_bytes;
    if (L.total == 0) L.total = 256;
    return GA_OK;
  }
  size_t sort_bytes = 0;
  int32_t *k = nullptr;
  hipError_t e = rocprim::radix_sort_pairs(nullptr, sort_bytes, k, k, k, k, (size_t)n_items, 0, L.bits);
  if (e != hipSuccess) return (int)e;
  L.temp_bytes = sort_bytes;
  L.key32 = off;       off += round_up((size_t)n_items * 4);
  L.key_sorted = off;  off += round_up((size_t)n_items * 4);
  L.ids = off;         off += round_up((size_t)n_items * 4);
  L.temp = off;        off += round_up(L.temp_bytes);
  L.side_bytes = 0;                           // one side after the other
  L.total = off;
  return GA_OK;
}

// sides keys grouped at once; S has the callers' arrays
int group_sides(GroupSide (&S)[2], int sides, int64_t n_keys, int64_t n_items, void *workspace,
                size_t workspace_bytes, hipStream_t s) {
  PrepLayout L;
  const int rc = prep_layout(n_keys, n_items, sides, L);
  if (rc != GA_OK) return rc;
  if (!workspace || workspace_bytes < L.total || !aligned(workspace, 256)) return GA_EWORKSPACE;
  char *ws = (char *)workspace;
  auto blocks = [](int64_t threads) { return (unsigned)((threads + kBlock - 1) / kBlock); };
  // the status words start at 0 (a fill kernel rather than a memset node keeps the
  // sequence capturable)
  hipLaunchKernelGGL(group_zero_kernel, dim3(blocks((int64_t)(L.zeroed_bytes / 16) + 1)), dim3(kBlock), 0, s,
                     (uint4 *)(ws + L.zeroed), (int64_t)(L.zeroed_bytes / 16), S[0].status,
                     S[sides - 1].status);
  if (L.counting) {
    GroupArgs A{};
    for (int k = 0; k < sides; ++k) {
      char *base = ws + k * L.side_bytes;
      S[k].pairs[0] = (uint2 *)(base + L.pairs[0]);
      S[k].pairs[1] = (uint2 *)(base + L.pairs[1]);
      S[k].counts = (int32_t *)(base + L.counts);
      S[k].key_sorted = (int32_t *)(base + L.key_sorted);
      S[k].spans = (int32_t *)(ws + L.zeroed) + (size_t)k * L.passes * L.spans * kMaxBins;
      A.side[k] = S[k];
    }
    A.n_keys = n_keys;
    A.n_items = n_items;
    A.span_shift = L.span_shift;
    A.n_spans = L.spans;
    for (int pass = 0; pass < L.passes && n_items > 0; ++pass) {
      A.pass = pass;
      A.shift = pass == 0 ? 0 : A.shift + A.bits;
      A.bits = (L.bits - A.shift + L.passes - pass - 1) / (L.passes - pass);
      A.first = pass == 0;
      A.last = pass == L.passes - 1;
      const dim3 grid((unsigned)L.blocks, (unsigned)sides);
      if (L.rounds == 4) {
        hipLaunchKernelGGL(group_count_kernel<4>, grid, dim3(kGroupThreads), 0, s, A);
        hipLaunchKernelGGL(group_scatter_kernel<4>, grid, dim3(kGroupThreads), 0, s, A);
      } else {
        hipLaunchKernelGGL(group_count_kernel<8>, grid, dim3(kGroupThreads), 0, s, A);
        hipLaunchKernelGGL(group_scatter_kernel<8>, grid, dim3(kGroupThreads), 0, s, A);
      }
    }
    hipLaunchKernelGGL(group_pointer_kernel, dim3(blocks(n_keys + 1), (unsigned)sides), dim3(kBlock), 0,
                       s, A);
    return launch_status();
  }
  int32_t *key32 = (int32_t *)(ws + L.key32);
  int32_t *key_sorted = (int32_t *)(ws + L.key_sorted);
  int32_t *ids = (int32_t *)(ws + L.ids);
  for (int k = 0; k < sides; ++k) {
    hipLaunchKernelGGL(prep_keys_kernel, dim3(blocks(n_items)), dim3(kBlock), 0, s, S[k].key, n_keys,
                       n_items, key32, ids, S[k].status);
    size_t tb = L.temp_bytes;
    hipError_t e = rocprim::radix_sort_pairs(ws + L.temp, tb, key32, key_sorted, ids, S[k].eid,
                                             (size_t)n_items, 0, L.bits, s);
    if (e != hipSuccess) return (int)e;
    hipLaunchKernelGGL(pointer_kernel<int32_t>, dim3(blocks(n_keys + 1)), dim3(kBlock), 0, s,
                       key_sorted, n_keys, n_items, S[k].pointer);
    if (S[k].nbr)
      hipLaunchKernelGGL(gather_other_kernel, dim3(blocks(n_items)), dim3(kBlock), 0, s, S[k].other,
                         S[k].eid, n_items, S[k].nbr);
  }
  return launch_status();
}

}  // namespace
}  // namespace ga

extern "C" {

size_t ga_group_edges_workspace_bytes(int64_t n_keys, int64_t n_items) {
  if (n_keys < 0 || n_items < 0 || n_keys > 0x7ffffffe || n_items > 0x7fffffff) return 0;
  ga::PrepLayout L;
  if (ga::prep_layout(n_keys, n_items, 1, L) != GA_OK) return 0;
  return L.total;
}

size_t ga_group_edges_both_workspace_bytes(int64_t n_keys, int64_t n_items) {
  if (n_keys < 0 || n_items < 0 || n_keys > 0x7ffffffe || n_items > 0x7fffffff) return 0;
  ga::PrepLayout L;
  if (ga::prep_layout(n_keys, n_items, 2, L) != GA_OK) return 0;
  return L.total;
}

int ga_group_edges(const int64_t *key, const int64_t *other, int64_t n_keys,
                   int64_t n_items, int32_t *pointer, int32_t *nbr, int32_t *eid,
                   int32_t *status, void *workspace, size_t workspace_bytes,
                   ga_stream_t stream) {
  using namespace ga;
  if (n_keys < 0 || n_items < 0 || n_keys > 0x7ffffffe || n_items > 0x7fffffff)
    return GA_EINVAL;
  if (!pointer || !status) return GA_EINVAL;
  if (n_items > 0 && (!key || !eid || n_keys == 0)) return GA_EINVAL;
  if (nbr && !other) return GA_EINVAL;
  GroupSide S[2] = {};
  S[0].key = key; S[0].other = other;
  S[0].pointer = pointer; S[0].nbr = nbr; S[0].eid = eid; S[0].status = status;
  return group_sides(S, 1, n_keys, n_items, workspace, workspace_bytes, (hipStream_t)stream);
}

int ga_group_edges_both(const int64_t *src, const int64_t *dst, int64_t n_keys, int64_t n_items,
                        int32_t *in_pointer, int32_t *in_nbr, int32_t *in_eid,
                        int32_t *out_pointer, int32_t *out_nbr, int32_t *out_eid,
                        int32_t *status, void *workspace, size_t workspace_bytes,
                        ga_stream_t stream) {
  using namespace ga;
  if (n_keys < 0 || n_items < 0 || n_keys > 0x7ffffffe || n_items > 0x7fffffff)
    return GA_EINVAL;
  if (!in_pointer || !out_pointer || !status) return GA_EINVAL;
  if (n_items > 0 && (!src || !dst || !in_nbr || !in_eid || !out_nbr || !out_eid || n_keys == 0))
    return GA_EINVAL;
  GroupSide S[2] = {};
  S[0].key = dst; S[0].other = src;
  S[0].pointer = in_pointer; S[0].nbr = in_nbr; S[0].eid = in_eid; S[0].status = status;
  S[1].key = src; S[1].other = dst;
  S[1].pointer = out_pointer; S[1].nbr = out_nbr; S[1].eid = out_eid; S[1].status = status + 1;
  return group_sides(S, 2, n_keys, n_items, workspace, workspace_bytes, (hipStream_t)stream);
}

int ga_row_lengths(const int32_t *pointer, int64_t n_rows, float least, float *out,
                   ga_stream_t stream) {
  using namespace ga;
  if (n_rows < 0 || n_rows > 0x7ffffffe || (n_rows > 0 && (!pointer || !out))) return GA_EINVAL;
  if (!aligned(pointer, 4) || !aligned(out, 4)) return GA_EALIGN;
  if (n_rows == 0) return GA_OK;
  hipLaunchKernelGGL(row_lengths_kernel, dim3((unsigned)((n_rows + kBlock - 1) / kBlock)), dim3(kBlock),
                     0, (hipStream_t)stream, pointer, n_rows, least, out);
  return launch_status();
}

int ga_degree_buckets(const int32_t *pointer, int64_t n_rows, int64_t *buckets, ga_stream_t stream) {
  using namespace ga;
  if (n_rows < 0 || n_rows > 0x7ffffffe || !buckets || (n_rows > 0 && !pointer)) return GA_EINVAL;
  if (!aligned(buckets, 8) || !aligned(pointer, 4)) return GA_EALIGN;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(fill_zero_kernel, dim3(1), dim3(kBlock), 0, s, (int32_t *)buckets,
                     (int64_t)(4 * GA_DEGREE_BUCKETS));
  const int64_t blocks = (n_rows + kBlock - 1) / kBlock;
  if (blocks > 0)
    hipLaunchKernelGGL(degree_buckets_kernel, dim3((unsigned)(blocks < 1024 ? blocks : 1024)),
                       dim3(kBlock), 0, s, pointer, n_rows, (unsigned long long *)buckets);
  return launch_status();
}

size_t ga_source_classes_workspace_bytes(int64_t n_edges, int64_t n_classes) {
  if (n_edges < 0 || n_edges > 0x7fffffff || n_classes < 2 || n_classes > ga::kMaxClasses) return 0;
  const size_t units = (size_t)((n_edges + ga::kPartSlots - 1) / ga::kPartSlots);
  return ga::round_up(units * (size_t)n_classes * 4 + 4);
}

int ga_source_classes_build(const int32_t *row_of_slot, const int32_t *nbr, int64_t n_rows,
                            int64_t n_edges, int64_t n_classes, int32_t *pointer, int32_t *rows,
                            int32_t *nbr_out, void *workspace, size_t workspace_bytes,
                            ga_stream_t stream) {
  using namespace ga;
  if (n_rows <= 0 || n_edges <= 0 || n_edges > 0x7fffffff) return GA_EINVAL;
  if (n_classes != 2 && n_classes != 4 && n_classes != 8) return GA_EINVAL;
  if (n_rows * n_classes > 0x7ffffffe) return GA_EUNSUPPORTED;
  if (!row_of_slot || !nbr || !pointer || !rows || !nbr_out) return GA_EINVAL;
  if (!workspace || workspace_bytes < ga_source_classes_workspace_bytes(n_edges, n_classes) ||
      !aligned(workspace, 4))
    return GA_EWORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  const int shift = ilog2_floor((uint64_t)n_classes);
  const int64_t units = (n_edges + kPartSlots - 1) / kPartSlots;
  const unsigned blocks = (unsigned)((units + kBlock / kWave - 1) / (kBlock / kWave));
  int32_t *counts = (int32_t *)workspace;
  hipLaunchKernelGGL(class_count_kernel, dim3(blocks), dim3(kBlock), 0, s, nbr, n_edges, shift,
                     units, counts);
  hipLaunchKernelGGL(class_scan_kernel, dim3(1), dim3(1024), 0, s, counts, units * n_classes);
  hipLaunchKernelGGL(class_scatter_kernel, dim3(blocks), dim3(kBlock), 0, s, row_of_slot, nbr,
                     n_rows, n_edges, shift, units, counts, rows, nbr_out);
  const int64_t n_keys = n_rows * n_classes;
  hipLaunchKernelGGL(pointer_kernel<int32_t>, dim3((unsigned)((n_keys + 1 + kBlock - 1) / kBlock)),
                     dim3(kBlock), 0, s, rows, n_keys, n_edges, pointer);
  return launch_status();
}

int ga_sorted_pointer(const int64_t *key, int64_t n_keys, int64_t n_items, int32_t *pointer,
                      int32_t *status, ga_stream_t stream) {
  using namespace ga;
  if (n_keys < 0 || n_items < 0 || n_keys > 0x7ffffffe || n_items > 0x7fffffff) return GA_EINVAL;
  if (!pointer || !status || (n_items > 0 && !key)) return GA_EINVAL;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(fill_zero_kernel, dim3(1), dim3(kBlock), 0, s, status, (int64_t)2);
  auto blocks = [](int64_t threads) { return dim3((unsigned)((threads + kBlock - 1) / kBlock)); };
  if (n_keys <= kSerialKeys) {
    hipLaunchKernelGGL(sorted_pointer_kernel<true>, blocks(n_items > 0 ? n_items : n_keys + 1),
                       dim3(kBlock), 0, s, key, n_keys, n_items, pointer, status);
    return launch_status();
  }
  if (n_items > 0)
    hipLaunchKernelGGL(sorted_pointer_kernel<false>, blocks(n_items), dim3(kBlock), 0, s, key, n_keys,
                       n_items, pointer, status);
  hipLaunchKernelGGL(pointer_kernel<int64_t>, blocks(n_keys + 1), dim3(kBlock), 0, s, key, n_keys,
                     n_items, pointer);
  return launch_status();
}

}  // extern "C"
