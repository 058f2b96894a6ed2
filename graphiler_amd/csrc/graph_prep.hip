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
//      use (rocPRIM device radix sort: a library sort, like a library GEMM),
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

// pointer[v] = number of items with key < v, v in [0, n_keys]
template <typename K>
__global__ __launch_bounds__(kBlock) void pointer_kernel(
    const K *__restrict__ key_sorted, int64_t n_keys, int64_t n_items,
    int32_t *__restrict__ pointer) {
  const int64_t v = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (v > n_keys) return;
  int64_t lo = 0, hi = n_items;          // first index with key_sorted[index] >= v
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if ((int64_t)key_sorted[mid] < v) lo = mid + 1; else hi = mid;
  }
  pointer[v] = (int32_t)lo;
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

inline size_t round_up(size_t v) { return (v + 255) & ~(size_t)255; }

struct PrepLayout {
  size_t key32, key_sorted, ids, temp, total;
  size_t temp_bytes;
};

int end_bit_for(int64_t n_keys) {
  int bits = 1;
  while (bits < 31 && ((int64_t)1 << bits) < n_keys) ++bits;
  return bits;
}

// Sizes only; nothing is launched (rocPRIM's calls with a null temporary
// buffer just report what they need).
int prep_layout(int64_t n_keys, int64_t n_items, PrepLayout &L) {
  size_t sort_bytes = 0;
  int32_t *k = nullptr;
  if (n_items > 0) {
    hipError_t e = rocprim::radix_sort_pairs(nullptr, sort_bytes, k, k, k, k,
                                             (size_t)n_items, 0, end_bit_for(n_keys));
    if (e != hipSuccess) return (int)e;
  }
  L.temp_bytes = sort_bytes;
  size_t off = 0;
  L.key32 = off;       off += round_up((size_t)n_items * 4);
  L.key_sorted = off;  off += round_up((size_t)n_items * 4);
  L.ids = off;         off += round_up((size_t)n_items * 4);
  L.temp = off;        off += round_up(L.temp_bytes);
  L.total = off;
  return GA_OK;
}

}  // namespace
}  // namespace ga

extern "C" {

size_t ga_group_edges_workspace_bytes(int64_t n_keys, int64_t n_items) {
  if (n_keys < 0 || n_items < 0 || n_keys > 0x7ffffffe || n_items > 0x7fffffff) return 0;
  ga::PrepLayout L;
  if (ga::prep_layout(n_keys, n_items, L) != GA_OK) return 0;
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
  PrepLayout L;
  const int rc = prep_layout(n_keys, n_items, L);
  if (rc != GA_OK) return rc;
  if (!workspace || workspace_bytes < L.total || !aligned(workspace, 256)) return GA_EWORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  char *ws = (char *)workspace;
  int32_t *key32 = (int32_t *)(ws + L.key32);
  int32_t *key_sorted = (int32_t *)(ws + L.key_sorted);
  int32_t *ids = (int32_t *)(ws + L.ids);
  void *temp = ws + L.temp;

  // the status word starts at 0; a fill kernel rather than a memset node keeps
  // the sequence capturable
  hipLaunchKernelGGL(fill_zero_kernel, dim3(1), dim3(kBlock), 0, s, status, (int64_t)1);
  if (n_items > 0) {
    const int64_t blocks = (n_items + kBlock - 1) / kBlock;
    hipLaunchKernelGGL(prep_keys_kernel, dim3((unsigned)blocks), dim3(kBlock), 0, s, key,
                       n_keys, n_items, key32, ids, status);
    size_t tb = L.temp_bytes;
    hipError_t e = rocprim::radix_sort_pairs(temp, tb, key32, key_sorted, ids, eid,
                                             (size_t)n_items, 0, end_bit_for(n_keys), s);
    if (e != hipSuccess) return (int)e;
  }
  const int64_t pblocks = (n_keys + 1 + kBlock - 1) / kBlock;
  hipLaunchKernelGGL(pointer_kernel<int32_t>, dim3((unsigned)pblocks), dim3(kBlock), 0, s, key_sorted,
                     n_keys, n_items, pointer);
  if (n_items > 0 && nbr) {
    const int64_t blocks = (n_items + kBlock - 1) / kBlock;
    hipLaunchKernelGGL(gather_other_kernel, dim3((unsigned)blocks), dim3(kBlock), 0, s, other,
                       eid, n_items, nbr);
  }
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
