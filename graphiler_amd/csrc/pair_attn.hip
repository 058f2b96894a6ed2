// The per-relation part of an HGT layer over the (destination, relation) pairs of a
// graph in one pass (examples/HGT/HGT.py:35-53, one launch for two typed products and
// the attention between them):
//
//   qp[r]  = q[dst(r)] @ A[type(r)]                         A: relation_att, transposed
//   s_i    = <k[src_i], qp[r]>            per head, for the slots i of pair r
//   vp[r]  = sum_i softmax_r(s)_i v[src_i],  lse[r] = log sum_i exp(s_i)
//   m[r]   = vp[r] @ M[type(r)]
//
// The pairs of a destination are weighed by the softmax of their lse afterwards.
//
// A workgroup takes a tile of up to 64 pairs of one relation.  The 64 rows stay in LDS from
// the gathered queries to the stored messages: every wavefront owns a quarter of the
// columns and multiplies all rows with its columns of a relation matrix; between the two
// products a lane group per row (16 bytes per lane) walks the pair's slots, gathering keys
// and values, with an online softmax.  As three launches the pairs' rows crossed memory four
// more times (qp and vp written and read back) and the matrix cores and the gathers never
// ran together.
//
// A matrix's columns are loaded for its product alone: the walk needs neither, and held
// across it (and several tiles per workgroup, whose addresses stay live as well) they made
// 12 of the 16 builds spill at five wavefronts per SIMD and left fp32 rows of 128 features
// at two or three.  72 to 107 registers now, nothing spilled, five to seven wavefronts (four
// where the tile's 35 KB of LDS allow no more).
//
// Bound: the gathered key and value rows, 2 F b bytes per edge, at the rate the caches
// behind the L2s deliver: 2 M edges in 269,078 pairs, 8 x 16 bf16, 1.09 GB of rows, of which
// 0.64 GB pass the L2s in 131 us, 4.9 TB/s (a large copy: 5.0).  The whole pair form (this pass, the transposed matrices, the sum
// of the pairs) as three launches -> matrices held -> now, us:
//   4.68 M edges, 1.95 M pairs: 1 x 64 fp32 1183 -> 809 -> 709, 8 x 16 bf16 1234 -> 699 -> 671,
//     2 x 64 fp32 2619 -> 1653 -> 1343, 2 x 64 bf16 1199 -> 875 -> 697
//   300 k edges, 100 k pairs: 1 x 64 fp32 99 -> 67 -> 59, 8 x 16 bf16 107 -> 63 -> 59
#include "common.h"
#include "typed_chunks.h"

namespace ga {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef short shortx4 __attribute__((ext_vector_type(4)));

constexpr int kPairRows = 64;       // pairs per tile
constexpr int kPairBatch = 4;       // slots whose rows are in flight per lane group: a
                                    // pair has two to eight edges where pairs are used
constexpr int kWaveCount = kBlock / kWave;

struct PairArgs {
  const int32_t *type_pointer;      // (n_types + 1) over the pairs in by_type order
  const int64_t *by_type;           // pair of row r
  const int64_t *dst_by_type;       // destination of row r
  const int32_t *pair_pointer;      // slots of a pair
  const int32_t *nbr;               // source node of a slot
  const void *q, *k, *v, *att, *msg;
  void *m;                          // (P, F), pair order
  float *lse;                       // (P, heads), pair order
  int n_types;
};

// Element of the (heads, D, D) matrices of a type that lane (col, lk) of a block holds
// first, and whether its s-th row belongs to the column's head (D < 16: two heads a block).
template <int D>
__device__ __forceinline__ uint32_t first(int col, int lk) {
  return (uint32_t)((D < 16 ? col & ~15 : col / D * D) + 4 * lk) * D + col % D;
}
template <int D>
__device__ __forceinline__ bool in_block(int col, int lk, int s) {
  return D >= 16 || ((col & ~15) + 4 * lk + s) / D == col / D;
}

// One 16 x 16 block of a product, k blocks of 16: the wavefront's weights and the
// multiplication of 16 tile rows.  D < 16: the block diagonal of two heads.
template <typename T, int D>
struct Block;

template <int D>
struct Block<float, D> {
  static constexpr int KB = D < 16 ? 1 : D / 16;
  float w[KB][4];
  __device__ __forceinline__ void load(const float *W, int col, int lk) {   // W: (heads, D, D) of the type
    const uint32_t at = first<D>(col, lk);
#pragma unroll
    for (int b = 0; b < KB; ++b)
#pragma unroll
      for (int s = 0; s < 4; ++s) w[b][s] = in_block<D>(col, lk, s) ? W[at + (16 * b + s) * D] : 0.0f;
  }
  __device__ __forceinline__ floatx4 mma(const float *row, int k0, int lk) const {
    floatx4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int b = 0; b < KB; ++b) {
      const float4 x = *reinterpret_cast<const float4 *>(row + k0 + 16 * b + 4 * lk);
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x.x, w[b][0], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x.y, w[b][1], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x.z, w[b][2], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w, w[b][3], acc, 0, 0, 0);
    }
    return acc;
  }
};

template <int D>
struct Block<bf16_t, D> {
  static constexpr int KB = D < 16 ? 1 : D / 16;
  uint2 w[KB];
  __device__ __forceinline__ void load(const bf16_t *W, int col, int lk) {
    const uint32_t at = first<D>(col, lk);
#pragma unroll
    for (int b = 0; b < KB; ++b) {
      uint32_t e[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) e[s] = in_block<D>(col, lk, s) ? W[at + (16 * b + s) * D] : 0u;
      w[b] = make_uint2(e[0] | (e[1] << 16), e[2] | (e[3] << 16));
    }
  }
  __device__ __forceinline__ floatx4 mma(const bf16_t *row, int k0, int lk) const {
    floatx4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int b = 0; b < KB; ++b) {
      const uint2 x = *reinterpret_cast<const uint2 *>(row + k0 + 16 * b + 4 * lk);
      acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(shortx4, x),
                                                      __builtin_bit_cast(shortx4, w[b]), acc, 0, 0, 0);
    }
    return acc;
  }
};

template <int LANES>
__device__ __forceinline__ float head_sum(float v) {     // over LANES adjacent lanes
  if constexpr (LANES >= 2) v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));
  if constexpr (LANES >= 4) v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, true));
  if constexpr (LANES >= 8) v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x141, 0xF, 0xF, true));
  if constexpr (LANES >= 16) v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x140, 0xF, 0xF, true));
  return v;
}

template <typename T, int F, int D>
__global__ __launch_bounds__(kBlock, F == 128 && sizeof(T) == 4 ? 4 : 5) void pair_attn_kernel(PairArgs A) {
  constexpr int VEC = 16 / (int)sizeof(T);
  constexpr int LPR = F / VEC;                    // lanes per row
  constexpr int G = kBlock / LPR;                 // lane groups
  constexpr int RPG = kPairRows / G;              // rows a group walks
  constexpr int CB = F / 16 / kWaveCount;         // column blocks per wavefront
  constexpr int H = F / D;
  constexpr int HL = D / VEC < 1 ? 1 : D / VEC;   // lanes per head
  constexpr int LD = F + VEC;                     // row stride of the tile
  static_assert(F % 64 == 0 && HL <= 16 && RPG >= 1, "layout");
  typedef Frag<T, VEC> IO;
  typedef typename IO::raw_t raw_t;
  __shared__ __attribute__((aligned(16))) T tile[kPairRows * LD];
  __shared__ int slot0[kPairRows], slot1[kPairRows], pair_of[kPairRows];
  const T *const q = (const T *)A.q, *const k = (const T *)A.k, *const v = (const T *)A.v;

  int type, row0, row1;
  if (!locate_chunk(A.type_pointer, A.n_types, kPairRows, blockIdx.x, type, row0, row1)) return;

  type = __builtin_amdgcn_readfirstlane(type);
  row0 = __builtin_amdgcn_readfirstlane(row0);
  row1 = __builtin_amdgcn_readfirstlane(row1);

  const int tid = threadIdx.x;
  const int lane64 = tid & (kWave - 1), wave = tid / kWave;
  const int lr = lane64 & 15, lk = lane64 >> 4;
  const int grp = tid / LPR, lane = tid % LPR, f0 = lane * VEC;

  // the wavefront's columns of a relation matrix
  auto columns = [&](const void *W, Block<T, D> (&w)[CB]) {
#pragma unroll
    for (int c = 0; c < CB; ++c)
      w[c].load((const T *)W + (int64_t)type * F * D, (wave * CB + c) * 16 + lr, lk);
  };
  // the tile's rows times the wavefront's columns, in place
  auto product = [&](const Block<T, D> (&w)[CB]) {
    floatx4 acc[CB][kPairRows / 16];
#pragma unroll
    for (int c = 0; c < CB; ++c) {
      const int col0 = (wave * CB + c) * 16;
      const int k0 = D < 16 ? col0 : col0 / D * D;
#pragma unroll
      for (int b = 0; b < kPairRows / 16; ++b) {
        acc[c][b] = w[c].mma(tile + (16 * b + lr) * LD, k0, lk);
        // heads of 64: the rows of all blocks at once would take 64 registers more
        if constexpr (D == 64) __builtin_amdgcn_sched_barrier(0);
      }
    }
    __syncthreads();                       // every wavefront has read all rows
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
      for (int b = 0; b < kPairRows / 16; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          f32_to_elem(acc[c][b][i], tile[(16 * b + 4 * lk + i) * LD + (wave * CB + c) * 16 + lr]);
    __syncthreads();
  };

  const int n = row1 - row0;             // at most kPairRows
  if (tid < kPairRows) {
    const int p = (int)A.by_type[row0 + min(tid, n - 1)];
    pair_of[tid] = p;
    slot0[tid] = A.pair_pointer[p];
    slot1[tid] = A.pair_pointer[p + 1];
  }
#pragma unroll
  for (int i = 0; i < RPG; ++i) {        // rows past the last one repeat it
    const int r = grp + i * G;
    const int64_t d = A.dst_by_type[row0 + min(r, n - 1)];
    *reinterpret_cast<raw_t *>(tile + r * LD + f0) = IO::load(q + d * F + f0);
  }
  {
    Block<T, D> w[CB];
    columns(A.att, w);
    __syncthreads();
    product(w);
  }

  // ---- attention inside the pairs: every G-th row of the tile, one after another (large
  // pairs lie side by side where the relation's popular destinations do) ----
  int r = grp;
  if (r < n) {
    float qf[VEC], acc[VEC], m = -INFINITY, l = 0.0f;
    auto open_row = [&]() {
      IO::widen(*reinterpret_cast<const raw_t *>(tile + r * LD + f0), qf);
#pragma unroll
      for (int e = 0; e < VEC; ++e) acc[e] = 0.0f;
      m = -INFINITY;
      l = 0.0f;
    };
    int pos = slot0[r], end = slot1[r];
    int ids = A.nbr[pos + min(lane & 3, end - 1 - pos)];
    open_row();
    while (true) {
      const int cnt = end - pos;         // at least one
      int nr = r, npos = pos + kPairBatch, nend = end;
      if (cnt <= kPairBatch) {
        nr = r + G;
        if (nr < n) { npos = slot0[nr]; nend = slot1[nr]; }
      }
      // sources of the next batch, whichever row it belongs to
      const int ids_next = nr < n ? A.nbr[npos + min(lane & 3, nend - 1 - npos)] : 0;
      const int g[kPairBatch] = {
          __builtin_amdgcn_update_dpp(0, ids, 0x00, 0xF, 0xF, true),      // quad_perm: lane t
          __builtin_amdgcn_update_dpp(0, ids, 0x55, 0xF, 0xF, true),
          __builtin_amdgcn_update_dpp(0, ids, 0xAA, 0xF, 0xF, true),
          __builtin_amdgcn_update_dpp(0, ids, 0xFF, 0xF, 0xF, true)};
      raw_t kx[kPairBatch], vx[kPairBatch];
#pragma unroll
      for (int t = 0; t < kPairBatch; ++t) {
        kx[t] = vx[t] = raw_t{};
        if (t < cnt) {
          kx[t] = IO::load(k + (int64_t)g[t] * F + f0);
          vx[t] = IO::load(v + (int64_t)g[t] * F + f0);
        }
      }
      float s[kPairBatch], bm = -INFINITY;
#pragma unroll
      for (int t = 0; t < kPairBatch; ++t) {
        float kf[VEC], d = 0.0f;
        IO::widen(kx[t], kf);
#pragma unroll
        for (int e = 0; e < VEC; ++e) d = fmaf(kf[e], qf[e], d);
        d = head_sum<HL>(d);
        s[t] = t < cnt ? d : -INFINITY;
        bm = fmaxf(bm, s[t]);
      }
      // exponentials from 0 while every score is -inf (see the fused GAT aggregation)
      const float nm = fmaxf(m, bm);
      const float ref = nm == -INFINITY ? 0.0f : nm;
      const float sc = __expf(m - ref);
      l *= sc;
#pragma unroll
      for (int e = 0; e < VEC; ++e) acc[e] *= sc;
      m = nm;
#pragma unroll
      for (int t = 0; t < kPairBatch; ++t) {
        if (t < cnt) {
          const float p = __expf(s[t] - ref);
          l += p;
          float vf[VEC];
          IO::widen(vx[t], vf);
#pragma unroll
          for (int e = 0; e < VEC; ++e) acc[e] = fmaf(p, vf[e], acc[e]);
        }
      }
      if (cnt <= kPairBatch) {           // the row is complete: over its own query row
        const float inv = 1.0f / l;
        float o[VEC];
#pragma unroll
        for (int e = 0; e < VEC; ++e) o[e] = acc[e] * inv;
        IO::store(tile + r * LD + f0, o);
        if (f0 % D == 0 || D < VEC) A.lse[(int64_t)pair_of[r] * H + f0 / D] = m + logf(l);
        r = nr;
        if (r >= n) break;
        open_row();
      }
      pos = npos;
      end = nend;
      ids = ids_next;
    }
  }
  {
    Block<T, D> w[CB];
    columns(A.msg, w);
    __syncthreads();
    product(w);
  }
#pragma unroll
  for (int i = 0; i < RPG; ++i) {
    const int row = grp + i * G;
    if (row < n)
      *reinterpret_cast<raw_t *>((T *)A.m + (int64_t)pair_of[row] * F + f0) =
          *reinterpret_cast<const raw_t *>(tile + row * LD + f0);
  }
}

template <typename T, int F, int D>
int launch_pairs(PairArgs &A, int64_t n_pairs, hipStream_t s) {
  const int64_t grid = (n_pairs + kPairRows - 1) / kPairRows + A.n_types;
  if (grid > 0x7fffffff) return GA_EUNSUPPORTED;
  hipLaunchKernelGGL((pair_attn_kernel<T, F, D>), dim3((unsigned)grid), dim3(kBlock), 0, s, A);
  return launch_status();
}

template <typename T>
int launch_pairs_dim(PairArgs &A, int64_t n_pairs, int64_t feat, int64_t dim, hipStream_t s) {
  if (feat == 64) {
    if (dim == 8) return launch_pairs<T, 64, 8>(A, n_pairs, s);
    if (dim == 16) return launch_pairs<T, 64, 16>(A, n_pairs, s);
    if (dim == 32) return launch_pairs<T, 64, 32>(A, n_pairs, s);
    if (dim == 64) return launch_pairs<T, 64, 64>(A, n_pairs, s);
  } else if (feat == 128) {
    if (dim == 8) return launch_pairs<T, 128, 8>(A, n_pairs, s);
    if (dim == 16) return launch_pairs<T, 128, 16>(A, n_pairs, s);
    if (dim == 32) return launch_pairs<T, 128, 32>(A, n_pairs, s);
    if (dim == 64) return launch_pairs<T, 128, 64>(A, n_pairs, s);
  }
  return GA_EUNSUPPORTED;
}

}  // namespace
}  // namespace ga

extern "C" int ga_pair_attention(const int32_t *type_pointer, int64_t n_types,
                                 const int64_t *by_type, const int64_t *dst_by_type,
                                 const int32_t *pair_pointer, const int32_t *nbr, const void *q,
                                 const void *k, const void *v, const void *att, const void *msg,
                                 void *m, float *lse, int64_t n_pairs, int64_t max_slots,
                                 int64_t heads, int64_t dim, int dtype, ga_stream_t stream) {
  if (n_types <= 0 || n_pairs < 0 || heads <= 0 || dim <= 0 || max_slots < 0) return GA_EINVAL;
  if (n_types > 0x7fffffff || n_pairs > 0x7fffffff || heads * dim > 0x7fffffff) return GA_EINVAL;
  if (dtype != GA_F32 && dtype != GA_BF16) return GA_EINVAL;
  if (n_pairs == 0) return GA_OK;
  if (!type_pointer || !by_type || !dst_by_type || !pair_pointer || !nbr || !q || !k || !v ||
      !att || !msg || !m || !lse)
    return GA_EINVAL;
  if (!ga::aligned(lse, 4)) return GA_EALIGN;
  // a lane group walks its rows alone (ga_pair_attention_preferred): 256 slots are 64
  // dependent batches, some 50 us
  if (max_slots > 256) return GA_EUNSUPPORTED;
  if (!ga::aligned(q, 16) || !ga::aligned(k, 16) || !ga::aligned(v, 16) || !ga::aligned(m, 16))
    return GA_EUNSUPPORTED;
  ga::PairArgs A{type_pointer, by_type, dst_by_type, pair_pointer, nbr, q, k, v, att, msg, m, lse,
                 (int)n_types};
  if (dtype == GA_F32)
    return ga::launch_pairs_dim<float>(A, n_pairs, heads * dim, dim, (hipStream_t)stream);
  return ga::launch_pairs_dim<ga::bf16_t>(A, n_pairs, heads * dim, dim, (hipStream_t)stream);
}

// Where the pass beats the three launches, from what the host knows.  A lane group walks
// rpg rows of a tile, four slots per dependent batch, and nobody helps it: the pass takes
// the longer of its share of the traffic and that chain, and large pairs come on top --
// taken as one and a half rows of the largest size on one group, between a lone large pair
// and many side by side.  The three launches pay for the pairs' rows in memory and for
// their own starts, but spread the slots evenly.  The figures (us; 0.72 per batch, 30 and
// 33 per 100 k pairs and 1 M edges of 256-byte rows) are fitted to 500 to 1.95 M pairs of 1
// to 256 slots; pair form against three launches, 1 x 64 fp32:
//   500 pairs of 16 / 32 / 256      29 : 34,  40 : 34,  199 : 40 us    (7 tiles for 256 CUs)
//   2,500 pairs of 16 / 32 / 100    30 : 36,  42 : 38,   91 : 48
//   10,000 pairs of 32 / 64         41 : 48,  65 : 59
//   40,000 pairs of 64 / 256       111 : 138, 359 : 378
//   100,000 pairs of 3 on average, 0.3 % of 64 / 128 / 256   84 : 99, 115 : 99, 177 : 100
//   1 M pairs of 3, 0.3 % of 128 / 256                      523 : 669, 656 : 696
extern "C" int ga_pair_attention_preferred(int64_t n_pairs, int64_t n_edges, int64_t max_slots,
                                           int64_t heads, int64_t dim, int dtype) {
  if (n_pairs <= 0 || n_edges < n_pairs || heads <= 0 || dim <= 0 || max_slots > 256) return 0;
  if (dtype != GA_F32 && dtype != GA_BF16) return 0;
  if ((heads * dim != 64 && heads * dim != 128) || (dim != 8 && dim != 16 && dim != 32 && dim != 64))
    return 0;
  const double rpg = (double)(heads * dim * (dtype == GA_F32 ? 4 : 2)) / 64;    // rows per lane group
  const double mean = (double)((n_edges / n_pairs + ga::kPairBatch - 1) / ga::kPairBatch);
  const double most = (double)((max_slots + ga::kPairBatch - 1) / ga::kPairBatch);
  const double p = 1e-3 * (double)n_pairs, e = 1e-3 * (double)n_edges, row = rpg / 4;
  const double share = (0.30 * p + 0.033 * e) * row, chain = 0.72 * rpg * mean;
  const double extra = most > mean ? 1.5 * 0.72 * (most - mean) : 0.0;
  const double pass = 20.0 + (share > chain ? share : chain) + extra;
  const double three = 36.0 + (0.43 * p + 0.033 * e) * row;
  return pass < three;
}
