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
// at two or three.
//
// Bound, 2 M edges in 269,078 pairs, 8 x 16 bf16: vector instructions, 4,240 per wavefront, 116
// of 131 us of issue; with the scores as v_dot2 of the rows as they come, one 32-bit offset for
// a key and a value row and hardware rounding 111 us (0.64 GB pass the L2s, 5.8 TB/s).  4.76 M
// edges in 1.95 M pairs, 1 x 64 fp32: products, walk and gathers each 200 to 280 us of 680 and
// only partly under one another; split products, eight features per lane, one load to find the
// tile and one a row, messages in the order they are made: 560 us.  Two to five wavefronts per
// SIMD, two or four slots in flight, the next batch's rows asked for before this one's work:
// within 3 % of one another.  The whole operator (matrices, this pass, the sum of the pairs), us:
//   4.76 M edges, 1.95 M pairs: 1 x 64 fp32 810 -> 674
//   2 M edges, 269 k pairs: 8 x 16 bf16 162 -> 137
//   1.2 M edges, 0.62 M pairs: 1 x 64 fp32 241 -> 193, 4 x 16 190 -> 177, bf16 144 -> 114 and
//     126 -> 108, 8 x 16 bf16 214 -> 187, fp32 373 -> 367, 16 x 8 fp32 383 -> 391
#pragma once

#include <type_traits>

#include "common.h"
#include "typed_chunks.h"

namespace ga {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef short shortx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr int kPairRows = 64;       // pairs per tile
constexpr int kPairBatch = 4;       // slots whose rows are in flight per lane group: a
                                    // pair has two to eight edges where pairs are used
constexpr int kWaveCount = kBlock / kWave;

struct PairArgs {
  const int4 *rows;                 // row r: first slot, end slot, destination, 0 ...
  const int4 *tiles;                // ... and tile t: type, first row, end row, 0; or these:
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

// the value of three pieces
__device__ __forceinline__ float joined(bf16_t p0, bf16_t p1, bf16_t p2) {
  return fmaf(fmaf(bf16_lo(p2), kPieceScale, bf16_lo(p1)), kPieceScale, bf16_lo(p0));
}

// Heads of 32 and 64 of rows of 64 fp32 features: the product on the bf16 instruction, at 16
// times the fp32 one's rate.  Operands are split into three bf16 pieces; six piece products
// are added in fp32, those of one weight (1, 2^-8, 2^-16) in an accumulator of their own.  The
// three left out are together below 2^-24 of |x||w|.  The tile's rows are kept split, three
// planes of 64 values side by side: split when an operand is read, every value would be split
// by every wavefront.  The matrices come split and in the order the lanes read them
// (pair_weights_kernel).  Messages of 1.2 M edges in 0.53 M pairs against float64, 2-norm /
// largest, on the fp32 instruction and here: heads of 64 1.63e-7 / 3.8e-7 and 0.71e-7 / 1.5e-7,
// of 32 1.20e-7 / 3.1e-7 and 0.61e-7 / 1.2e-7, heads of 64 of values in [0, 1) 1.19e-7 / 4.9e-7
// and 0.57e-7 / 2.1e-7.  (Pieces cut off at eight bits and added in one accumulator: 1.30e-7 /
// 4.7e-7, and up to 7.8 x 2^-24 of |x||w| left out; 636 us instead of 640 for the operator on
// 1.95 M pairs, 1 x 64.)
template <int D>
struct SplitBlock {
  static constexpr int KB = D / 32;
  uint4 w[KB][3];
  static __device__ __forceinline__ uint32_t unit(int col_block, int b, int piece, int lane) {
    return ((col_block * KB + b) * 3 + piece) * kWave + lane;
  }
  __device__ __forceinline__ void load(const uint4 *W, int col_block, int lane) {
#pragma unroll
    for (int b = 0; b < KB; ++b)
#pragma unroll
      for (int q = 0; q < 3; ++q) w[b][q] = W[unit(col_block, b, q, lane)];
  }
  // row: planes of 64 values
  __device__ __forceinline__ floatx4 mma(const bf16_t *row, int k0, int lk) const {
    floatx4 acc[3] = {};
#pragma unroll
    for (int b = 0; b < KB; ++b) {
      uint4 x[3];
#pragma unroll
      for (int q = 0; q < 3; ++q)
        x[q] = *reinterpret_cast<const uint4 *>(row + 64 * q + k0 + 32 * b + 8 * lk);
#pragma unroll
      for (int px = 0; px < 3; ++px)
#pragma unroll
        for (int pw = 0; pw < 3 - px; ++pw)
          acc[px + pw] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8, x[px]), __builtin_bit_cast(bf16x8, w[b][pw]), acc[px + pw],
              0, 0, 0);
    }
    floatx4 sum;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      sum[i] = fmaf(fmaf(acc[2][i], kPieceScale, acc[1][i]), kPieceScale, acc[0][i]);
    return sum;
  }
  // the same product on the fp32 instruction, for operands that are not finite: their pieces
  // give NaN where fp32 products may give inf
  static __device__ floatx4 mma_f32(const bf16_t *row, const uint4 *W, int col_block, int k0, int lr,
                                    int lk) {
    floatx4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int k = 0; k < D; k += 4) {
      const int kk = k + lk;             // of the head; the matrix's lane (kk % 32 / 8, column)
      const bf16_t *x = row + k0 + kk;
      const bf16_t *w = (const bf16_t *)(W + unit(col_block, kk / 32, 0, kk % 32 / 8 * 16 + lr)) + kk % 8;
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(joined(x[0], x[64], x[128]),
                                                 joined(w[0], w[8 * kWave], w[16 * kWave]), acc, 0, 0, 0);
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

// Rows of F floats, a lane's features in two 16-byte pieces half a row apart.
template <int F>
struct HalfRows {
  struct raw_t { float4 lo, hi; };
  static __device__ __forceinline__ raw_t load(const float *p) {
    return {*reinterpret_cast<const float4 *>(p), *reinterpret_cast<const float4 *>(p + F / 2)};
  }
  static __device__ __forceinline__ void widen(const raw_t &r, float (&f)[8]) {
    f[0] = r.lo.x; f[1] = r.lo.y; f[2] = r.lo.z; f[3] = r.lo.w;
    f[4] = r.hi.x; f[5] = r.hi.y; f[6] = r.hi.z; f[7] = r.hi.w;
  }
  static __device__ __forceinline__ void store(float *p, const float (&f)[8]) {
    *reinterpret_cast<float4 *>(p) = make_float4(f[0], f[1], f[2], f[3]);
    *reinterpret_cast<float4 *>(p + F / 2) = make_float4(f[4], f[5], f[6], f[7]);
  }
};

// The shapes whose products are split: heads of 32 features fill the k of an instruction.  Rows
// of 128 stay on the fp32 instruction, not measured otherwise: three planes of pieces would
// make a tile of 49 KB, three workgroups to a CU where the pass now has four.
template <typename T, int F, int D>
constexpr bool kSplitShape = sizeof(T) == 4 && F == 64 && D >= 32;

// TILES: the tiles and rows of PairArgs (else the five columns below them); matrices of split
// shapes are then split; messages and log-sum-exps leave in row order, and key and value rows
// lie inside 4 GB, so that a slot's address is one 32-bit offset for both.
template <typename T, int F, int D, bool TILES>
__global__ __launch_bounds__(kBlock, F == 128 && sizeof(T) == 4 ? 4 : (F == 64 && sizeof(T) == 4 && D == 64 && TILES ? 4 : 5))
void pair_attn_kernel(PairArgs A) {
  constexpr bool kSplit = TILES && kSplitShape<T, F, D>;
  // Features per lane.  One head of 64 fp32 features: eight, two 16-byte pieces half a row
  // apart -- addresses, masks, exponentials and lane sums of a slot cost the same for four
  // features as for eight (with neighbouring pieces every load touches both lines of a row).
  constexpr bool kHalves = kSplit && D == F;
  constexpr int VEC = kHalves ? 8 : 16 / (int)sizeof(T);
  constexpr int LPR = F / VEC;                    // lanes per row
  constexpr int G = kBlock / LPR;                 // lane groups
  constexpr int RPG = kPairRows / G;              // rows a group walks
  constexpr int CB = F / 16 / kWaveCount;         // column blocks per wavefront
  constexpr int H = F / D;
  constexpr int HL = D / VEC < 1 ? 1 : D / VEC;   // lanes per head
  // row stride of the tile: 16 bytes past the row, or past its three planes of pieces
  constexpr int LD = (kSplit ? F * 3 / 2 : F) + 16 / (int)sizeof(T);
  static_assert(F % 64 == 0 && HL <= 16 && RPG >= 1, "layout");
  typedef std::conditional_t<kHalves, HalfRows<F>, Frag<T, kHalves ? 16 / (int)sizeof(T) : VEC>> IO;
  typedef typename IO::raw_t raw_t;
  __shared__ __attribute__((aligned(16))) T tile[kPairRows * LD];
  // first slot, end slot, pair (TILES: row): a lane group's rows are its own
  __shared__ int slot0[kPairRows], slot1[kPairRows], pair_of[kPairRows];
  const T *const q = (const T *)A.q, *const k = (const T *)A.k, *const v = (const T *)A.v;

  int type, row0, row1;
  if constexpr (TILES) {
    const int4 t = A.tiles[blockIdx.x];
    type = t.x;
    row0 = t.y;
    row1 = t.z;
    if (type < 0) return;
  } else if (!locate_chunk(A.type_pointer, A.n_types, kPairRows, blockIdx.x, type, row0, row1)) {
    return;
  }
  type = __builtin_amdgcn_readfirstlane(type);
  row0 = __builtin_amdgcn_readfirstlane(row0);
  row1 = __builtin_amdgcn_readfirstlane(row1);

  const int tid = threadIdx.x;
  const int lane64 = tid & (kWave - 1), wave = tid / kWave;
  const int lr = lane64 & 15, lk = lane64 >> 4;
  const int grp = tid / LPR, lane = tid % LPR, f0 = lane * (kHalves ? VEC / 2 : VEC);

  // a row of the tile as the operand of a product: a row or, split, its pieces in its place
  typedef std::conditional_t<kSplit, SplitBlock<D>, Block<T, D>> Weights;
  typedef std::conditional_t<kSplit, bf16_t, T> operand_t;
  auto put_operand = [&](int r, const float (&x)[VEC]) {
    if constexpr (kSplit) {
      uint32_t p[3][VEC / 2];
      split(x, p);
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int h = 0; h < VEC / 4; ++h)
          *reinterpret_cast<uint2 *>((operand_t *)(tile + r * LD) + F * i + h * (F / 2) + f0) =
              make_uint2(p[i][2 * h], p[i][2 * h + 1]);
    } else {
      IO::store(tile + r * LD + f0, x);
    }
  };
  // the type's matrix, and the wavefront's columns of it
  auto matrix = [&](const void *W) {
    if constexpr (kSplit) return (const uint4 *)W + (int64_t)type * (F * D * 3 / 8);
    else return (const T *)W + (int64_t)type * F * D;
  };
  auto columns = [&](const void *W, Weights (&w)[CB]) {
#pragma unroll
    for (int c = 0; c < CB; ++c) {
      if constexpr (kSplit) w[c].load(matrix(W), wave * CB + c, lane64);
      else w[c].load(matrix(W), (wave * CB + c) * 16 + lr, lk);
    }
  };
  // the tile's rows times the wavefront's columns, in place
  auto product = [&](const void *W, const Weights (&w)[CB]) {
    floatx4 acc[CB][kPairRows / 16];
#pragma unroll
    for (int c = 0; c < CB; ++c) {
      const int col0 = (wave * CB + c) * 16;
      const int k0 = D < 16 ? col0 : col0 / D * D;
#pragma unroll
      for (int b = 0; b < kPairRows / 16; ++b) {
        acc[c][b] = w[c].mma((const operand_t *)(tile + (16 * b + lr) * LD), k0, lk);
        // heads of 64: the rows of all blocks at once would take 64 registers more
        if constexpr (D == 64) __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (kSplit) {
        float finite = 0.0f;
#pragma unroll
        for (int b = 0; b < kPairRows / 16; ++b)
#pragma unroll
          for (int i = 0; i < 4; ++i) finite = fmaf(acc[c][b][i], 0.0f, finite);
        if (__ballot(finite != 0.0f)) {
#pragma unroll
          for (int b = 0; b < kPairRows / 16; ++b)
            acc[c][b] = Weights::mma_f32((const operand_t *)(tile + (16 * b + lr) * LD), matrix(W),
                                         wave * CB + c, k0, lr, lk);
        }
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
  int ids = 0;                           // sources of a batch of slots: one a lane of four
  int64_t dst[RPG];
  if constexpr (TILES) {
#pragma unroll
    for (int i = 0; i < RPG; ++i) {      // rows past the last one repeat it
      const int r = grp + i * G, at = row0 + min(r, n - 1);
      const int4 x = A.rows[at];
      if (lane == 0) {
        pair_of[r] = at;
        slot0[r] = x.x;
        slot1[r] = x.y;
      }
      dst[i] = x.z;
      if (i == 0) ids = A.nbr[x.x + min(lane & 3, x.y - 1 - x.x)];
    }
  } else {
    if (tid < kPairRows) {
      const int p = (int)A.by_type[row0 + min(tid, n - 1)];
      pair_of[tid] = p;
      slot0[tid] = A.pair_pointer[p];
      slot1[tid] = A.pair_pointer[p + 1];
    }
#pragma unroll
    for (int i = 0; i < RPG; ++i) dst[i] = A.dst_by_type[row0 + min(grp + i * G, n - 1)];
  }
#pragma unroll
  for (int i = 0; i < RPG; ++i) {
    const raw_t x = IO::load(q + dst[i] * F + f0);
    if constexpr (kSplit) {
      float xf[VEC];
      IO::widen(x, xf);
      put_operand(grp + i * G, xf);
    } else {
      *reinterpret_cast<raw_t *>(tile + (grp + i * G) * LD + f0) = x;
    }
  }
  {
    Weights w[CB];
    columns(A.att, w);
    __syncthreads();
    product(A.att, w);
  }

  // ---- attention inside the pairs: every G-th row of the tile, one after another (large
  // pairs lie side by side where the relation's popular destinations do) ----
  int r = grp;
  if (r < n) {
    // bf16 scores: two products an instruction, the keys as they come
    constexpr bool kDot2 = sizeof(T) == 2;
    float qf[VEC], acc[VEC], m = -INFINITY, l = 0.0f;
    raw_t qr;
    auto open_row = [&]() {
      qr = IO::load(tile + r * LD + f0);
      if constexpr (!kDot2) IO::widen(qr, qf);
#pragma unroll
      for (int e = 0; e < VEC; ++e) acc[e] = 0.0f;
      m = -INFINITY;
      l = 0.0f;
    };
    int pos = slot0[r], end = slot1[r];
    if constexpr (!TILES) ids = A.nbr[pos + min(lane & 3, end - 1 - pos)];
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
        kx[t] = raw_t{};                   // scores past the pair's end are formed, not used
        if (t < cnt) {
          if constexpr (TILES) {
            const uint32_t at = ((uint32_t)g[t] * F + f0) * (uint32_t)sizeof(T);
            kx[t] = IO::load((const T *)((const char *)k + at));
            vx[t] = IO::load((const T *)((const char *)v + at));
          } else {
            kx[t] = IO::load(k + (int64_t)g[t] * F + f0);
            vx[t] = IO::load(v + (int64_t)g[t] * F + f0);
          }
        }
      }
      float s[kPairBatch], bm = -INFINITY;
#pragma unroll
      for (int t = 0; t < kPairBatch; ++t) {
        float d = 0.0f;
        if constexpr (kDot2) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            d = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, (&kx[t].x)[e]),
                                                __builtin_bit_cast(bf16x2, (&qr.x)[e]), d, false);
        } else {
          float kf[VEC];
          IO::widen(kx[t], kf);
#pragma unroll
          for (int e = 0; e < VEC; ++e) d = fmaf(kf[e], qf[e], d);
        }
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
        put_operand(r, o);
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
  if constexpr (kSplit) {
    // rows no pair owns hold the first product: as pieces, some of its halves are not finite,
    // and the wavefront would repeat the second on the fp32 instruction (a tile in five)
    const float zero[VEC] = {};
#pragma unroll
    for (int i = 0; i < RPG; ++i)
      if (grp + i * G >= n) put_operand(grp + i * G, zero);
  }
  {
    Weights w[CB];
    columns(A.msg, w);
    __syncthreads();
    product(A.msg, w);
  }
#pragma unroll
  for (int i = 0; i < RPG; ++i) {
    const int row = grp + i * G;
    if (row < n) {
      T *const to = (T *)A.m + (int64_t)pair_of[row] * F + f0;
      const raw_t x = IO::load(tile + row * LD + f0);
      if constexpr (kHalves) {
        float xf[VEC];
        IO::widen(x, xf);
        IO::store(to, xf);
      } else {
        *reinterpret_cast<raw_t *>(to) = x;
      }
    }
  }
}

template <typename T, int F, int D, bool TILES>
int launch_pairs(PairArgs &A, int64_t n_pairs, hipStream_t s) {
  const int64_t grid = (n_pairs + kPairRows - 1) / kPairRows + A.n_types;
  if (grid > 0x7fffffff) return GA_EUNSUPPORTED;
  hipLaunchKernelGGL((pair_attn_kernel<T, F, D, TILES>), dim3((unsigned)grid), dim3(kBlock), 0, s, A);
  return launch_status();
}

template <typename T, bool TILES>
int launch_pairs_dim(PairArgs &A, int64_t n_pairs, int64_t feat, int64_t dim, hipStream_t s) {
  if (feat == 64) {
    if (dim == 8) return launch_pairs<T, 64, 8, TILES>(A, n_pairs, s);
    if (dim == 16) return launch_pairs<T, 64, 16, TILES>(A, n_pairs, s);
    if (dim == 32) return launch_pairs<T, 64, 32, TILES>(A, n_pairs, s);
    if (dim == 64) return launch_pairs<T, 64, 64, TILES>(A, n_pairs, s);
  } else if (feat == 128) {
    if (dim == 8) return launch_pairs<T, 128, 8, TILES>(A, n_pairs, s);
    if (dim == 16) return launch_pairs<T, 128, 16, TILES>(A, n_pairs, s);
    if (dim == 32) return launch_pairs<T, 128, 32, TILES>(A, n_pairs, s);
    if (dim == 64) return launch_pairs<T, 128, 64, TILES>(A, n_pairs, s);
  }
  return GA_EUNSUPPORTED;
}

inline int check_pairs(const PairArgs &A, int64_t max_slots) {
  if (!A.nbr || !A.q || !A.k || !A.v || !A.att || !A.msg || !A.m || !A.lse) return GA_EINVAL;
  if (!aligned(A.lse, 4)) return GA_EALIGN;
  // a lane group walks its rows alone (ga_pair_attention_preferred): 256 slots are 64
  // dependent batches, some 50 us
  if (max_slots > 256) return GA_EUNSUPPORTED;
  if (!aligned(A.q, 16) || !aligned(A.k, 16) || !aligned(A.v, 16) || !aligned(A.m, 16))
    return GA_EUNSUPPORTED;
  return GA_OK;
}
inline bool pair_counts_ok(int64_t n_types, int64_t n_pairs, int64_t max_slots, int64_t heads, int64_t dim,
                    int dtype) {
  return n_types > 0 && n_pairs >= 0 && heads > 0 && dim > 0 && max_slots >= 0 &&
         n_types <= 0x7fffffff && n_pairs <= 0x7fffffff && heads * dim <= 0x7fffffff &&
         (dtype == GA_F32 || dtype == GA_BF16);
}

}  // namespace
}  // namespace ga
