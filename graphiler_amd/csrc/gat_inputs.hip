// GAT layer that aggregates its inputs instead of its projected rows (bf16):
//   out[v, h, :] = (sum over the in-edges e of v of alpha[e, h] x[src(e), :]) @ W_h,
// the same layer as projecting first (examples/GAT/GAT.py:25-36), whose sum over edges and
// whose product are both linear.  An edge then moves a row of the layer's input, K values,
// instead of a row of heads x D: with 100 inputs and four heads of 64 that is 256 bytes
// instead of 512, and the pass over the edges is bound by the bytes that it gathers.
//
// Rows are copied once into a table whose rows are whole 128-byte lines and carry the node's
// source terms <x, W_h a_l[h]> at their end, so an edge touches no second table.  Destinations
// are walked in order of their length, four to a wavefront (no lane waits for a longer
// neighbour, no state crosses lanes), longer ones in pieces; 16 destinations' sums meet in LDS
// and leave through W on the matrix cores.  Nothing between x, W and the result is rounded
// below fp32 (projecting first rounds z to bf16: error against float64 2.0e-3 -> 1.66e-3 of
// the layer's norm, the rounding of the result).
//
// Layer, projecting first -> here, us (four heads of 64 unless said): 64.3 M R-MAT edges, 100
// inputs 4800 -> 3180 (table 255, pass 2870 = 5.7 TB/s of random rows of 256 bytes, which is
// what bounds it; long rows 58); 11.8 M edges, 100 inputs 894 -> 405; 10.5 M edges, 50 inputs,
// eight heads 2570 -> 870; 10 M uniform edges, 100 inputs 1120 -> 520.
#include "common.h"

#include <type_traits>

namespace ga {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kTileRows = 16;          // destinations of a workgroup
constexpr int kLanes = 16;             // lanes that walk a destination: 8 inputs each
constexpr int kMaxK = 8 * kLanes;
constexpr int kUnroll = 8;

template <int L>
__device__ __forceinline__ uint32_t row_bcast(uint32_t v) {
  return __builtin_amdgcn_update_dpp(0, v, 0x150 + L, 0xF, 0xF, true);
}
template <int L>
__device__ __forceinline__ float row_bcast(float v) {
  return __uint_as_float(row_bcast<L>(__float_as_uint(v)));
}
template <int I, int N, typename F>
__device__ __forceinline__ void unrolled(F &&f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>());
    unrolled<I + 1, N>(f);
  }
}
__device__ __forceinline__ float finite_or_zero(float v) { return v == -INFINITY ? 0.0f : v; }
__device__ __forceinline__ float leaky(float s, float slope) { return s > 0.0f ? s : s * slope; }

// ------------------------------------------------------------------ small operands ----
// Columns of a chunk (one head's, 64 at most): block c of chunk ch holds the columns
// ch * 16 C + n C + c, so that lane n of the product has C neighbouring ones.
__host__ __device__ inline int chunk_blocks(int dim) { return dim >= 64 ? 4 : dim / 16; }

__global__ __launch_bounds__(kBlock) void gat_inputs_weights_kernel(
    const bf16_t *__restrict__ W, const float *__restrict__ a_l, const float *__restrict__ a_r, int K,
    int ksteps, int heads, int dim, uint4 *__restrict__ packed, float *__restrict__ wa,
    int32_t *__restrict__ not_finite) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *not_finite = 0;
  const int M = heads * dim, C = chunk_blocks(dim);
  const int n_packed = M / 16 * ksteps * kWave;
  int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n_packed) {                       // (block, k step, lane): k = 32 ks + 8 q .. + 7 of its column
    const int lane = i & (kWave - 1), ks = i / kWave % ksteps, b = i / kWave / ksteps;
    const int col = b / C * 16 * C + (lane & 15) * C + b % C, k0 = ks * 32 + (lane >> 4) * 8;
    uint32_t h[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) h[j] = k0 + j < K ? W[(int64_t)(k0 + j) * M + col] : 0;
    packed[i] = make_uint4(h[0] | h[1] << 16, h[2] | h[3] << 16, h[4] | h[5] << 16, h[6] | h[7] << 16);
    return;
  }
  i -= n_packed;
  if (i < 2 * heads * kMaxK) {              // wa[side][h][k] = <W[k, h, :], a[h, :]>
    const int k = i % kMaxK, h = i / kMaxK % heads;
    const float *a = (i / kMaxK / heads ? a_r : a_l) + h * dim;
    float s = 0.0f;
    if (k < K)
      for (int d = 0; d < dim; ++d) s = fmaf(bf16_lo(W[(int64_t)k * M + h * dim + d]), a[d], s);
    wa[i] = s;
  }
}

// Row v of the gathered table: the K inputs, zeros, and in its last 4 H bytes the source terms
// <x, wa[0][h]> as fp32; er[v, h] = <x, wa[1][h]>.
template <int H, int PIECE>
__global__ __launch_bounds__(kBlock) void gat_inputs_rows_kernel(
    const bf16_t *__restrict__ X, const float *__restrict__ wa, int64_t rows, int K, int row_bytes,
    int stride, char *__restrict__ table, float *__restrict__ er, int32_t *__restrict__ not_finite) {
  const int j = threadIdx.x & (kLanes - 1);
  float al[H][8], ar[H][8];
#pragma unroll
  for (int h = 0; h < H; ++h)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      al[h][e] = wa[h * kMaxK + 8 * j + e];
      ar[h][e] = wa[(H + h) * kMaxK + 8 * j + e];
    }
  for (int64_t v = (int64_t)blockIdx.x * (kBlock / kLanes) + threadIdx.x / kLanes; v < rows;
       v += (int64_t)gridDim.x * (kBlock / kLanes)) {
    uint32_t w[4] = {0, 0, 0, 0};
    const bf16_t *src = X + v * K + 8 * j;
#pragma unroll
    for (int e = 0; e < 8; e += PIECE)
      if (8 * j + e < K) {
        if constexpr (PIECE == 8) {
          const uint4 t = *reinterpret_cast<const uint4 *>(src);
          w[0] = t.x; w[1] = t.y; w[2] = t.z; w[3] = t.w;
        } else if constexpr (PIECE == 4) {
          const uint2 t = *reinterpret_cast<const uint2 *>(src + e);
          w[e / 2] = t.x; w[e / 2 + 1] = t.y;
        } else if constexpr (PIECE == 2) {
          w[e / 2] = *reinterpret_cast<const uint32_t *>(src + e);
        } else {
          w[e / 2] |= (uint32_t)src[e] << (16 * (e & 1));
        }
      }
    bool odd = false;                     // an exponent of ones
#pragma unroll
    for (int e = 0; e < 4; ++e)
      odd = odd || (w[e] & 0x7f80u) == 0x7f80u || (w[e] & 0x7f800000u) == 0x7f800000u;
    if (odd) *not_finite = 1;             // every writer stores the same value
    float l[H], r[H];
#pragma unroll
    for (int h = 0; h < H; ++h) {
      l[h] = r[h] = 0.0f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x = e & 1 ? bf16_hi(w[e / 2]) : bf16_lo(w[e / 2]);
        l[h] = fmaf(x, al[h][e], l[h]);
        r[h] = fmaf(x, ar[h][e], r[h]);
      }
      l[h] = row16_sum(l[h]);
      r[h] = row16_sum(r[h]);
    }
    // the source terms replace the words of the row's end
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const int at = row_bytes - 4 * (H - h) - 16 * j;        // my word they fall on
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = at == 4 * e ? __float_as_uint(l[h]) : w[e];
    }
    if (16 * j < row_bytes)
      *reinterpret_cast<uint4 *>(table + v * stride + 16 * j) = make_uint4(w[0], w[1], w[2], w[3]);
#pragma unroll
    for (int h = 0; h < H; ++h)
      if (j == h) er[v * H + h] = r[h];
  }
}

// -------------------------------------------------------------------------- the pass ----
struct GatInputs {
  const int4 *rows;             // (n_rows): node, first and end slot; n_light short rows by falling length, then the long ones
  const int2 *pieces;           // (n_pieces): first and end slot of a piece of a long row
  const int32_t *piece_first;   // (n_long + 1): first piece of a long row
  const int32_t *nbr;
  const char *table;
  const float *er;
  const int32_t *not_finite;    // set: X has values that are not finite
  const uint4 *packed;
  float *partial;               // (n_pieces) states
  bf16_t *out;
  uint64_t table_bytes;
  int n_light, n_long, n_pieces, piece_blocks;
  int K, ksteps, dim, row_bytes, stride, act;
  float slope;
};

template <int H>
struct State {
  static constexpr int HH = H > 1 ? H / 2 : 1;      // heads whose softmax a lane keeps
  static constexpr int kSets = (H + 3) / 4;
  static constexpr int kFloats = H * kMaxK + 2 * H; // of a stored state
  floatx4 sum[kSets][8];        // [h / 4][e][h % 4]: input 8 j + e of lane j, head h
  float m[HH], l[HH];           // of heads hp * HH + i, hp = lane / 8
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int k = 0; k < kSets; ++k)
#pragma unroll
      for (int e = 0; e < 8; ++e) sum[k][e] = floatx4{0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < HH; ++i) { m[i] = -INFINITY; l[i] = 0.0f; }
  }
};

// The weights of a batch on their way between lanes, and zeros for lanes of other rows.
template <int H>
struct WeightSlots {
  float p[kBlock / kWave][4][H][8];
  float zero[8];
};

// Slots [a, b) of one destination by my 16 lanes, four destinations a wavefront: online softmax
// per head, a rescale per batch of eight slots where a maximum has moved.  Lane j forms the
// logits of slot j % 8 for its half of the heads, from the terms at the end of that slot's row.
//
// The weighted sum is a matrix product: rows (destination, head), k (destination, slot), columns
// inputs, with zeros in the weights where the destinations differ.  Lane j holds the inputs
// 8 j .. 8 j + 7 of eight slots, so column block e takes input 8 j + e from lane j: the operand
// is a transposition inside the lane, and a destination's sums come out in its own 16 lanes.
// The weights stay fp32 (three bf16 pieces, x is bf16 as it is).  32 byte permutations and 24
// matrix instructions a batch instead of 320 vector instructions: with those the pass was
// bound by vector issue (64.3 M edges, 100 inputs, four heads 3.27 ms).
// A zero weight does not silence an input that is not finite, so with such inputs (FINITE false)
// the same sum is taken with multiply-adds, which keep a destination to its own lanes.
//
// The loop is uniform: a matrix instruction takes all lanes, and a destination whose slots are
// used up adds zeros.
template <int H, bool FINITE>
__device__ __forceinline__ void walk(const GatInputs &A, rsrc_t table, int a, int b, const float *er,
                                     WeightSlots<H> &slots, State<H> &st) {
  constexpr int HH = State<H>::HH;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int j = lane & (kLanes - 1), q = lane / kLanes, t8 = j & 7;
  const int hp = H > 1 ? j >> 3 : 0;
  const uint32_t x_lane = 16 * j < A.row_bytes ? 16u * j : 0u;
  const uint32_t el_lane = (uint32_t)(A.row_bytes - 4 * H + 4 * HH * hp);
  float er_mine[HH];
#pragma unroll
  for (int i = 0; i < HH; ++i) er_mine[i] = er[hp * HH + i];
  st.clear();
  // the longest of the wavefront's four
  int steps = (b - a + kUnroll - 1) / kUnroll;
  steps = max(max(__builtin_amdgcn_readlane(steps, 0), __builtin_amdgcn_readlane(steps, 16)),
              max(__builtin_amdgcn_readlane(steps, 32), __builtin_amdgcn_readlane(steps, 48)));
  auto index = [&](int s) { return s + t8 < b ? (uint32_t)A.nbr[s + t8] * (uint32_t)A.stride : 0u; };
  float *p_mine = &slots.p[wave][q][hp * HH][t8];
  const float *p_row[State<H>::kSets];      // the weights of row j of the product
#pragma unroll
  for (int k = 0; k < State<H>::kSets; ++k)
    p_row[k] = (j >> 2) == q && 4 * k + (j & 3) < H ? &slots.p[wave][q][(4 * k + (j & 3)) % H][0] : slots.zero;
  uint32_t off = index(a);
  for (int step = 0, s = a; step < steps; ++step, s += kUnroll) {
    uint4 x[kUnroll];
    unrolled<0, kUnroll>([&](auto t) __attribute__((always_inline)) {
      x[t] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(table, x_lane + row_bcast<t>(off), 0, 0));
    });
    float s_[HH];
    if constexpr (HH == 4) {
      const float4 e = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(table, off + el_lane, 0, 0));
      s_[0] = e.x; s_[1] = e.y; s_[2] = e.z; s_[3] = e.w;
    } else if constexpr (HH == 2) {
      const float2 e = __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(table, off + el_lane, 0, 0));
      s_[0] = e.x; s_[1] = e.y;
    } else {
      s_[0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(table, off + el_lane, 0, 0));
    }
    off = index(s + kUnroll);         // of the next batch, behind this one's rows
    const bool live = s + t8 < b;
    float p[HH], corr[HH];
    bool moved = false;
#pragma unroll
    for (int i = 0; i < HH; ++i) {
      s_[i] = live ? leaky(s_[i] + er_mine[i], A.slope) : -INFINITY;
      float m = s_[i];                // over the eight lanes of my half
      m = fmaxf(m, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(m), 0xB1, 0xF, 0xF, true)));
      m = fmaxf(m, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(m), 0x4E, 0xF, 0xF, true)));
      m = fmaxf(m, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(m), 0x141, 0xF, 0xF, true)));
      const float top = fmaxf(st.m[i], m), ref = finite_or_zero(top);
      moved = moved || top > st.m[i];
      corr[i] = __expf(st.m[i] - ref);
      p[i] = __expf(s_[i] - ref);
      st.l[i] = st.l[i] * corr[i] + row8_sum(p[i]);
      st.m[i] = top;
    }
    if constexpr (FINITE) {
#pragma unroll
      for (int i = 0; i < HH; ++i) p_mine[8 * i] = p[i];
    }
    if (__builtin_amdgcn_ballot_w64(moved) != 0) {
      unrolled<0, H>([&](auto h) __attribute__((always_inline)) {
        const float c = row_bcast<(H > 1 ? 8 * (h / HH) : 0)>(corr[h % HH]);
#pragma unroll
        for (int e = 0; e < 8; ++e) st.sum[h / 4][e][h % 4] *= c;
      });
    }
    if constexpr (FINITE) {
      __builtin_amdgcn_wave_barrier();
      uint4 w[State<H>::kSets][3];
#pragma unroll
      for (int k = 0; k < State<H>::kSets; ++k) {
        const float4 lo = *reinterpret_cast<const float4 *>(p_row[k]);
        const float4 up = *reinterpret_cast<const float4 *>(p_row[k] + 4);
        const float v[8] = {lo.x, lo.y, lo.z, lo.w, up.x, up.y, up.z, up.w};
        split8(v, w[k][0], w[k][1], w[k][2]);
      }
      __builtin_amdgcn_wave_barrier();
      unrolled<0, 4>([&](auto d) __attribute__((always_inline)) {      // inputs 2 d and 2 d + 1
        auto word = [&](int t) { return d == 0 ? x[t].x : d == 1 ? x[t].y : d == 2 ? x[t].z : x[t].w; };
        constexpr uint32_t lo = 0x05040100u, hi = 0x07060302u;
        uint4 f[2];
        f[0] = uint4{__builtin_amdgcn_perm(word(1), word(0), lo), __builtin_amdgcn_perm(word(3), word(2), lo),
                     __builtin_amdgcn_perm(word(5), word(4), lo), __builtin_amdgcn_perm(word(7), word(6), lo)};
        f[1] = uint4{__builtin_amdgcn_perm(word(1), word(0), hi), __builtin_amdgcn_perm(word(3), word(2), hi),
                     __builtin_amdgcn_perm(word(5), word(4), hi), __builtin_amdgcn_perm(word(7), word(6), hi)};
#pragma unroll
        for (int piece = 2; piece >= 0; --piece)
#pragma unroll
          for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int k = 0; k < State<H>::kSets; ++k)
              st.sum[k][2 * d + e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  __builtin_bit_cast(bf16x8, w[k][piece]), __builtin_bit_cast(bf16x8, f[e]),
                  st.sum[k][2 * d + e], 0, 0, 0);
      });
    } else {
      unrolled<0, kUnroll>([&](auto t) __attribute__((always_inline)) {
        const float f[8] = {bf16_lo(x[t].x), bf16_hi(x[t].x), bf16_lo(x[t].y), bf16_hi(x[t].y),
                            bf16_lo(x[t].z), bf16_hi(x[t].z), bf16_lo(x[t].w), bf16_hi(x[t].w)};
        if (s + t < b)                // a used-up destination reads row 0, which may be anything
          unrolled<0, H>([&](auto h) __attribute__((always_inline)) {
            const float w = row_bcast<t + (H > 1 ? 8 * (h / HH) : 0)>(p[h % HH]);
#pragma unroll
            for (int e = 0; e < 8; ++e) st.sum[h / 4][e][h % 4] = fmaf(w, f[e], st.sum[h / 4][e][h % 4]);
          });
      });
    }
  }
}

// The tile's sums, (row, head, k) with kPitch floats a head, through W and out.
__host__ __device__ constexpr int head_pitch(int K) { return (K + 7) / 8 * 8 + 4; }

template <int H>
__device__ __forceinline__ void put_state(const GatInputs &A, float *sums, const State<H> &st, bool any) {
  constexpr int HH = State<H>::HH;
  const int j = threadIdx.x & (kLanes - 1), pitch = head_pitch(A.K);
  float *mine = sums + (threadIdx.x / kLanes) * (H * pitch) + 8 * j;
  unrolled<0, H>([&](auto h) __attribute__((always_inline)) {
    const float l = row_bcast<(H > 1 ? 8 * (h / HH) : 0)>(st.l[h % HH]);
    const float inv = any ? 1.0f / l : 0.0f;       // no edges: a row of zeros
    if (8 * j < A.K) {
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = 8 * j + e < A.K ? st.sum[h / 4][e][h % 4] * inv : 0.0f;
      *reinterpret_cast<float4 *>(mine + h * pitch) = make_float4(v[0], v[1], v[2], v[3]);
      *reinterpret_cast<float4 *>(mine + h * pitch + 4) = make_float4(v[4], v[5], v[6], v[7]);
    }
  });
}

__device__ __forceinline__ float activated(float v, int act) {
  return act == GA_ACT_RELU ? relu_keep_nan(v) : act == GA_ACT_ELU ? elu(v) : v;
}

// A row that no edge leads to is zeros whatever W holds, and zeros times a W that is not finite are
// not: my 16 lanes store it, the product leaves it out.  (A mark in the product's stores instead
// cost the pass over 64.3 M edges 35 of 3180 us.)
__device__ __forceinline__ void store_zeros(const GatInputs &A, int heads, int node) {
  const int M = heads * A.dim;
  for (int c = 4 * (threadIdx.x & (kLanes - 1)); c < M; c += 4 * kLanes)
    *reinterpret_cast<uint2 *>(A.out + (int64_t)node * M + c) = make_uint2(0u, 0u);
}

template <int H, int C>
__device__ __forceinline__ void project(const GatInputs &A, const float *sums, const int *nodes) {
  const int lane = threadIdx.x & (kWave - 1), n = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int M = H * A.dim, pitch = head_pitch(A.K);
  for (int ch = wave; ch < M / (16 * C); ch += kBlock / kWave) {
    const int head = ch * 16 * C / A.dim;
    const float *row = sums + n * (H * pitch) + head * pitch + 8 * q;
    const uint4 *w = A.packed + (int64_t)ch * C * A.ksteps * kWave + lane;
    floatx4 acc[C];
#pragma unroll
    for (int c = 0; c < C; ++c) acc[c] = floatx4{0, 0, 0, 0};
    for (int ks = 0; ks < A.ksteps; ++ks) {
      uint4 wf[C];
#pragma unroll
      for (int c = 0; c < C; ++c) wf[c] = w[(c * A.ksteps + ks) * kWave];
      float4 lo = make_float4(0.0f, 0.0f, 0.0f, 0.0f), up = lo;
      if (32 * ks + 8 * q < A.K) {
        lo = *reinterpret_cast<const float4 *>(row + 32 * ks);
        up = *reinterpret_cast<const float4 *>(row + 32 * ks + 4);
      }
      const float v[8] = {lo.x, lo.y, lo.z, lo.w, up.x, up.y, up.z, up.w};
      uint4 p[3];
      split8(v, p[0], p[1], p[2]);
#pragma unroll
      for (int k = 2; k >= 0; --k)
#pragma unroll
        for (int c = 0; c < C; ++c)
          acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, p[k]),
                                                           __builtin_bit_cast(bf16x8, wf[c]), acc[c], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int node = nodes[4 * q + i];
      if (node < 0) continue;
      bf16_t *o = A.out + (int64_t)node * M + ch * 16 * C + n * C;
      float v[C];
#pragma unroll
      for (int c = 0; c < C; ++c) v[c] = activated(acc[c][i], A.act);
      if constexpr (C == 4)
        *reinterpret_cast<uint2 *>(o) = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
      else if constexpr (C == 2)
        *reinterpret_cast<uint32_t *>(o) = pack_bf16(v[0], v[1]);
      else
        *o = (bf16_t)f32_to_bf16_bits(v[0]);
    }
  }
}

template <int H>
__device__ __forceinline__ void project_tile(const GatInputs &A, const float *sums, const int *nodes) {
  if (A.dim >= 64) project<H, 4>(A, sums, nodes);
  else if (A.dim == 32) project<H, 2>(A, sums, nodes);
  else project<H, 1>(A, sums, nodes);
}

// Wavefronts per SIMD: four (116 registers with four heads; left to itself the compiler takes
// enough for three, 3.45 against 3.18 ms on 64.3 M edges, and five spill), three for eight heads.
template <int H>
__global__ __launch_bounds__(kBlock, H == 8 ? 3 : 4) void gat_inputs_kernel(GatInputs A) {
  extern __shared__ __attribute__((aligned(16))) float sums[];
  __shared__ __attribute__((aligned(16))) WeightSlots<H> slots;
  __shared__ int nodes[kTileRows];
  if (threadIdx.x < 8) slots.zero[threadIdx.x] = 0.0f;
  __syncthreads();
  const bool finite = *A.not_finite == 0;
  constexpr int HH = State<H>::HH;
  const int group = threadIdx.x / kLanes, j = threadIdx.x & (kLanes - 1);
  const rsrc_t table = make_rsrc(A.table, A.table_bytes);
  State<H> st;
  if ((int)blockIdx.x < A.piece_blocks) {           // pieces of the long rows
    const int p = blockIdx.x * kTileRows + group, n_pieces = A.piece_first[A.n_long];
    if ((int)blockIdx.x * kTileRows >= n_pieces) return;
    const int2 piece = p < n_pieces ? A.pieces[p] : make_int2(0, 0);
    // the long row the piece belongs to
    int lo = 0, up = A.n_long;
    while (up - lo > 1) {
      const int mid = (lo + up) >> 1;
      if (A.piece_first[mid] <= p) lo = mid; else up = mid;
    }
    const int node = A.rows[A.n_light + lo].x;
    if (finite) walk<H, true>(A, table, piece.x, piece.y, A.er + (int64_t)node * H, slots, st);
    else walk<H, false>(A, table, piece.x, piece.y, A.er + (int64_t)node * H, slots, st);
    if (p >= n_pieces) return;
    float *o = A.partial + (int64_t)p * State<H>::kFloats;
    unrolled<0, H>([&](auto h) __attribute__((always_inline)) {
      const floatx4(&v)[8] = st.sum[h / 4];
      *reinterpret_cast<float4 *>(o + h * kMaxK + 8 * j) = make_float4(v[0][h % 4], v[1][h % 4], v[2][h % 4], v[3][h % 4]);
      *reinterpret_cast<float4 *>(o + h * kMaxK + 8 * j + 4) = make_float4(v[4][h % 4], v[5][h % 4], v[6][h % 4], v[7][h % 4]);
    });
    if ((j & 7) == 0 && (H > 1 || j == 0))
#pragma unroll
      for (int i = 0; i < HH; ++i) {
        o[H * kMaxK + (j >> 3) * HH + i] = st.m[i];
        o[H * kMaxK + H + (j >> 3) * HH + i] = st.l[i];
      }
    return;
  }
  const int at = (blockIdx.x - A.piece_blocks) * kTileRows + group;
  int4 row = make_int4(-1, 0, 0, 0);
  if (at < A.n_light) row = A.rows[at];
  const bool any = row.z > row.y;
  if (j == 0) nodes[group] = any ? row.x : -1;
  const float *er = A.er + (int64_t)(row.x < 0 ? 0 : row.x) * H;
  if (finite) walk<H, true>(A, table, row.y, row.z, er, slots, st);
  else walk<H, false>(A, table, row.y, row.z, er, slots, st);
  put_state<H>(A, sums, st, any);
  if (!any && row.x >= 0) store_zeros(A, H, row.x);
  __syncthreads();
  project_tile<H>(A, sums, nodes);
}

// The long rows: the states of their pieces in order, then as above.
template <int H>
__global__ __launch_bounds__(kBlock) void gat_inputs_long_kernel(GatInputs A) {
  extern __shared__ __attribute__((aligned(16))) float sums[];
  __shared__ int nodes[kTileRows];
  constexpr int HH = State<H>::HH;
  const int group = threadIdx.x / kLanes, j = threadIdx.x & (kLanes - 1);
  const int hp = H > 1 ? j >> 3 : 0;
  const int at = blockIdx.x * kTileRows + group;
  State<H> st;
  st.clear();
  int node = -1;
  if (at < A.n_long) {
    node = A.rows[A.n_light + at].x;
    const int p1 = A.piece_first[at + 1];
    constexpr int F = 4;              // states at a time: their loads are in flight together
    for (int p = A.piece_first[at]; p < p1; p += F) {
      const float *o[F];
      float old[HH], add[F][HH];
#pragma unroll
      for (int f = 0; f < F; ++f) o[f] = A.partial + (int64_t)min(p + f, p1 - 1) * State<H>::kFloats;
#pragma unroll
      for (int i = 0; i < HH; ++i) {
        float m[F], l[F], top = st.m[i];
#pragma unroll
        for (int f = 0; f < F; ++f) {
          m[f] = p + f < p1 ? o[f][H * kMaxK + hp * HH + i] : -INFINITY;
          l[f] = o[f][H * kMaxK + H + hp * HH + i];
        }
#pragma unroll
        for (int f = 0; f < F; ++f) top = fmaxf(top, m[f]);
        const float ref = finite_or_zero(top);
        old[i] = __expf(st.m[i] - ref);
        st.l[i] *= old[i];
#pragma unroll
        for (int f = 0; f < F; ++f) {
          add[f][i] = __expf(m[f] - ref);
          st.l[i] += l[f] * add[f][i];
        }
        st.m[i] = top;
      }
      unrolled<0, H>([&](auto h) __attribute__((always_inline)) {
        constexpr int src = H > 1 ? 8 * (h / HH) : 0;
        const float so = row_bcast<src>(old[h % HH]);
        float4 lo[F], up[F];
#pragma unroll
        for (int f = 0; f < F; ++f) {
          lo[f] = *reinterpret_cast<const float4 *>(o[f] + h * kMaxK + 8 * j);
          up[f] = *reinterpret_cast<const float4 *>(o[f] + h * kMaxK + 8 * j + 4);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) st.sum[h / 4][e][h % 4] *= so;
#pragma unroll
        for (int f = 0; f < F; ++f) {
          const float sn = row_bcast<src>(add[f][h % HH]);
          const float v[8] = {lo[f].x, lo[f].y, lo[f].z, lo[f].w, up[f].x, up[f].y, up[f].z, up[f].w};
#pragma unroll
          for (int e = 0; e < 8; ++e) st.sum[h / 4][e][h % 4] = fmaf(v[e], sn, st.sum[h / 4][e][h % 4]);
        }
      });
    }
  }
  if (j == 0) nodes[group] = node;
  put_state<H>(A, sums, st, node >= 0);
  __syncthreads();
  project_tile<H>(A, sums, nodes);
}

// ------------------------------------------------------------------------- the plan ----
// rows with at most `longest` slots get the key longest - length, longer ones longest + 1
__global__ __launch_bounds__(kBlock) void gat_rows_keys_kernel(const int32_t *__restrict__ pointer,
                                                               int64_t n_rows, int longest,
                                                               int64_t *__restrict__ key) {
  const int64_t v = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (v >= n_rows) return;
  const int d = pointer[v + 1] - pointer[v];
  key[v] = d <= longest ? longest - d : longest + 1;
}

__global__ __launch_bounds__(kBlock) void gat_rows_fill_kernel(const int32_t *__restrict__ pointer,
                                                               const int32_t *__restrict__ order,
                                                               int64_t n_rows,
                                                               const int32_t *__restrict__ light_end,
                                                               int4 *__restrict__ rows,
                                                               int32_t *__restrict__ n_light) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i == 0) *n_light = *light_end;
  if (i >= n_rows) return;
  const int v = order[i];
  rows[i] = make_int4(v, pointer[v], pointer[v + 1], 0);
}

// one workgroup: pieces of the long rows, in order
__global__ __launch_bounds__(1024) void gat_pieces_kernel(const int4 *__restrict__ rows, int n_long,
                                                          int longest, int32_t *__restrict__ piece_first,
                                                          int2 *__restrict__ pieces) {
  __shared__ int32_t wave_sum[1024 / kWave];
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  int32_t before = 0;
  for (int base = 0; base < n_long; base += 1024) {
    const int i = base + threadIdx.x;
    const int4 row = i < n_long ? rows[i] : make_int4(0, 0, 0, 0);
    const int32_t c = (row.z - row.y + longest - 1) / longest;
    int32_t incl = c;
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
    if (i < n_long) {
      const int32_t first = in_front + incl - c;
      piece_first[i] = first;
      for (int k = 0; k < c; ++k)
        pieces[first + k] = make_int2(row.y + k * longest, min(row.y + (k + 1) * longest, row.z));
    }
    before += all;
    __syncthreads();
  }
  if (threadIdx.x == 0) piece_first[n_long] = before;
}

inline size_t round_up(size_t v) { return (v + 255) & ~(size_t)255; }

// Everything of one call but the partial states and the result.
struct InputsLayout {
  int row_bytes, stride, ksteps;
  size_t table, er, packed, wa, flag, partial, total;
};
bool inputs_layout(int64_t n_rows, int64_t K, int64_t heads, int64_t dim, int64_t n_pieces, InputsLayout &L) {
  if (heads != 1 && heads != 2 && heads != 4 && heads != 8) return false;
  if (dim != 16 && dim != 32 && (dim % 64 != 0 || dim > 256)) return false;
  if (K <= 0 || 2 * K + 4 * heads > 2 * kMaxK) return false;
  L.row_bytes = 2 * K + 4 * heads <= kMaxK ? kMaxK : 2 * kMaxK;
  // rows of two 128-byte lines meet in few memory channels where ids are structured: a line
  // further apart 3.64 -> 3.27 ms over 64.3 M R-MAT edges (with half a line 3.50; node bits folded
  // onto the lowest ones instead 5.1)
  L.stride = L.row_bytes == 2 * kMaxK && n_rows * L.row_bytes > (4 << 20) ? 3 * kMaxK : L.row_bytes;
  L.ksteps = (int)((K + 31) / 32);
  if (n_rows * L.stride > 0x7fffffff) return false;
  size_t off = 0;
  L.table = off;    off += round_up((size_t)n_rows * L.stride);
  L.er = off;       off += round_up((size_t)n_rows * heads * 4);
  L.packed = off;   off += round_up((size_t)(heads * dim / 16) * L.ksteps * kWave * 16);
  L.wa = off;       off += round_up((size_t)2 * heads * kMaxK * 4);
  L.flag = off;     off += 256;
  L.partial = off;  off += round_up((size_t)n_pieces * (heads * kMaxK + 2 * heads) * 4);
  L.total = off;
  return true;
}

template <int H>
int launch_inputs(const bf16_t *X, const bf16_t *W, const float *a_l, const float *a_r, GatInputs &A,
                  float *er, float *wa, uint4 *packed, char *table, int32_t *flag, int64_t n_rows, hipStream_t s) {
  A.not_finite = flag;
  const int packs = H * A.dim / 16 * A.ksteps * kWave + 2 * H * kMaxK;
  hipLaunchKernelGGL(gat_inputs_weights_kernel, dim3((packs + kBlock - 1) / kBlock), dim3(kBlock), 0, s, W,
                     a_l, a_r, A.K, A.ksteps, H, A.dim, packed, wa, flag);
  const int64_t row_blocks = (n_rows + kTileRows - 1) / kTileRows;
  const dim3 rgrid((unsigned)(row_blocks < 4096 ? row_blocks : 4096));
#define GA_ROWS(PIECE)                                                                              \
  hipLaunchKernelGGL((gat_inputs_rows_kernel<H, PIECE>), rgrid, dim3(kBlock), 0, s, X, wa, n_rows, A.K, \
                     A.row_bytes, A.stride, table, er, flag)
  if (A.K % 8 == 0 && aligned(X, 16)) GA_ROWS(8);
  else if (A.K % 4 == 0 && aligned(X, 8)) GA_ROWS(4);
  else if (A.K % 2 == 0 && aligned(X, 4)) GA_ROWS(2);
  else GA_ROWS(1);
#undef GA_ROWS
  const size_t lds = (size_t)kTileRows * H * head_pitch(A.K) * sizeof(float);
  static_assert(kTileRows * H * head_pitch(kMaxK - 2 * H) * sizeof(float) + sizeof(WeightSlots<H>) +
                        kTileRows * sizeof(int) <= 64 * 1024,
                "more than a launch gets without asking");
  A.piece_blocks = (A.n_pieces + kTileRows - 1) / kTileRows;
  const int tiles = (A.n_light + kTileRows - 1) / kTileRows;
  if (A.piece_blocks + tiles > 0)
    hipLaunchKernelGGL((gat_inputs_kernel<H>), dim3((unsigned)(A.piece_blocks + tiles)), dim3(kBlock), lds, s, A);
  if (A.n_long > 0)
    hipLaunchKernelGGL((gat_inputs_long_kernel<H>), dim3((unsigned)((A.n_long + kTileRows - 1) / kTileRows)),
                       dim3(kBlock), lds, s, A);
  return launch_status();
}

struct RowsLayout {
  size_t key, order, pointer, status, group, group_bytes, total;
};
RowsLayout rows_layout(int64_t n_rows, int64_t longest) {
  RowsLayout L;
  L.group_bytes = ga_group_edges_workspace_bytes(longest + 2, n_rows);
  size_t off = 0;
  L.key = off;      off += round_up((size_t)n_rows * 8);
  L.order = off;    off += round_up((size_t)n_rows * 4);
  L.pointer = off;  off += round_up((size_t)(longest + 3) * 4);
  L.status = off;   off += 256;
  L.group = off;    off += round_up(L.group_bytes);
  L.total = off;
  return L;
}

}  // namespace
}  // namespace ga

extern "C" {

int64_t ga_gat_rows_longest(int64_t n_edges) {
  // 16 lanes walk a row, 16,384 such groups are resident at a time: a piece of twice a group's
  // share ends with the others, between 256 and 2,048 slots (400,000 edges, eight heads of 64:
  // 64 slots 332 us, 128 193, 256 149: the states of more pieces are added one after the other)
  int64_t c = 256;
  while (c < 2048 && c * 8192 < n_edges) c *= 2;
  return c;
}

size_t ga_gat_rows_workspace_bytes(int64_t n_rows, int64_t longest) {
  if (n_rows < 0 || n_rows > 0x7ffffffe || longest < 1 || longest > (1 << 20)) return 0;
  return ga::rows_layout(n_rows, longest).total;
}

int ga_gat_rows_build(const int32_t *pointer, int64_t n_rows, int64_t longest, int32_t *rows,
                      int32_t *n_light, void *workspace, size_t workspace_bytes, ga_stream_t stream) {
  using namespace ga;
  if (n_rows <= 0 || n_rows > 0x7ffffffe || longest < 1 || longest > (1 << 20)) return GA_EINVAL;
  if (!pointer || !rows || !n_light) return GA_EINVAL;
  if (!aligned(rows, 16) || !aligned(n_light, 4)) return GA_EALIGN;
  const RowsLayout L = rows_layout(n_rows, longest);
  if (!workspace || workspace_bytes < L.total || !aligned(workspace, 256)) return GA_EWORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  char *ws = (char *)workspace;
  int64_t *key = (int64_t *)(ws + L.key);
  int32_t *order = (int32_t *)(ws + L.order), *ptr = (int32_t *)(ws + L.pointer);
  const unsigned blocks = (unsigned)((n_rows + kBlock - 1) / kBlock);
  hipLaunchKernelGGL(gat_rows_keys_kernel, dim3(blocks), dim3(kBlock), 0, s, pointer, n_rows, (int)longest, key);
  const int rc = ga_group_edges(key, nullptr, longest + 2, n_rows, ptr, nullptr, order,
                                (int32_t *)(ws + L.status), ws + L.group, L.group_bytes, stream);
  if (rc != GA_OK) return rc;
  hipLaunchKernelGGL(gat_rows_fill_kernel, dim3(blocks), dim3(kBlock), 0, s, pointer, order, n_rows,
                     ptr + longest + 1, (int4 *)rows, n_light);
  return launch_status();
}

int ga_gat_pieces_build(const int32_t *long_rows, int64_t n_long, int64_t longest,
                        int32_t *piece_first, int32_t *pieces, ga_stream_t stream) {
  using namespace ga;
  if (n_long < 0 || n_long > 0x7ffffffe || longest < 1 || longest > (1 << 20)) return GA_EINVAL;
  if (!piece_first || (n_long > 0 && (!long_rows || !pieces))) return GA_EINVAL;
  if (!aligned(long_rows, 16) || !aligned(pieces, 8)) return GA_EALIGN;
  hipLaunchKernelGGL(gat_pieces_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, (const int4 *)long_rows,
                     (int)n_long, (int)longest, piece_first, (int2 *)pieces);
  return launch_status();
}

size_t ga_gat_inputs_workspace_bytes(int64_t n_rows, int64_t K, int64_t heads, int64_t dim, int64_t n_pieces) {
  ga::InputsLayout L;
  if (n_rows < 0 || n_rows > 0x7ffffffe || n_pieces < 0 || n_pieces > 0x7ffffffe ||
      !ga::inputs_layout(n_rows, K, heads, dim, n_pieces, L))
    return 0;
  return L.total;
}

int ga_gat_inputs(const int32_t *rows, int64_t n_light, const int32_t *piece_first, const int32_t *pieces,
                  int64_t n_pieces, const int32_t *nbr, const void *X, const void *W, const float *a_l,
                  const float *a_r, void *out, int64_t n_rows, int64_t K, int64_t heads, int64_t dim,
                  float slope, int activation, void *workspace, size_t workspace_bytes,
                  ga_stream_t stream) {
  using namespace ga;
  if (activation < GA_ACT_NONE || activation > GA_ACT_ELU) return GA_EINVAL;
  if (n_rows < 0 || n_rows > 0x7ffffffe || n_light < 0 || n_light > n_rows || n_pieces < 0) return GA_EINVAL;
  InputsLayout L;
  if (!inputs_layout(n_rows, K, heads, dim, n_pieces, L)) return GA_EUNSUPPORTED;
  if (n_rows == 0) return GA_OK;
  const int64_t n_long = n_rows - n_light;
  if (!rows || !nbr || !X || !W || !a_l || !a_r || !out || (n_long > 0 && (!piece_first || !pieces || n_pieces == 0)))
    return GA_EINVAL;
  if (!aligned(rows, 16) || !aligned(pieces, 8) || !aligned(X, 2) || !aligned(W, 2) || !aligned(out, 8))
    return GA_EALIGN;
  if (!workspace || workspace_bytes < L.total || !aligned(workspace, 256)) return GA_EWORKSPACE;
  char *ws = (char *)workspace;
  GatInputs A{};
  A.rows = (const int4 *)rows;
  A.pieces = (const int2 *)pieces;
  A.piece_first = piece_first;
  A.nbr = nbr;
  A.table = ws + L.table;
  A.er = (const float *)(ws + L.er);
  A.packed = (const uint4 *)(ws + L.packed);
  A.partial = (float *)(ws + L.partial);
  A.out = (bf16_t *)out;
  A.table_bytes = (uint64_t)n_rows * L.stride;
  A.n_light = (int)n_light;
  A.n_long = (int)n_long;
  A.n_pieces = n_long > 0 ? (int)n_pieces : 0;
  A.K = (int)K;
  A.ksteps = L.ksteps;
  A.dim = (int)dim;
  A.row_bytes = L.row_bytes;
  A.stride = L.stride;
  A.act = activation;
  A.slope = slope;
#define GA_INPUTS(H)                                                                                  \
  return launch_inputs<H>((const bf16_t *)X, (const bf16_t *)W, a_l, a_r, A, (float *)(ws + L.er),     \
                          (float *)(ws + L.wa), (uint4 *)(ws + L.packed), ws + L.table,                \
                          (int32_t *)(ws + L.flag), n_rows,                                            \
                          (hipStream_t)stream)
  switch (heads) {
    case 1: GA_INPUTS(1);
    case 2: GA_INPUTS(2);
    case 4: GA_INPUTS(4);
    default: GA_INPUTS(8);
  }
#undef GA_INPUTS
}

}  // extern "C"
