// Fused GAT aggregation for gfx950: u_add_v -> leaky_relu -> edge softmax ->
// u_mul_e sum in one pass over the in-adjacency, nothing per-edge materialised.
//
// Same run-based schedule as the SpMM (row_runs.h: equal runs of slots, one lane
// group per run, rows shared between runs chained in LDS and, across
// workgroups, by a second kernel), with an online softmax state per lane:
// running maximum m, running denominator l and the un-normalised weighted sum
// acc.  Two states merge as
//   M = max(m1, m2); l = l1 e^(m1-M) + l2 e^(m2-M); acc likewise,
// so partial rows combine exactly like partial sums, in run order.
//
// The same pass with per-edge operands (EDGE): the logits are given per edge
// and the weighted rows are per-edge rows, both read through the edge-id
// column: out[v] = sum_e softmax_v(logit)[e] * m[e], the SegmentSoftmax ->
// mul -> SpMMEdge tail of examples/HGT/HGT.py:50-53 with no attention tensor.
#include <mutex>

#include "row_runs.h"

namespace ga {
namespace {

__device__ __forceinline__ float leaky(float t, float slope) {
  return t >= 0.0f ? t : t * slope;
}

// The running maximum as the point the exponentials are taken from: while every
// logit seen so far is -inf (masked edges) the maximum is -inf too and
// exp(-inf - -inf) would be NaN; taken from 0 instead, such edges weigh 0 and a
// later finite logit rescales the (empty) state by exp(-inf) = 0.  A row whose
// logits are all -inf ends with a zero denominator and yields NaN, as the
// reference's softmax does (segment_softmax_kernel.cu:9-49).
__device__ __forceinline__ float finite_or_zero(float m) {
  return m == -INFINITY ? 0.0f : m;
}

// State per lane: VEC un-normalised weighted sums, then the running maximum m
// and the running denominator l of the lane's head.
// MODE selects where the logits come from:
//   kGatNode  el[src] + er[dst] through leaky_relu (the GAT chain),
//   kGatEdge  given per edge (EDGE operands, see the header comment),
//   kGatFromZ <z[src, h, :], a_l[h, :]> + er[dst] through leaky_relu: the source
//             term is recomputed from the row that is gathered anyway instead of
//             being gathered itself -- a separate (N, heads) table costs one more
//             memory sector per edge once it no longer fits the caches.
constexpr int kGatNode = 0, kGatEdge = 1, kGatFromZ = 2;

// Sum over `lanes` adjacent lanes (a power of two <= 16, aligned), in every lane.
__device__ __forceinline__ float lanes_sum(float v, int lanes) {
  if (lanes >= 2) v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));
  if (lanes >= 4) v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, true));
  if (lanes >= 8) v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x141, 0xF, 0xF, true));
  if (lanes >= 16) v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x140, 0xF, 0xF, true));
  return v;
}

// d[t] of the GL lanes of a head, summed over them: lane i gets the sum of slot (i & 7).
// Halving the slots a lane keeps at every step costs as many instructions as summing all
// eight in every lane, and leaves each sum in one lane.
template <int CTRL>
__device__ __forceinline__ float plus_other(float v) {      // v plus the DPP partner's
  return v + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}
template <int GL>
__device__ __forceinline__ float sum_by_slot(float (&d)[kUnroll], int sub) {
  if constexpr (GL == 16) {
#pragma unroll
    for (int t = 0; t < kUnroll; ++t) d[t] = plus_other<0x140>(d[t]);         // row_mirror
  }
  float e[4], f[2];
#pragma unroll
  for (int t = 0; t < 4; ++t) {                                               // row_half_mirror
    const float lo = plus_other<0x141>(d[t]), hi = plus_other<0x141>(d[4 + t]);
    e[t] = sub & 4 ? hi : lo;
  }
#pragma unroll
  for (int t = 0; t < 2; ++t) {                                               // quad_perm [2,3,0,1]
    const float lo = plus_other<0x4E>(e[t]), hi = plus_other<0x4E>(e[2 + t]);
    f[t] = sub & 2 ? hi : lo;
  }
  const float lo = plus_other<0xB1>(f[0]), hi = plus_other<0xB1>(f[1]);       // quad_perm [1,0,3,2]
  return sub & 1 ? hi : lo;
}

// SPREAD: the lane's features lie a lane-group width apart (rows that 16-byte
// accesses do not tile); they share the lane's one (m, l) pair, i.e. one head.
// ACT: the activation compiled into the row store (GA_ACT_RELU / GA_ACT_ELU), or
// kActRuntime = the one named by Args::act (the less common lane layouts; one build
// for all three).  The compiled-in forms keep the dead branches out of the kernel:
// the store sits at five places of the run loop, under divergence, so its length is
// paid once per closed row and wavefront, not per element.
constexpr int kActRuntime = -1;
template <typename T, int VEC, int MODE = kGatNode, bool SPREAD = false, int ACT = kActRuntime,
          int GL = 0>
struct GatPolicy {
  static constexpr bool EDGE = MODE == kGatEdge;
  typedef T out_t;
  static constexpr int kVec = VEC;
  static constexpr int kState = VEC + 2;
  static constexpr bool kSpread = SPREAD;
  static constexpr int kGL = GL;
  struct Args {
    const int32_t *nbr;   // kGatEdge: the edge-id column, or null when slot = edge id
    const float *el;      // kGatEdge: per-edge logits (E, heads); kGatFromZ: a_l (heads*dph)
    const float *er;      // kGatEdge: unused
    const T *z;           // kGatEdge: per-edge rows (E, heads*dph)
    int heads;
    int dph;
    float slope;
    bool ids_vec;   // row_of_slot and nbr are 16-byte aligned
    int head_lanes; // kGatFromZ: lanes that share a head (dph / VEC)
    int stride_shift;   // SPREAD: log2 of the lanes per group, set by the launcher
    int act;            // GA_ACT_*: applied to the finished row before it is stored
    int z_stride;       // elements from a row of z to the next
  };
  static __device__ __forceinline__ void init(float (&st)[VEC + 2]) {
#pragma unroll
    for (int v = 0; v < VEC; ++v) st[v] = 0.0f;
    st[VEC] = -INFINITY;
    st[VEC + 1] = 0.0f;
  }
  static __device__ __forceinline__ void merge(float (&dst)[VEC + 2], const float *src) {
    const float nm = fmaxf(dst[VEC], src[VEC]);
    const float ref = finite_or_zero(nm);
    const float sa = __expf(dst[VEC] - ref), sb = __expf(src[VEC] - ref);
#pragma unroll
    for (int v = 0; v < VEC; ++v) dst[v] = dst[v] * sa + src[v] * sb;
    dst[VEC + 1] = dst[VEC + 1] * sa + src[VEC + 1] * sb;
    dst[VEC] = nm;
  }
  static __device__ __forceinline__ void finish(const float (&st)[VEC + 2], float (&o)[VEC]) {
    const float inv = 1.0f / st[VEC + 1];
#pragma unroll
    for (int v = 0; v < VEC; ++v) o[v] = st[v] * inv;
  }
  static __device__ __forceinline__ void empty_row(float (&o)[VEC]) {
#pragma unroll
    for (int v = 0; v < VEC; ++v) o[v] = 0.0f;
  }
  static __device__ __forceinline__ void emit(const Args &A, out_t *out, int64_t row, int feat,
                                              int f0, const float (&st)[kState]) {
    const int act = ACT == kActRuntime ? A.act : ACT;
    if (act == GA_ACT_NONE) {
      emit_row<GatPolicy>(out, row, feat, f0, st, A.stride_shift);
      return;
    }
    // the activation of the layer (relu, or elu with alpha = 1) on the fp32 row, before
    // it is rounded and stored: the row is not written and read again for it
    typedef RowIO<out_t, VEC, SPREAD> IO;
    float o[VEC];
    finish(st, o);
#pragma unroll
    for (int v = 0; v < VEC; ++v) o[v] = act == GA_ACT_ELU ? elu(o[v]) : relu_keep_nan(o[v]);
    IO::store(out + row * feat + f0, o, IO::lane(A.stride_shift, feat - f0));
  }
  static __device__ __forceinline__ void emit_empty(const Args &A, out_t *out, int64_t row,
                                                    int feat, int f0) {
    emit_empty_row<GatPolicy>(out, row, feat, f0, A.stride_shift);
  }

  template <class Close>
  static __device__ __forceinline__ void walk(const Args &A,
                                              const int32_t *__restrict__ row_of_slot,
                                              int64_t a, int64_t b, int f0, int feat,
                                              float (&st)[VEC + 2], int &cur,
                                              Close &&close_segment) {
    static_assert(!(SPREAD && MODE == kGatFromZ), "the per-head dot product needs consecutive features");
    typedef RowIO<T, VEC, SPREAD> IO;
    const typename IO::lane_t ln = IO::lane(A.stride_shift, feat - f0);
    const int h = SPREAD ? 0 : f0 / A.dph;
    float al[VEC];
#pragma unroll
    for (int v = 0; v < VEC; ++v) al[v] = MODE == kGatFromZ ? A.el[f0 + v] : 0.0f;
    if constexpr (GL > 0) {
      typedef GroupCol<GL> Col;
      const int sub = threadIdx.x & (GL - 1);
      GroupIds<GL> ids, next;
      ids.load(row_of_slot, A.nbr, a, b, sub);
      for (int64_t j = a; j < b; j += kUnroll) {
        typename IO::raw_t x[kUnroll];
        float sv;                   // lane i holds the logit of slot (i & 7)
        if constexpr (MODE == kGatFromZ) {
          sv = A.er[(int64_t)ids.my_row(sub) * A.heads + h];
        } else if constexpr (MODE == kGatEdge) {
          if constexpr (GL == 16) {     // lanes 8 .. 15 hold the indices
            sv = A.el[(int64_t)(sub & 8 ? ids.row : 0) * A.heads + h];
            const float o = other_half(sv);
            sv = sub & 8 ? sv : o;
          } else {
            sv = A.el[(int64_t)ids.idx * A.heads + h];
          }
        } else if constexpr (GL == 16) {    // one load for both terms, each from its half
          sv = (sub & 8 ? A.el : A.er)[(int64_t)ids.row * A.heads + h];
          sv = leaky(sv + other_half(sv), A.slope);
        } else {
          sv = leaky(A.el[(int64_t)ids.idx * A.heads + h] + A.er[(int64_t)ids.row * A.heads + h],
                     A.slope);
        }
        static_for<kUnroll>([&](auto t) {
          x[t] = IO::load(A.z + (int64_t)ids.template index_of<t>() * A.z_stride + f0, ln);
        });
        // the columns of the next batch arrive while this batch's rows are added; asked for
        // after the gathers (GroupIds)
        __builtin_amdgcn_sched_barrier(0);
        next.load(row_of_slot, A.nbr, j + kUnroll, b, sub);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (MODE == kGatFromZ) {
          // every live lane of a head runs this together (heads tile the row)
          float d[kUnroll];
#pragma unroll
          for (int t = 0; t < kUnroll; ++t) {
            float xf[VEC];
            IO::widen(x[t], xf);
            d[t] = 0.0f;
#pragma unroll
            for (int v = 0; v < VEC; ++v) d[t] = fmaf(xf[v], al[v], d[t]);
          }
          sv = leaky(sum_by_slot<GL>(d, sub) + sv, A.slope);
        }
        const bool one_row = j + kUnroll <= b && ids.template row_of<0>() == cur &&
                             ids.template row_of<kUnroll - 1>() == cur;
        if (one_row) {
          // whole batch inside the open row (rows are sorted): one rescale
          const float nm = fmaxf(st[VEC], Col::max(sv));
          const float ref = finite_or_zero(nm);
          const float sc = __expf(st[VEC] - ref);
          st[VEC + 1] *= sc;
#pragma unroll
          for (int v = 0; v < VEC; ++v) st[v] *= sc;
          st[VEC] = nm;
          const float pv = __expf(sv - ref);    // one exponential per slot, not per slot and lane
          st[VEC + 1] += Col::sum(pv);
          static_for<kUnroll>([&](auto t) {
            const float p = Col::template get<t>(pv);
            float xf[VEC];
            IO::widen(x[t], xf);
#pragma unroll
            for (int v = 0; v < VEC; ++v) st[v] = fmaf(p, xf[v], st[v]);
          });
        } else {
          static_for<kUnroll>([&](auto t) {
            if (j + t < b) {
              const int r = ids.template row_of<t>();
              if (r != cur) {
                close_segment();
                cur = r;
                init(st);
              }
              const float s = Col::template get<t>(sv);
              const float nm = fmaxf(st[VEC], s);
              const float ref = finite_or_zero(nm);
              const float sc = __expf(st[VEC] - ref);
              const float p = __expf(s - ref);
              st[VEC + 1] = st[VEC + 1] * sc + p;
              float xf[VEC];
              IO::widen(x[t], xf);
#pragma unroll
              for (int v = 0; v < VEC; ++v) st[v] = fmaf(p, xf[v], st[v] * sc);
              st[VEC] = nm;
            }
          });
        }
        ids = next;
      }
      return;
    }
    for (int64_t j = a; j < b; j += kUnroll) {
      int r[kUnroll], g[kUnroll];
      float s[kUnroll];
      typename IO::raw_t x[kUnroll];
      load_ids8(row_of_slot, j, b, A.ids_vec, r);
      if (EDGE && !A.nbr) {
#pragma unroll
        for (int t = 0; t < kUnroll; ++t) g[t] = (int)(j + t < b ? j + t : b - 1);
      } else {
        load_ids8(A.nbr, j, b, A.ids_vec, g);
      }
#pragma unroll
      for (int t = 0; t < kUnroll; ++t) {
        x[t] = IO::load(A.z + (int64_t)g[t] * A.z_stride + f0, ln);
        if constexpr (MODE == kGatEdge)
          s[t] = A.el[(int64_t)g[t] * A.heads + h];
        else if constexpr (MODE == kGatNode)
          s[t] = leaky(A.el[(int64_t)g[t] * A.heads + h] + A.er[(int64_t)r[t] * A.heads + h],
                       A.slope);
        else
          s[t] = A.er[(int64_t)r[t] * A.heads + h];
      }
      if constexpr (MODE == kGatFromZ) {
        // every live lane of a head runs this together (heads tile the row)
#pragma unroll
        for (int t = 0; t < kUnroll; ++t) {
          float xf[VEC];
          IO::widen(x[t], xf);
          float d = 0.0f;
#pragma unroll
          for (int v = 0; v < VEC; ++v) d = fmaf(xf[v], al[v], d);
          s[t] = leaky(lanes_sum(d, A.head_lanes) + s[t], A.slope);
        }
      }
      const bool one_row = j + kUnroll <= b && r[0] == cur && r[kUnroll - 1] == cur;
      if (one_row) {
        // whole batch inside the open row (rows are sorted): one rescale
        float bm = s[0];
#pragma unroll
        for (int t = 1; t < kUnroll; ++t) bm = fmaxf(bm, s[t]);
        const float nm = fmaxf(st[VEC], bm);
        const float ref = finite_or_zero(nm);
        const float sc = __expf(st[VEC] - ref);
        st[VEC + 1] *= sc;
#pragma unroll
        for (int v = 0; v < VEC; ++v) st[v] *= sc;
        st[VEC] = nm;
#pragma unroll
        for (int t = 0; t < kUnroll; ++t) {
          const float p = __expf(s[t] - ref);
          st[VEC + 1] += p;
          float xf[VEC];
          IO::widen(x[t], xf);
#pragma unroll
          for (int v = 0; v < VEC; ++v) st[v] = fmaf(p, xf[v], st[v]);
        }
      } else {
#pragma unroll
        for (int t = 0; t < kUnroll; ++t) {
          if (j + t < b) {
            if (r[t] != cur) {
              close_segment();
              cur = r[t];
              init(st);
            }
            const float nm = fmaxf(st[VEC], s[t]);
            const float ref = finite_or_zero(nm);
            const float sc = __expf(st[VEC] - ref);
            const float p = __expf(s[t] - ref);
            st[VEC + 1] = st[VEC + 1] * sc + p;
            float xf[VEC];
            IO::widen(x[t], xf);
#pragma unroll
            for (int v = 0; v < VEC; ++v) st[v] = fmaf(p, xf[v], st[v] * sc);
            st[VEC] = nm;
          }
        }
      }
    }
  }
};

// Dot-product attention over an adjacency: slot i of row r weighs the value row
// v[nbr[i]] with softmax_r(<k[nbr[i]], q[qrow[i]]>), per head; beside the weighted sum
// the row's log-sum-exp is written, so that rows which are pieces of one softmax (the
// (destination, relation) pairs of an HGT layer) can be combined afterwards.  State,
// merge and finish are the fused GAT aggregation's; only the logits differ: a second
// gathered row (k) and the slot's query row, which consecutive slots of a pair share.
template <typename T, int VEC>
struct DotAttnPolicy : GatPolicy<T, VEC, kGatEdge, false> {
  typedef GatPolicy<T, VEC, kGatEdge, false> Base;
  struct Args {
    const int32_t *nbr;    // key / value row of a slot
    const int32_t *qrow;   // query row of a slot
    const T *k, *q, *v;    // rows of heads * dph features
    float *lse;            // (n_rows, heads) or null
    const int32_t *lse_index;   // row r's log-sum-exp goes to row lse_index[r] of lse; null: r
    int heads;
    int dph;
    int head_lanes;        // lanes that share a head (dph / VEC)
    bool ids_vec;          // row_of_slot, nbr and qrow are 16-byte aligned
  };
  static __device__ __forceinline__ void emit(const Args &A, T *out, int64_t row, int feat, int f0,
                                              const float (&st)[VEC + 2]) {
    emit_row<DotAttnPolicy>(out, row, feat, f0, st);
    if (A.lse && f0 % A.dph == 0)
      A.lse[(A.lse_index ? (int64_t)A.lse_index[row] : row) * A.heads + f0 / A.dph] =
          st[VEC] + logf(st[VEC + 1]);
  }
  static __device__ __forceinline__ void emit_empty(const Args &A, T *out, int64_t row, int feat,
                                                    int f0) {
    emit_empty_row<DotAttnPolicy>(out, row, feat, f0);
    if (A.lse && f0 % A.dph == 0)
      A.lse[(A.lse_index ? (int64_t)A.lse_index[row] : row) * A.heads + f0 / A.dph] = -INFINITY;
  }

  template <class Close>
  static __device__ __forceinline__ void walk(const Args &A,
                                              const int32_t *__restrict__ row_of_slot,
                                              int64_t a, int64_t b, int f0, int feat,
                                              float (&st)[VEC + 2], int &cur,
                                              Close &&close_segment) {
    typedef RowIO<T, VEC, false> IO;
    const typename IO::lane_t ln = IO::lane(0, feat - f0);
    for (int64_t j = a; j < b; j += kUnroll) {
      int r[kUnroll], g[kUnroll], qr[kUnroll];
      float s[kUnroll];
      typename IO::raw_t x[kUnroll], kx[kUnroll], qx[kUnroll];
      load_ids8(row_of_slot, j, b, A.ids_vec, r);
      load_ids8(A.nbr, j, b, A.ids_vec, g);
      load_ids8(A.qrow, j, b, A.ids_vec, qr);
#pragma unroll
      for (int t = 0; t < kUnroll; ++t) {
        kx[t] = IO::load(A.k + (int64_t)g[t] * feat + f0, ln);
        qx[t] = IO::load(A.q + (int64_t)qr[t] * feat + f0, ln);
        x[t] = IO::load(A.v + (int64_t)g[t] * feat + f0, ln);
      }
      // every live lane of a head runs this together (heads tile the row)
#pragma unroll
      for (int t = 0; t < kUnroll; ++t) {
        float kf[VEC], qf[VEC];
        IO::widen(kx[t], kf);
        IO::widen(qx[t], qf);
        float d = 0.0f;
#pragma unroll
        for (int v = 0; v < VEC; ++v) d = fmaf(kf[v], qf[v], d);
        s[t] = lanes_sum(d, A.head_lanes);
      }
      const bool one_row = j + kUnroll <= b && r[0] == cur && r[kUnroll - 1] == cur;
      if (one_row) {
        // whole batch inside the open row (rows are sorted): one rescale
        float bm = s[0];
#pragma unroll
        for (int t = 1; t < kUnroll; ++t) bm = fmaxf(bm, s[t]);
        const float nm = fmaxf(st[VEC], bm);
        const float ref = finite_or_zero(nm);
        const float sc = __expf(st[VEC] - ref);
        st[VEC + 1] *= sc;
#pragma unroll
        for (int v = 0; v < VEC; ++v) st[v] *= sc;
        st[VEC] = nm;
#pragma unroll
        for (int t = 0; t < kUnroll; ++t) {
          const float p = __expf(s[t] - ref);
          st[VEC + 1] += p;
          float xf[VEC];
          IO::widen(x[t], xf);
#pragma unroll
          for (int v = 0; v < VEC; ++v) st[v] = fmaf(p, xf[v], st[v]);
        }
      } else {
#pragma unroll
        for (int t = 0; t < kUnroll; ++t) {
          if (j + t < b) {
            if (r[t] != cur) {
              close_segment();
              cur = r[t];
              Base::init(st);
            }
            const float nm = fmaxf(st[VEC], s[t]);
            const float ref = finite_or_zero(nm);
            const float sc = __expf(st[VEC] - ref);
            const float p = __expf(s[t] - ref);
            st[VEC + 1] = st[VEC + 1] * sc + p;
            float xf[VEC];
            IO::widen(x[t], xf);
#pragma unroll
            for (int v = 0; v < VEC; ++v) st[v] = fmaf(p, xf[v], st[v] * sc);
            st[VEC] = nm;
          }
        }
      }
    }
  }
};

template <typename T, int VEC>
int launch_dot_attn(const int32_t *pointer, const int32_t *row_of_slot, const int32_t *nbr,
                    const int32_t *qrow, const void *k, const void *q, const void *v, void *out,
                    float *lse, const int32_t *lse_index, int64_t n_rows, int64_t n_edges, int heads,
                    int dim, float *ws, size_t ws_bytes, hipStream_t stream) {
  typedef DotAttnPolicy<T, VEC> P;
  const int head_lanes = dim / VEC;
  if (dim % VEC != 0 || head_lanes > 16 || (head_lanes & (head_lanes - 1)) != 0)
    return GA_EUNSUPPORTED;
  const bool ids_vec = aligned(row_of_slot, 16) && aligned(nbr, 16) && aligned(qrow, 16);
  typename P::Args args{nbr, qrow, (const T *)k, (const T *)q, (const T *)v, lse, lse_index,
                        heads, dim, head_lanes, ids_vec};
  return launch_runs<P>(args, pointer, row_of_slot, out, n_rows, n_edges, heads * dim, ws,
                        stream, ws_bytes);
}

// bf16 rows of several heads, the same values stored through pack_bf16_opaque: 124 registers and
// four wavefronts per SIMD where the build above takes 150 to 168 and three (125 and four
// while every value was rounded by five instructions).  Fewer wavefronts with more loads of
// their own are the better form on large tables that fill their lane groups: 4 x 64 on 64 M
// R-MAT edges 6737 (four) : 6539 us, on 8 M uniform edges 846 : 797, and of narrow rows (3 x 32 on
// 64 M 3256 : 3157).  Rows of more than 16 lanes that do not (5 x 64 on 11.6 M R-MAT edges 943 :
// 1050, on 12 M uniform edges 1804 : 1950, 3 x 64 on 16 M 936 : 1033) and short lists (4 x 64 on
// 600 k uniform edges 56 : 59, 8 x 64 on 400 k 61 : 67) take this one.
template <int ACT>
struct GatOpaqueStore : GatPolicy<bf16_t, 8, kGatNode, false, ACT, 0> {
  typedef GatPolicy<bf16_t, 8, kGatNode, false, ACT, 0> Base;
  static __device__ __forceinline__ void emit(const typename Base::Args &, bf16_t *out, int64_t row,
                                              int feat, int f0, const float (&st)[Base::kState]) {
    float o[8];
    Base::finish(st, o);
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      if (ACT == GA_ACT_ELU) o[v] = elu(o[v]);
      if (ACT == GA_ACT_RELU) o[v] = relu_keep_nan(o[v]);
    }
    *reinterpret_cast<uint4 *>(out + row * feat + f0) =
        make_uint4(pack_bf16_opaque(o[0], o[1]), pack_bf16_opaque(o[2], o[3]),
                   pack_bf16_opaque(o[4], o[5]), pack_bf16_opaque(o[6], o[7]));
  }
};

template <typename T, int VEC, int MODE = kGatNode, bool SPREAD = false, int ACT = kActRuntime,
          int GL = 0>
int launch_gat(const int32_t *pointer, const int32_t *row_of_slot,
               const int32_t *nbr, const float *el, const float *er,
               const void *z, void *out, int64_t n_rows, int64_t n_edges,
               int heads, int dim, float slope, float *ws, hipStream_t stream,
               size_t ws_bytes = SIZE_MAX, int act = GA_ACT_NONE, size_t *size_only = nullptr,
               int z_stride = 0) {      // 0: rows of z side by side
  // the 16-byte lane layouts of the node forms (every benchmarked shape) get a build per
  // activation; everything else reads it from the arguments
  if constexpr (ACT == kActRuntime && !SPREAD && MODE != kGatEdge && VEC > 1) {
    if (act == GA_ACT_NONE)
      return launch_gat<T, VEC, MODE, SPREAD, GA_ACT_NONE>(pointer, row_of_slot, nbr, el, er, z, out,
                                                           n_rows, n_edges, heads, dim, slope, ws,
                                                           stream, ws_bytes, act, size_only, z_stride);
    if (act == GA_ACT_RELU)
      return launch_gat<T, VEC, MODE, SPREAD, GA_ACT_RELU>(pointer, row_of_slot, nbr, el, er, z, out,
                                                           n_rows, n_edges, heads, dim, slope, ws,
                                                           stream, ws_bytes, act, size_only, z_stride);
    return launch_gat<T, VEC, MODE, SPREAD, GA_ACT_ELU>(pointer, row_of_slot, nbr, el, er, z, out,
                                                        n_rows, n_edges, heads, dim, slope, ws, stream,
                                                        ws_bytes, act, size_only, z_stride);
  }
  if constexpr (GL == 0 && VEC > 1 && MODE != kGatFromZ) {
    // lane groups of eight lanes and more share the columns and the logits they form from
    // them, where the sharing lanes lie in one head (two fp32 heads of 32 are eight lanes
    // each: they keep their own reads)
    const bool one_head = heads == 1;
    const int lanes = (heads * dim + VEC - 1) / VEC;
#define GA_GAT_GL(N)                                                                            \
  return launch_gat<T, VEC, MODE, SPREAD, ACT, N>(pointer, row_of_slot, nbr, el, er, z, out,    \
                                                  n_rows, n_edges, heads, dim, slope, ws, stream, \
                                                  ws_bytes, act, size_only, z_stride)
    // per-edge rows stream: where they fill the lane group sharing gives nothing (108,368
    // uniform edges, fp32 rows of 128 and 512: 0.95 times the speed; 1 M edges: 1.03 .. 1.08).
    // The same holds where they are gathered through an id column (the pairs of a relation
    // attention by rank): own -> shared reads 1 x 64 fp32 11.5 -> 11.8 us on 100 k rows, 24.5 ->
    // 24.5 on 269 k, 37.8 -> 35.6 on 530 k, 114.7 -> 112.9 on 1.95 M, bf16 within 2 %
    const bool streams = MODE == kGatEdge && !SPREAD && (lanes & (lanes - 1)) == 0;
    if (lanes > 8 && !streams && (one_head || dim % (16 * VEC) == 0)) GA_GAT_GL(16);
    if (lanes > 4 && lanes <= 8 && !streams && one_head) GA_GAT_GL(8);
#undef GA_GAT_GL
  }
  typedef GatPolicy<T, VEC, MODE, SPREAD, ACT, GL> P;
  const bool ids_vec = aligned(row_of_slot, 16) && (!nbr || aligned(nbr, 16));
  const int head_lanes = dim / VEC;
  if (MODE == kGatFromZ &&
      (dim % VEC != 0 || head_lanes > 16 || (head_lanes & (head_lanes - 1)) != 0))
    return GA_EUNSUPPORTED;
  if constexpr (GL == 0 && VEC > 1 && MODE == kGatFromZ) {
#define GA_GAT_GL(N)                                                                            \
  return launch_gat<T, VEC, MODE, SPREAD, ACT, N>(pointer, row_of_slot, nbr, el, er, z, out,    \
                                                  n_rows, n_edges, heads, dim, slope, ws, stream, \
                                                  ws_bytes, act, size_only, z_stride)
    if (ga_gat_from_z_shares_logits(n_rows, heads, dim, z_stride, sizeof(T) == 4 ? GA_F32 : GA_BF16)) {
      if (head_lanes == 16) GA_GAT_GL(16);
      GA_GAT_GL(8);
    }
#undef GA_GAT_GL
  }
  typename P::Args args{nbr, el, er, (const T *)z, heads, dim, slope, ids_vec, head_lanes, 0, act,
                        z_stride ? z_stride : heads * dim};
  if constexpr (sizeof(T) == 2 && VEC == 8 && MODE == kGatNode && !SPREAD && GL == 0 &&
                ACT != kActRuntime) {
    const int lanes = heads * dim / VEC;
    if ((lanes > 16 && (lanes & (lanes - 1)) != 0) || n_edges < (1 << 20))
      return launch_runs<GatOpaqueStore<ACT>>(args, pointer, row_of_slot, out, n_rows, n_edges,
                                              heads * dim, ws, stream, ws_bytes, size_only);
  }
  return launch_runs<P>(args, pointer, row_of_slot, out, n_rows, n_edges,
                        heads * dim, ws, stream, ws_bytes, size_only);
}

// The element type and lane layout ga_gat_aggregate runs for a shape, launched
// with `ws` (capacity `ws_bytes`) as the partial-row scratch.
int gat_aggregate_dispatch(const int32_t *pointer, const int32_t *row_of_slot,
                           const int32_t *nbr, const float *el, const float *er,
                           const void *z, void *out, int64_t n_rows, int64_t n_edges,
                           int heads, int dim, float slope, int dtype, float *ws,
                           size_t ws_bytes, hipStream_t s, int act = GA_ACT_NONE,
                           size_t *size_only = nullptr, int z_stride = 0) {
  // (a stride is whole 16-byte pieces: checked where it comes in)
  const bool vec_ok = aligned(out, 16) && (!z || aligned(z, 16));
  if (dtype == GA_F32) {
    if (vec_ok && dim % 4 == 0)
      return launch_gat<float, 4>(pointer, row_of_slot, nbr, el, er, z, out, n_rows, n_edges,
                                  heads, dim, slope, ws, s, ws_bytes, act, size_only, z_stride);
    if (heads == 1 && dim >= 3 && dim <= 256)   // rows that 16-byte accesses do not tile
      return launch_gat<float, 4, kGatNode, true>(pointer, row_of_slot, nbr, el, er, z, out,
                                                  n_rows, n_edges, 1, dim, slope, ws, s, ws_bytes, act, size_only, z_stride);
    return launch_gat<float, 1>(pointer, row_of_slot, nbr, el, er, z, out, n_rows, n_edges,
                                heads, dim, slope, ws, s, ws_bytes, act, size_only, z_stride);
  }
  if (vec_ok && dim % 8 == 0)
    return launch_gat<bf16_t, 8>(pointer, row_of_slot, nbr, el, er, z, out, n_rows, n_edges,
                                 heads, dim, slope, ws, s, ws_bytes, act, size_only, z_stride);
  if (heads == 1 && dim >= 3 && dim <= 256)
    return launch_gat<bf16_t, 4, kGatNode, true>(pointer, row_of_slot, nbr, el, er, z, out,
                                                 n_rows, n_edges, 1, dim, slope, ws, s, ws_bytes, act, size_only, z_stride);
  return launch_gat<bf16_t, 1>(pointer, row_of_slot, nbr, el, er, z, out, n_rows, n_edges,
                               heads, dim, slope, ws, s, ws_bytes, act, size_only, z_stride);
}

// Argument checks shared by ga_gat_aggregate and ga_gat_aggregate_static
// (everything but the workspace).  GA_OK with *nothing_to_do set for n_rows == 0.
int gat_aggregate_check(const int32_t *pointer, const int32_t *row_of_slot,
                        const int32_t *nbr, const float *el, const float *er,
                        const void *z, const void *out, int64_t n_rows, int64_t n_edges,
                        int64_t heads, int64_t dim, int dtype, bool *nothing_to_do) {
  *nothing_to_do = false;
  if (n_rows < 0 || n_edges < 0 || heads <= 0 || dim <= 0) return GA_EINVAL;
  if (n_rows > 0x7fffffff || n_edges > 0x7fffffff || heads * dim > 0x7fffffff)
    return GA_EINVAL;
  if (dtype != GA_F32 && dtype != GA_BF16) return GA_EINVAL;
  if (n_rows == 0) {
    *nothing_to_do = true;
    return GA_OK;
  }
  if (!pointer || !out) return GA_EINVAL;
  if (n_edges > 0 && (!row_of_slot || !nbr || !el || !er || !z)) return GA_EINVAL;
  const size_t esz = dtype == GA_F32 ? 4 : 2;
  if (!aligned(out, esz) || (z && !aligned(z, esz)) || (el && !aligned(el, 4)) ||
      (er && !aligned(er, 4)))
    return GA_EALIGN;
  return GA_OK;
}

// Scratch of ga_gat_aggregate_static: the partial rows that ga_gat_aggregate
// takes as its workspace, held by the library itself.  Every device the library
// runs on has its own copy of this array at its own address; host code never
// uses the array's name as an address, only the pointer that
// hipGetSymbolAddress returned for the current device (static_scratch_for).
static __device__ __align__(256) unsigned char scratch[GA_STATIC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
std::mutex scratch_mutex;
void *scratch_ptr[kMaxDevices];   // per device, filled on the first call there

int static_scratch_for_current_device(void **ptr) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= kMaxDevices) return GA_EUNSUPPORTED;
  std::lock_guard<std::mutex> lock(scratch_mutex);
  if (!scratch_ptr[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (!p) return GA_EINVAL;
    scratch_ptr[dev] = p;
  }
  *ptr = scratch_ptr[dev];
  return GA_OK;
}

}  // namespace
}  // namespace ga

extern "C" {

size_t ga_gat_workspace_bytes(int64_t n_edges, int64_t feat, int64_t heads) {
  if (heads <= 0) return 0;
  // up to three state floats per feature (scalar path: sum, max, denominator)
  return ga::runs_workspace_bytes(n_edges, feat, 3);
}

int ga_gat_aggregate(const int32_t *pointer, const int32_t *row_of_slot,
                     const int32_t *nbr, const float *el, const float *er,
                     const void *z, void *out, int64_t n_rows, int64_t n_edges,
                     int64_t heads, int64_t dim, float slope, int dtype,
                     void *workspace, size_t workspace_bytes,
                     ga_stream_t stream) {
  return ga_gat_aggregate_act(pointer, row_of_slot, nbr, el, er, z, out, n_rows, n_edges, heads,
                              dim, slope, GA_ACT_NONE, dtype, workspace, workspace_bytes, stream);
}

int ga_gat_aggregate_act(const int32_t *pointer, const int32_t *row_of_slot,
                         const int32_t *nbr, const float *el, const float *er,
                         const void *z, void *out, int64_t n_rows, int64_t n_edges,
                         int64_t heads, int64_t dim, float slope, int activation, int dtype,
                         void *workspace, size_t workspace_bytes, ga_stream_t stream) {
  if (activation < GA_ACT_NONE || activation > GA_ACT_ELU) return GA_EINVAL;
  bool nothing = false;
  const int rc = ga::gat_aggregate_check(pointer, row_of_slot, nbr, el, er, z, out, n_rows,
                                         n_edges, heads, dim, dtype, &nothing);
  if (rc != GA_OK || nothing) return rc;
  if (n_edges > 0 &&
      (!workspace || !ga::aligned(workspace, 16) ||
       ga_gat_workspace_bytes(n_edges, heads * dim, heads) > workspace_bytes))
    return GA_EWORKSPACE;
  return ga::gat_aggregate_dispatch(pointer, row_of_slot, nbr, el, er, z, out, n_rows, n_edges,
                                    (int)heads, (int)dim, slope, dtype, (float *)workspace,
                                    workspace_bytes, (hipStream_t)stream, activation);
}

int ga_gat_aggregate_static(const int32_t *pointer, const int32_t *row_of_slot,
                            const int32_t *nbr, const float *el, const float *er,
                            const void *z, void *out, int64_t n_rows, int64_t n_edges,
                            int64_t heads, int64_t dim, float slope, int dtype,
                            ga_stream_t stream) {
  bool nothing = false;
  const int rc = ga::gat_aggregate_check(pointer, row_of_slot, nbr, el, er, z, out, n_rows,
                                         n_edges, heads, dim, dtype, &nothing);
  if (rc != GA_OK || nothing) return rc;
  void *ws = nullptr;
  const int sc = ga::static_scratch_for_current_device(&ws);
  if (sc != GA_OK) return sc;
  // The kernels write every partial row before the fix-up pass reads it, so the
  // previous call's contents need no clearing.
  const int lr = ga::gat_aggregate_dispatch(pointer, row_of_slot, nbr, el, er, z, out, n_rows,
                                            n_edges, (int)heads, (int)dim, slope, dtype,
                                            (float *)ws, (size_t)GA_STATIC_SCRATCH_BYTES,
                                            (hipStream_t)stream);
  return lr == GA_EWORKSPACE ? GA_ESCRATCH : lr;
}

int64_t ga_gat_static_scratch_needed(int64_t n_edges, int64_t heads, int64_t dim, int dtype,
                                     int rows_16_byte_aligned) {
  if (n_edges < 0 || heads <= 0 || dim <= 0 || n_edges > 0x7fffffff ||
      heads * dim > 0x7fffffff || (dtype != GA_F32 && dtype != GA_BF16))
    return GA_EINVAL;
  if (n_edges == 0) return 0;
  // the dispatch itself, asked for the size of the layout it would launch: the two
  // addresses below only carry the alignment and are never dereferenced
  const void *row = (const void *)(uintptr_t)(rows_16_byte_aligned ? 16 : (dtype == GA_F32 ? 4 : 2));
  size_t needed = 0;
  const int rc = ga::gat_aggregate_dispatch(nullptr, nullptr, nullptr, nullptr, nullptr, row,
                                            (void *)row, 1, n_edges, (int)heads, (int)dim, 0.0f,
                                            dtype, nullptr, 0, nullptr, GA_ACT_NONE, &needed);
  return rc == GA_OK ? (int64_t)needed : (int64_t)rc;
}

int ga_edge_softmax_sum(const int32_t *pointer, const int32_t *row_of_slot,
                        const int32_t *eid, const float *logit, const void *m,
                        void *out, int64_t n_rows, int64_t n_edges, int64_t heads,
                        int64_t dim, int dtype, void *workspace,
                        size_t workspace_bytes, ga_stream_t stream) {
  if (n_rows < 0 || n_edges < 0 || heads <= 0 || dim <= 0) return GA_EINVAL;
  if (n_rows > 0x7fffffff || n_edges > 0x7fffffff || heads * dim > 0x7fffffff)
    return GA_EINVAL;
  if (dtype != GA_F32 && dtype != GA_BF16) return GA_EINVAL;
  if (n_rows == 0) return GA_OK;
  if (!pointer || !out) return GA_EINVAL;
  const int64_t feat = heads * dim;
  if (n_edges > 0) {
    if (!row_of_slot || !logit || !m) return GA_EINVAL;
    if (!workspace || !ga::aligned(workspace, 16) ||
        ga_gat_workspace_bytes(n_edges, feat, heads) > workspace_bytes)
      return GA_EWORKSPACE;
  }
  const size_t esz = dtype == GA_F32 ? 4 : 2;
  if (!ga::aligned(out, esz) || (m && !ga::aligned(m, esz)) ||
      (logit && !ga::aligned(logit, 4)))
    return GA_EALIGN;
  const bool vec_ok = ga::aligned(out, 16) && (!m || ga::aligned(m, 16));
  hipStream_t s = (hipStream_t)stream;
  float *ws = (float *)workspace;
  const int h = (int)heads, d = (int)dim;
  if (dtype == GA_F32) {
    if (vec_ok && dim % 4 == 0)
      return ga::launch_gat<float, 4, ga::kGatEdge>(pointer, row_of_slot, eid, logit, nullptr, m,
                                            out, n_rows, n_edges, h, d, 0.0f, ws, s);
    if (heads == 1 && dim >= 3 && dim <= 256)   // rows that 16-byte accesses do not tile
      return ga::launch_gat<float, 4, ga::kGatEdge, true>(pointer, row_of_slot, eid, logit, nullptr,
                                                          m, out, n_rows, n_edges, 1, d, 0.0f, ws, s);
    return ga::launch_gat<float, 1, ga::kGatEdge>(pointer, row_of_slot, eid, logit, nullptr, m, out,
                                          n_rows, n_edges, h, d, 0.0f, ws, s);
  }
  if (vec_ok && dim % 8 == 0)
    return ga::launch_gat<ga::bf16_t, 8, ga::kGatEdge>(pointer, row_of_slot, eid, logit, nullptr, m,
                                               out, n_rows, n_edges, h, d, 0.0f, ws, s);
  if (heads == 1 && dim >= 3 && dim <= 256)
    return ga::launch_gat<ga::bf16_t, 4, ga::kGatEdge, true>(pointer, row_of_slot, eid, logit, nullptr,
                                                             m, out, n_rows, n_edges, 1, d, 0.0f, ws, s);
  return ga::launch_gat<ga::bf16_t, 1, ga::kGatEdge>(pointer, row_of_slot, eid, logit, nullptr, m,
                                             out, n_rows, n_edges, h, d, 0.0f, ws, s);
}

int ga_dot_attention_sum(const int32_t *pointer, const int32_t *row_of_slot,
                         const int32_t *nbr, const int32_t *qrow, const void *k, const void *q,
                         const void *v, void *out, float *lse, const int32_t *lse_index,
                         int64_t n_rows, int64_t n_edges, int64_t heads, int64_t dim, int dtype,
                         void *workspace, size_t workspace_bytes, ga_stream_t stream) {
  if (n_rows < 0 || n_edges < 0 || heads <= 0 || dim <= 0) return GA_EINVAL;
  if (n_rows > 0x7fffffff || n_edges > 0x7fffffff || heads * dim > 0x7fffffff)
    return GA_EINVAL;
  if (dtype != GA_F32 && dtype != GA_BF16) return GA_EINVAL;
  if (n_rows == 0) return GA_OK;
  if (!pointer || !out) return GA_EINVAL;
  const int64_t feat = heads * dim;
  if (n_edges > 0) {
    if (!row_of_slot || !nbr || !qrow || !k || !q || !v) return GA_EINVAL;
    if (!workspace || !ga::aligned(workspace, 16) ||
        ga_gat_workspace_bytes(n_edges, feat, heads) > workspace_bytes)
      return GA_EWORKSPACE;
  }
  if ((lse && !ga::aligned(lse, 4)) || (lse_index && !ga::aligned(lse_index, 4))) return GA_EALIGN;
  if (lse_index && !lse) return GA_EINVAL;
  // rows are read and written in 16-byte pieces that do not straddle a head
  const int vec = dtype == GA_F32 ? 4 : 8;
  if (!ga::aligned(out, 16) || (k && !ga::aligned(k, 16)) || (q && !ga::aligned(q, 16)) ||
      (v && !ga::aligned(v, 16)) || dim % vec != 0)
    return GA_EUNSUPPORTED;
  hipStream_t s = (hipStream_t)stream;
  if (dtype == GA_F32)
    return ga::launch_dot_attn<float, 4>(pointer, row_of_slot, nbr, qrow, k, q, v, out, lse,
                                         lse_index, n_rows, n_edges, (int)heads, (int)dim,
                                         (float *)workspace, workspace_bytes, s);
  return ga::launch_dot_attn<ga::bf16_t, 8>(pointer, row_of_slot, nbr, qrow, k, q, v, out, lse,
                                            lse_index, n_rows, n_edges, (int)heads, (int)dim,
                                            (float *)workspace, workspace_bytes, s);
}

int ga_gat_aggregate_from_z(const int32_t *pointer, const int32_t *row_of_slot,
                            const int32_t *nbr, const float *a_l, const float *er,
                            const void *z, void *out, int64_t n_rows, int64_t n_edges,
                            int64_t heads, int64_t dim, float slope, int dtype,
                            void *workspace, size_t workspace_bytes, ga_stream_t stream) {
  return ga_gat_aggregate_from_z_act(pointer, row_of_slot, nbr, a_l, er, z, out, n_rows, n_edges,
                                     heads, dim, slope, GA_ACT_NONE, dtype, workspace,
                                     workspace_bytes, stream);
}

static int gat_from_z(const int32_t *pointer, const int32_t *row_of_slot, const int32_t *nbr,
                      const float *a_l, const float *er, const void *z, int z_stride, void *out,
                      int64_t n_rows, int64_t n_edges, int64_t heads, int64_t dim, float slope,
                      int activation, int dtype, void *workspace, size_t workspace_bytes,
                      ga_stream_t stream) {
  if (activation < GA_ACT_NONE || activation > GA_ACT_ELU) return GA_EINVAL;
  if (n_rows < 0 || n_edges < 0 || heads <= 0 || dim <= 0) return GA_EINVAL;
  if (n_rows > 0x7fffffff || n_edges > 0x7fffffff || heads * dim > 0x7fffffff)
    return GA_EINVAL;
  if (dtype != GA_F32 && dtype != GA_BF16) return GA_EINVAL;
  if (n_rows == 0) return GA_OK;
  if (!pointer || !out) return GA_EINVAL;
  const int64_t feat = heads * dim;
  if (n_edges > 0) {
    if (!row_of_slot || !nbr || !a_l || !er || !z) return GA_EINVAL;
    if (!workspace || !ga::aligned(workspace, 16) ||
        ga_gat_workspace_bytes(n_edges, feat, heads) > workspace_bytes)
      return GA_EWORKSPACE;
  }
  const size_t esz = dtype == GA_F32 ? 4 : 2;
  if (!ga::aligned(out, esz) || (z && !ga::aligned(z, esz)) ||
      (a_l && !ga::aligned(a_l, 4)) || (er && !ga::aligned(er, 4)))
    return GA_EALIGN;
  const bool vec_ok = ga::aligned(out, 16) && (!z || ga::aligned(z, 16));
  hipStream_t s = (hipStream_t)stream;
  float *ws = (float *)workspace;
  const int h = (int)heads, d = (int)dim;
  if (dtype == GA_F32) {
    if (vec_ok && dim % 4 == 0)
      return ga::launch_gat<float, 4, ga::kGatFromZ>(pointer, row_of_slot, nbr, a_l, er, z, out,
                                                     n_rows, n_edges, h, d, slope, ws, s, SIZE_MAX, activation,
                                                     nullptr, z_stride);
    return ga::launch_gat<float, 1, ga::kGatFromZ>(pointer, row_of_slot, nbr, a_l, er, z, out,
                                                   n_rows, n_edges, h, d, slope, ws, s, SIZE_MAX, activation,
                                                     nullptr, z_stride);
  }
  if (vec_ok && dim % 8 == 0)
    return ga::launch_gat<ga::bf16_t, 8, ga::kGatFromZ>(pointer, row_of_slot, nbr, a_l, er, z,
                                                        out, n_rows, n_edges, h, d, slope, ws, s, SIZE_MAX, activation,
                                                     nullptr, z_stride);
  return ga::launch_gat<ga::bf16_t, 1, ga::kGatFromZ>(pointer, row_of_slot, nbr, a_l, er, z, out,
                                                      n_rows, n_edges, h, d, slope, ws, s, SIZE_MAX, activation,
                                                     nullptr, z_stride);
}

int ga_gat_aggregate_from_z_act(const int32_t *pointer, const int32_t *row_of_slot,
                                const int32_t *nbr, const float *a_l, const float *er,
                                const void *z, void *out, int64_t n_rows, int64_t n_edges,
                                int64_t heads, int64_t dim, float slope, int activation,
                                int dtype, void *workspace, size_t workspace_bytes,
                                ga_stream_t stream) {
  return gat_from_z(pointer, row_of_slot, nbr, a_l, er, z, 0, out, n_rows, n_edges, heads, dim,
                    slope, activation, dtype, workspace, workspace_bytes, stream);
}

// Whether the lanes of a head (8 or 16 of them) form a slot's logit and exponential once, or
// every lane for itself.  Once is a third fewer instructions and one more wavefront per
// SIMD: faster where instructions bound the walk, slower where rows side by side meet in few
// memory channels, which more wavefronts in flight make worse.  us, every lane -> once, R-MAT
// and uniform graphs of 12 to 50 edges per node:
//   rows apart, 64 M R-MAT edges     4 x 64 bf16 4864 -> 4466, 2 x 64 2968 -> 2718
//   bf16 side by side, 128 to 384 and 640 bytes   0.67 .. 0.93 of the time at all sizes
//     512 bytes    120 MB 830 -> 784, 360 MB 969 -> 911, 614 MB 2348 -> 2361, 1.25 GB 5705 -> 6186
//     1024 bytes   100 MB 380 -> 321 (uniform 431 -> 440), 240 MB 1495 -> 1497 (1647 -> 1674),
//                  720 MB 1762 -> 1843, 2.5 GB 12237 -> 12568
//   fp32 side by side, 128 to 512 bytes   up to 60 MB 0.79 .. 1.03, from 120 MB on 0.98 .. 1.05
//     384 and 768 bytes   up to 540 MB 0.75 .. 1.03, above 0.95 .. 1.05
int ga_gat_from_z_shares_logits(int64_t n_rows, int64_t heads, int64_t dim, int64_t z_stride,
                                int dtype) {
  if (n_rows < 0 || heads <= 0 || dim <= 0 || (dtype != GA_F32 && dtype != GA_BF16)) return 0;
  const int64_t esz = dtype == GA_F32 ? 4 : 2, piece = 16 / esz;
  if (dim != 8 * piece && dim != 16 * piece) return 0;
  if (z_stride > heads * dim) return 1;
  const int64_t row = heads * dim * esz;
  const bool power = (row & (row - 1)) == 0;
  if (dtype == GA_F32) return n_rows <= ((power ? 64ll : 640ll) << 20) / row;
  return row % 512 != 0 || n_rows <= ((row % 1024 != 0 ? 768ll : 192ll) << 20) / row;
}

// Rows of whole multiples of 256 bytes are kept 128 bytes further apart where their table is
// larger than an L2.  Graph generators and loaders give popular nodes ids with structure
// (many zero bits in R-MAT), and with rows a power of two apart those ids' rows meet in a
// few of the memory channels, which change every 128 bytes; how many also depends on where
// the table lies (1 x 64 fp32 on 11.6 M edges, the same table in four places: 264 to 320 us,
// apart 245 to 272).  Side by side -> 128 bytes further apart (64 or 256 bytes: slower), us, the
// projection and the aggregation over three buffers in turn, R-MAT:
//   2.4 M nodes, 64 M edges      1 x 64 fp32 3575 -> 3075, 2 x 64 bf16 3298 -> 2627, 4 x 64 6207 -> 4604
//   700 k nodes, 8 M edges       1 x 64 fp32 472 -> 420, 2 x 64 bf16 471 -> 447, 4 x 64 948 -> 810
//   233 k nodes, 11.6 M edges    1 x 64 fp32 459 -> 440 (level, 431, in other runs), 2 x 64 bf16
//                                446 -> 444, 4 x 64 fp32 1882 -> 1358
//   100 k nodes, 3 M edges       1 x 64 fp32 106 -> 106, 2 x 64 202 -> 175, 4 x 64 398 -> 354
// Uniform ids, tables below 32 MB and rows of 768 bytes: level (within 1.4 %).  The price is
// memory: half as much z again at 256 bytes a row, a quarter at 512, an eighth at 1024.
int64_t ga_gather_row_stride(int64_t n_rows, int64_t feat, int dtype) {
  if (n_rows < 0 || feat <= 0 || (dtype != GA_F32 && dtype != GA_BF16)) return 0;
  const int64_t esz = dtype == GA_F32 ? 4 : 2;
  return feat * esz % 256 == 0 && n_rows > (4 << 20) / (feat * esz) ? feat + 128 / esz : feat;
}

int ga_gat_aggregate_strided(const int32_t *pointer, const int32_t *row_of_slot,
                             const int32_t *nbr, const float *source, const float *er,
                             const void *z, int64_t z_stride, void *out, int64_t n_rows,
                             int64_t n_edges, int64_t heads, int64_t dim, float slope, int from_z,
                             int activation, int dtype, void *workspace, size_t workspace_bytes,
                             ga_stream_t stream) {
  if (activation < GA_ACT_NONE || activation > GA_ACT_ELU) return GA_EINVAL;
  bool nothing = false;
  const int rc = ga::gat_aggregate_check(pointer, row_of_slot, nbr, source, er, z, out, n_rows,
                                         n_edges, heads, dim, dtype, &nothing);
  if (rc != GA_OK || nothing) return rc;
  const int64_t piece = dtype == GA_F32 ? 4 : 8;
  if (z_stride < heads * dim || z_stride > 0x7fffffff) return GA_EINVAL;
  if (dim % piece || z_stride % piece || !ga::aligned(z, 16) || !ga::aligned(out, 16))
    return GA_EUNSUPPORTED;
  if (from_z)
    return gat_from_z(pointer, row_of_slot, nbr, source, er, z, (int)z_stride, out, n_rows, n_edges,
                      heads, dim, slope, activation, dtype, workspace, workspace_bytes, stream);
  if (n_edges > 0 &&
      (!workspace || !ga::aligned(workspace, 16) ||
       ga_gat_workspace_bytes(n_edges, heads * dim, heads) > workspace_bytes))
    return GA_EWORKSPACE;
  return ga::gat_aggregate_dispatch(pointer, row_of_slot, nbr, source, er, z, out, n_rows, n_edges,
                                    (int)heads, (int)dim, slope, dtype, (float *)workspace,
                                    workspace_bytes, (hipStream_t)stream, activation, nullptr,
                                    (int)z_stride);
}

}  // extern "C"
