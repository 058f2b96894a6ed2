// The pair attention over prepared tiles, rows and matrices, and their preparation.
#include "pair_attn.h"

namespace ga {
namespace {

// the tiles and rows of PairArgs, one wavefront per tile
__global__ __launch_bounds__(kWave) void pair_tiles_kernel(PairArgs A, int4 *__restrict__ rows,
                                                           int4 *__restrict__ tiles) {
  int type = -1, row0 = 0, row1 = 0;
  const bool mine = locate_chunk(A.type_pointer, A.n_types, kPairRows, blockIdx.x, type, row0, row1);
  if (threadIdx.x == 0) tiles[blockIdx.x] = make_int4(mine ? type : -1, row0, row1, 0);
  const int r = row0 + (int)threadIdx.x;
  if (!mine || r >= row1) return;
  const int p = (int)A.by_type[r];
  rows[r] = make_int4(A.pair_pointer[p], A.pair_pointer[p + 1], (int)A.dst_by_type[r], 0);
}

// The matrices of the split shapes: att transposed and times its scale (an fp32 product
// rounded once), msg as it is, both split, in the order in which the lanes of
// SplitBlock::load read them.  blockIdx.y: att | msg; a thread per lane of a block of 32 k.
template <int D, typename S>
__global__ __launch_bounds__(kBlock) void pair_weights_kernel(
    const float *__restrict__ att, const S *__restrict__ scale, float factor,
    const float *__restrict__ msg, uint4 *__restrict__ att_out, uint4 *__restrict__ msg_out,
    int64_t n_units) {
  constexpr int H = 64 / D, KB = D / 32;
  const int64_t u = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (u >= n_units) return;
  const int lane = (int)(u % kWave), b = (int)(u / kWave % KB), cb = (int)(u / kWave / KB % 4);
  const int64_t t = u / kWave / KB / 4;
  const int col = cb * 16 + lane % 16, k = 32 * b + lane / 16 * 8;
  const int64_t block = t * H + col / D;
  float x[8];
#pragma unroll
  for (int j = 0; j < 8; ++j)
    x[j] = blockIdx.y ? msg[(block * D + k + j) * D + col % D]
                      : att[(block * D + col % D) * D + k + j] *
                            (scale ? elem_to_f32(scale[block]) : 1.0f) * factor;
  uint32_t p[3][4];
  split(x, p);
  uint4 *const out = (blockIdx.y ? msg_out : att_out) + t * (64 * D * 3 / 8);
#pragma unroll
  for (int q = 0; q < 3; ++q)
    out[SplitBlock<D>::unit(cb, b, q, lane)] = make_uint4(p[q][0], p[q][1], p[q][2], p[q][3]);
}

}  // namespace
}  // namespace ga

extern "C" int64_t ga_pair_tiles_capacity(int64_t n_pairs, int64_t n_types) {
  return n_pairs < 0 || n_types < 0 ? 0 : (n_pairs + ga::kPairRows - 1) / ga::kPairRows + n_types;
}

extern "C" int ga_pair_tiles_build(const int32_t *type_pointer, int64_t n_types,
                                   const int64_t *by_type, const int64_t *dst_by_type,
                                   const int32_t *pair_pointer, int64_t n_pairs, int32_t *rows,
                                   int32_t *tiles, ga_stream_t stream) {
  if (n_types <= 0 || n_pairs < 0 || n_types > 0x7fffffff || n_pairs > 0x7fffffff) return GA_EINVAL;
  if (n_pairs == 0) return GA_OK;
  if (!type_pointer || !by_type || !dst_by_type || !pair_pointer || !rows || !tiles) return GA_EINVAL;
  if (!ga::aligned(rows, 16) || !ga::aligned(tiles, 16)) return GA_EALIGN;
  const int64_t grid = ga_pair_tiles_capacity(n_pairs, n_types);
  if (grid > 0x7fffffff) return GA_EUNSUPPORTED;
  ga::PairArgs A{};
  A.type_pointer = type_pointer;
  A.by_type = by_type;
  A.dst_by_type = dst_by_type;
  A.pair_pointer = pair_pointer;
  A.n_types = (int)n_types;
  hipLaunchKernelGGL(ga::pair_tiles_kernel, dim3((unsigned)grid), dim3(ga::kWave), 0,
                     (hipStream_t)stream, A, (int4 *)rows, (int4 *)tiles);
  return ga::launch_status();
}

extern "C" size_t ga_pair_weights_bytes(int64_t n_types, int64_t heads, int64_t dim, int dtype) {
  if (n_types <= 0 || n_types > 0x7fffffff || dtype != GA_F32 || heads <= 0 || heads * dim != 64 || dim < 32)
    return 0;
  return (size_t)n_types * 64 * (size_t)dim * 6;
}

extern "C" int ga_pair_weights(const float *att, const void *scale, int scale_dtype, float factor,
                               const float *msg, void *att_out, void *msg_out, int64_t n_types,
                               int64_t heads, int64_t dim, ga_stream_t stream) {
  using namespace ga;
  if (ga_pair_weights_bytes(n_types, heads, dim, GA_F32) == 0) return GA_EUNSUPPORTED;
  if (!att || !msg || !att_out || !msg_out) return GA_EINVAL;
  if (scale_dtype != GA_F32 && scale_dtype != GA_BF16) return GA_EINVAL;
  if (!aligned(att, 4) || !aligned(msg, 4) || !aligned(att_out, 16) || !aligned(msg_out, 16) ||
      (scale && !aligned(scale, scale_dtype == GA_F32 ? 4 : 2)))
    return GA_EALIGN;
  const int64_t n_units = n_types * 4 * (dim / 32) * kWave;
  const dim3 grid((unsigned)((n_units + kBlock - 1) / kBlock), 2);
  hipStream_t s = (hipStream_t)stream;
#define GA_PAIR_WEIGHTS(D, S)                                                                 \
  hipLaunchKernelGGL((pair_weights_kernel<D, S>), grid, dim3(kBlock), 0, s, att, (const S *)scale, \
                     factor, msg, (uint4 *)att_out, (uint4 *)msg_out, n_units)
  if (dim == 64) {
    if (scale_dtype == GA_F32) GA_PAIR_WEIGHTS(64, float);
    else GA_PAIR_WEIGHTS(64, bf16_t);
  } else {
    if (scale_dtype == GA_F32) GA_PAIR_WEIGHTS(32, float);
    else GA_PAIR_WEIGHTS(32, bf16_t);
  }
#undef GA_PAIR_WEIGHTS
  return launch_status();
}

// a slot's address is a 32-bit offset
extern "C" int ga_pair_tiles_fit(int64_t n_nodes, int64_t heads, int64_t dim, int dtype) {
  if (n_nodes < 0 || n_nodes > 0x7fffffff || heads <= 0 || dim <= 0 || heads > 0x7fffffff / dim ||
      (dtype != GA_F32 && dtype != GA_BF16))
    return 0;
  return n_nodes <= 0xffffffffll / (heads * dim * (dtype == GA_F32 ? 4 : 2));
}

extern "C" int ga_pair_attention_tiles(const int32_t *rows, const int32_t *tiles, int64_t n_types,
                                       const int32_t *nbr, const void *q, const void *k,
                                       const void *v, const void *att, const void *msg, void *m,
                                       float *lse, int64_t n_pairs, int64_t n_nodes,
                                       int64_t max_slots, int64_t heads, int64_t dim, int dtype,
                                       ga_stream_t stream) {
  if (!ga::pair_counts_ok(n_types, n_pairs, max_slots, heads, dim, dtype) || n_nodes < 0)
    return GA_EINVAL;
  if (n_pairs == 0) return GA_OK;
  if (!rows || !tiles) return GA_EINVAL;
  if (!ga::aligned(rows, 16) || !ga::aligned(tiles, 16)) return GA_EALIGN;
  ga::PairArgs A{(const int4 *)rows, (const int4 *)tiles, nullptr, nullptr, nullptr, nullptr, nbr,
                 q, k, v, att, msg, m, lse, (int)n_types};
  const int rc = ga::check_pairs(A, max_slots);
  if (rc != GA_OK) return rc;
  if (!ga_pair_tiles_fit(n_nodes, heads, dim, dtype)) return GA_EUNSUPPORTED;
  if (ga_pair_weights_bytes(n_types, heads, dim, dtype) > 0 &&
      (!ga::aligned(att, 16) || !ga::aligned(msg, 16)))
    return GA_EALIGN;
  if (dtype == GA_F32)
    return ga::launch_pairs_dim<float, true>(A, n_pairs, heads * dim, dim, (hipStream_t)stream);
  return ga::launch_pairs_dim<ga::bf16_t, true>(A, n_pairs, heads * dim, dim, (hipStream_t)stream);
}
