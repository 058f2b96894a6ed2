// Typed linear of fp32 node (or edge) rows sorted by type, for up to four weight tensors of one
// shape over the same rows (HGT's K, Q and V, examples/HGT/HGT.py:35-44) in one launch:
//   Y_g[r, :] = X[r, :] @ W_g[type(r)],  times a factor per row or a gate per type.
//
// A product of 94,000 rows of 64 moves 48 MB, ten microseconds' worth: what it takes is the chain
// of a workgroup -- find the chunk, fetch W, fetch rows, multiply, store -- and the launches.
// So the tensors are the second grid dimension of one launch, W goes to LDS once per chunk in
// the order in which the matrix instruction reads it (one 16-byte read per lane and piece), the
// rows go straight from memory to their operand, and a lane stores C neighbouring columns of a
// row at once.  fp32 on the bf16 instruction as in the dense projection: three pieces a value
// (cut off, rounded, rest), six of nine products; values that are not finite are multiplied
// again without the split.
// us before (a launch a tensor, fp32 instruction, rows of two tiles a workgroup) -> here, one tensor
// and three: 93,773 x 64 -> 64 19 -> 14, 57 -> 30; 128 -> 128 70 -> 39, 210 -> 86; 5,000 x 64 -> 64
// 7.3 -> 6.5, 21 -> 7; 1 M x 64 -> 64, 200 types 141 -> 122, 403 -> 314; 5.6 M x 16 -> 64 378 -> 365.
// Error against float64 1.4e-7 -> 0.96e-7 at K = 64 (positive products 1.2e-7 -> 0.74e-7).
#include "typed_chunks.h"
#include "typed_rows.h"

namespace ga {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kWaves = kBlock / kWave;

// x = p0 + p1 + p2; eight values -> three packed operands
__device__ __forceinline__ void split8(const float (&v)[8], uint4 &p0, uint4 &p1, uint4 &p2) {
  uint32_t a[8], b[4], c[8];
#pragma unroll
  for (int j = 0; j < 8; j += 2) {
    a[j] = __float_as_uint(v[j]);
    a[j + 1] = __float_as_uint(v[j + 1]);
    const float r0 = v[j] - __uint_as_float(a[j] & 0xffff0000u);
    const float r1 = v[j + 1] - __uint_as_float(a[j + 1] & 0xffff0000u);
    b[j / 2] = pack_bf16(r0, r1);
    c[j] = __float_as_uint(r0 - bf16_lo(b[j / 2]));
    c[j + 1] = __float_as_uint(r1 - bf16_hi(b[j / 2]));
  }
  constexpr uint32_t hi = 0x07060302u;
  p0 = uint4{__builtin_amdgcn_perm(a[1], a[0], hi), __builtin_amdgcn_perm(a[3], a[2], hi),
             __builtin_amdgcn_perm(a[5], a[4], hi), __builtin_amdgcn_perm(a[7], a[6], hi)};
  p1 = uint4{b[0], b[1], b[2], b[3]};
  p2 = uint4{__builtin_amdgcn_perm(c[1], c[0], hi), __builtin_amdgcn_perm(c[3], c[2], hi),
             __builtin_amdgcn_perm(c[5], c[4], hi), __builtin_amdgcn_perm(c[7], c[6], hi)};
}

// KS steps of 32 k, C blocks of 16 columns a pass: block c holds the columns 16 C pass + n C + c
template <int KS, int C>
__global__ __launch_bounds__(kBlock, KS == 4 ? 2 : 3) void typed_rows_kernel(TypedRows p, int chunk_rows, int passes) {
  __shared__ __attribute__((aligned(16))) uint4 wp[KS][C][3][kWave];
  __shared__ int odd;                 // W has values that are not finite
  int type, row0, row1;
  if (threadIdx.x == 0) odd = 0;
  if (!locate_chunk(p.tp, p.n_types, chunk_rows, blockIdx.x, type, row0, row1)) return;
  const int which = blockIdx.y / passes, col0 = blockIdx.y % passes * 16 * C;
  const int K = p.K, M = p.M;
  const float *W = p.W[which] + (int64_t)type * K * M + col0;
  const int lane = threadIdx.x & (kWave - 1), n = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);

  // A lane's eight k of a step are 4 q .. 4 q + 3 and 16 more: the four lanes of a row read 64
  // bytes side by side with either load (of X; W is put down in the same order).
  struct Tile { float4 x[KS][2]; };
  auto fetch = [&](int r, Tile &t) __attribute__((always_inline)) {
    const float *x = p.X + (int64_t)min(r + n, row1 - 1) * K + 4 * q;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        t.x[ks][h] = ks * 32 + 16 * h + 4 * q < K ? *reinterpret_cast<const float4 *>(x + ks * 32 + 16 * h)
                                                 : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  };
  Tile t;
  const int first = row0 + 16 * wave;
  if (first < row1) fetch(first, t);  // on its way while W is prepared
  __syncthreads();
  for (int i = threadIdx.x; i < KS * C * kWave; i += kBlock) {
    const int l = i & (kWave - 1), c = i / kWave % C, ks = i / kWave / C;
    const int k0 = ks * 32 + (l >> 4) * 4;
    const float *w = W + (l & 15) * C + c;
    float v[8], z = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int k = k0 + (j & 3) + 4 * (j & 4);
      v[j] = k < K ? w[(int64_t)k * M] : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) z = fmaf(v[j], 0.0f, z);
    if (z != 0.0f) odd = 1;           // NaN: every writer stores the same value
    split8(v, wp[ks][c][0][l], wp[ks][c][1][l], wp[ks][c][2][l]);
  }
  __syncthreads();
  float gate = 1.0f;
  if (p.gate) {
    const float g = p.gate[type];
    gate = p.gate_sigmoid ? 1.0f / (1.0f + expf(-g)) : g;
  }
  const bool w_odd = odd != 0;
  for (int r = first; r < row1; r += 16 * kWaves) {
    const Tile now = t;
    asm volatile("" ::: "memory");    // W is read from LDS every time: held, it takes 96 registers
    if (r + 16 * kWaves < row1) fetch(r + 16 * kWaves, t);
    floatx4 acc[C];
#pragma unroll
    for (int c = 0; c < C; ++c) acc[c] = floatx4{0, 0, 0, 0};
    float z = 0.0f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const float4 lo = now.x[ks][0], up = now.x[ks][1];
      const float v[8] = {lo.x, lo.y, lo.z, lo.w, up.x, up.y, up.z, up.w};
#pragma unroll
      for (int j = 0; j < 8; ++j) z = fmaf(v[j], 0.0f, z);
      uint4 xp[3];
      split8(v, xp[0], xp[1], xp[2]);
      constexpr int px[6] = {2, 0, 1, 1, 0, 0}, pw[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const uint4 wf[3] = {wp[ks][c][0][lane], wp[ks][c][1][lane], wp[ks][c][2][lane]};
#pragma unroll
        for (int m = 0; m < 6; ++m)
          acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, xp[px[m]]),
                                                           __builtin_bit_cast(bf16x8, wf[pw[m]]), acc[c], 0, 0, 0);
      }
    }
    if (w_odd || __builtin_amdgcn_ballot_w64(z != 0.0f) != 0) {
#pragma unroll
      for (int c = 0; c < C; ++c) acc[c] = floatx4{0, 0, 0, 0};
      for (int k = 0; k < K; ++k)
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            acc[c][i] = fmaf(p.X[(int64_t)min(r + 4 * q + i, row1 - 1) * K + k],
                             W[(int64_t)k * M + n * C + c], acc[c][i]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = r + 4 * q + i;
      if (row >= row1) continue;
      const float f = p.row_scale ? p.row_scale[row] : gate;
      float *y = p.Y[which] + (int64_t)row * M + col0 + n * C;
      if constexpr (C == 4)
        *reinterpret_cast<float4 *>(y) = make_float4(acc[0][i] * f, acc[1][i] * f, acc[2][i] * f, acc[3][i] * f);
      else if constexpr (C == 2)
        *reinterpret_cast<float2 *>(y) = make_float2(acc[0][i] * f, acc[1][i] * f);
      else
        *y = acc[0][i] * f;
    }
  }
}

template <int KS>
int launch(const TypedRows &p, hipStream_t s) {
  const int C = p.M >= 64 ? 4 : p.M / 16, passes = p.M / (16 * C);
  // chunks of whole rounds of the four wavefronts, about five workgroups to a CU
  const int64_t want = (p.rows * p.n_weights * passes + 1279) / 1280;
  const int chunk = (int)(want < 64 ? 64 : want > 1024 ? 1024 : (want + 63) / 64 * 64);
  const int64_t chunks = p.rows / chunk + p.n_types;      // every type has a ragged last one
  if (chunks > 0x7fffffff) return GA_EUNSUPPORTED;
  const dim3 grid((unsigned)chunks, (unsigned)(p.n_weights * passes));
  if (C == 4) hipLaunchKernelGGL((typed_rows_kernel<KS, 4>), grid, dim3(kBlock), 0, s, p, chunk, passes);
  else if (C == 2) hipLaunchKernelGGL((typed_rows_kernel<KS, 2>), grid, dim3(kBlock), 0, s, p, chunk, passes);
  else hipLaunchKernelGGL((typed_rows_kernel<KS, 1>), grid, dim3(kBlock), 0, s, p, chunk, passes);
  return launch_status();
}

}  // namespace

int typed_rows_launch(const TypedRows &p, hipStream_t s) {
  if (p.K % 4 || p.K > 128 || (p.M != 16 && p.M != 32 && p.M % 64)) return GA_EUNSUPPORTED;
  if (p.rows > 0x7fffffff || p.n_weights * (p.M / 16) > 65535) return GA_EUNSUPPORTED;
  if (!aligned(p.X, 16)) return GA_EUNSUPPORTED;
  for (int i = 0; i < p.n_weights; ++i)
    if (!aligned(p.Y[i], 16) || !aligned(p.W[i], 4)) return GA_EUNSUPPORTED;
  if (p.K <= 32) return launch<1>(p, s);
  if (p.K <= 64) return launch<2>(p, s);
  return launch<4>(p, s);
}

}  // namespace ga
