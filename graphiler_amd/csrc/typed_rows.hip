// Typed linear of fp32 node (or edge) rows sorted by type, for up to four weight tensors of one
// shape over the same rows (HGT's K, Q and V, examples/HGT/HGT.py:35-44) in one launch:
//   Y_g[r, :] = X[r, :] @ W_g[type(r)],  times a factor per row or a gate per type.
//
// A product of 94,000 rows of 64 moves 48 MB, ten microseconds' worth: what it takes is the chain
// of a workgroup -- find the chunk, fetch W, fetch rows, multiply, store -- and the launches.
// So the tensors are the second grid dimension of one launch, W goes to LDS once per chunk in
// the order in which the matrix instruction reads it (one 16-byte read per lane and piece), the
// rows go straight from memory to their operand, and a lane stores C neighbouring columns of a
// row at once.  fp32 on the bf16 instruction: three pieces a value, scaled so that they reach as
// far down as floats do, eight of nine products (the ninth is below 2^-32 of the whole; two more
// left out cost a lone product up to another rounding), those of one weight in a sum of their own.
// What comes out not finite is multiplied again without the split.
// us before (a launch a tensor, fp32 instruction, rows of two tiles a workgroup) -> here, one tensor
// and three: 93,773 x 64 -> 64 19 -> 15.9, 54 -> 31; 128 -> 128 69 -> 43, 208 -> 93; 5,000 x 64 -> 64
// 7.2 -> 6.1, 21 -> 6.6; 1 M x 64 -> 64, 200 types 117 -> 116, 351 -> 324; 5.7 M x 16 -> 64 378 -> 367.
// (This kernel on the fp32 instruction: 17.7 and 38, 46 and 117, 120 and 328.)  Error against
// float64 at K = 64 1.44e-7 -> 0.45e-7, positive products 1.15e-7 -> 0.49e-7; K = 16 0.74e-7 -> 0.29e-7.
#include "typed_chunks.h"
#include "typed_rows.h"

namespace ga {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kWaves = kBlock / kWave;

// KS steps of 32 k, C blocks of 16 columns a pass: block c holds the columns 16 C pass + n C + c
template <int KS, int C>
__global__ __launch_bounds__(kBlock, KS == 4 ? 2 : KS == 2 ? 3 : 6) void typed_rows_kernel(TypedRows p, int chunk_rows, int passes) {
  __shared__ __attribute__((aligned(16))) uint4 wp[KS][C][3][kWave];
  int type, row0, row1;
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
  for (int i = threadIdx.x; i < KS * C * kWave; i += kBlock) {
    const int l = i & (kWave - 1), c = i / kWave % C, ks = i / kWave / C;
    const int k0 = ks * 32 + (l >> 4) * 4;
    const float *w = W + (l & 15) * C + c;
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int k = k0 + (j & 3) + 4 * (j & 4);
      v[j] = k < K ? w[(int64_t)k * M] : 0.0f;
    }
    uint32_t p3[3][4];
    split<8, false>(v, p3);
#pragma unroll
    for (int h = 0; h < 3; ++h) wp[ks][c][h][l] = make_uint4(p3[h][0], p3[h][1], p3[h][2], p3[h][3]);
  }
  __syncthreads();
  float gate = 1.0f;
  if (p.gate) {
    const float g = p.gate[type];
    gate = p.gate_sigmoid ? 1.0f / (1.0f + expf(-g)) : g;
  }
  for (int r = first; r < row1; r += 16 * kWaves) {
    const Tile now = t;
    asm volatile("" ::: "memory");    // W is read from LDS every time: held, it takes 96 registers
    if (r + 16 * kWaves < row1) fetch(r + 16 * kWaves, t);
    uint4 xf[KS][3];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const float4 lo = now.x[ks][0], up = now.x[ks][1];
      const float v[8] = {lo.x, lo.y, lo.z, lo.w, up.x, up.y, up.z, up.w};
      uint32_t xp[3][4];
      split<8, false>(v, xp);
#pragma unroll
      for (int h = 0; h < 3; ++h) xf[ks][h] = make_uint4(xp[h][0], xp[h][1], xp[h][2], xp[h][3]);
    }
    floatx4 acc[C];
    bool finite = true;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      floatx4 part[4] = {};           // products of pieces of one weight together: 1, 2^-8, 2^-16, 2^-24
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const uint4 wf[3] = {wp[ks][c][0][lane], wp[ks][c][1][lane], wp[ks][c][2][lane]};
        constexpr int px[8] = {0, 0, 1, 0, 1, 2, 1, 2}, pw[8] = {0, 1, 0, 2, 1, 0, 2, 1};
#pragma unroll
        for (int m = 0; m < 8; ++m)
          part[px[m] + pw[m]] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8, xf[ks][px[m]]), __builtin_bit_cast(bf16x8, wf[pw[m]]),
              part[px[m] + pw[m]], 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[c][i] = fmaf(fmaf(fmaf(part[3][i], kPieceScale, part[2][i]), kPieceScale, part[1][i]),
                         kPieceScale, part[0][i]);
        finite = finite && isfinite(acc[c][i]);
      }
    }
    // What is not finite is multiplied again without the split: pieces of an infinity are NaN,
    // and those of a product that overflows may do so with either sign.
    if (__builtin_amdgcn_ballot_w64(!finite) != 0) {
      floatx4 again[C];
#pragma unroll
      for (int c = 0; c < C; ++c) again[c] = floatx4{0, 0, 0, 0};
      for (int k = 0; k < K; ++k)
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            again[c][i] = fmaf(p.X[(int64_t)min(r + 4 * q + i, row1 - 1) * K + k],
                               W[(int64_t)k * M + n * C + c], again[c][i]);
#pragma unroll
      for (int c = 0; c < C; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[c][i] = isfinite(acc[c][i]) ? acc[c][i] : again[c][i];
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
  // chunks of whole rounds of the four wavefronts, as many as the chip holds at a time (four a CU;
  // of 128 values 1,280 are faster than 1,024 or 768: three tensors 93 : 103 us)
  const int64_t target = KS == 4 ? 1280 : 1024;
  const int64_t want = (p.rows * p.n_weights * passes + target - 1) / target;
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
