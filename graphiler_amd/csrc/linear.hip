// Dense node projection with the GAT attention terms in its epilogue (fp32):
//   Z = X @ W,  el[n, h] = <Z[n, h, :], a_l[h, :]>,  er[n, h] = <Z[n, h, :], a_r[h, :]>
// i.e. the dense operators that precede the graph chain in the reference's GAT
// plan (mm(h, fc_weight) and the two halves of mm(z2, attn_weight),
// examples/GAT/GAT.py:25-29 after the split / reorder passes) as one kernel, so
// Z is written once and never re-read for the attention terms.
//
// Tall-skinny GEMM with fp32 operands and fp32 results on the bf16 matrix
// instruction (v_mfma_f32_16x16x32_bf16, 16x the rate of the fp32 one): every
// operand value is split into three bf16 pieces, x = x0 + x1 + x2 (8 significant
// bits each, 24 in all; exact down to 2^-110, below which the third leaves bf16's
// range), and the product is accumulated in fp32 from the six piece products x0w0 +
// x0w1 + x1w0 + x1w1 + x0w2 + x2w0; each is exact in fp32.  The first piece is cut off (no
// value of float's range overflows), the second rounded to nearest: a second piece reaches 2^-7
// and a third 2^-16 of its value, so the three dropped products stay below 2^-22 of |x||w|
// (3.94 x 2^-24 at x = w = 1.0078; 0.36 x 2^-24 root mean square) and have no sign of their own.
// With all three pieces cut off they had the product's, which showed where all products are
// positive (error against float64, 2-norm, 40,000 x 1433 -> 64 1.3e-6 -> 6.2e-7, the vendor GEMM
// 5.8e-7; 232,965 x 602 3.3e-7 -> 3.1e-7, 3.7e-7; both signs 3.7e-7 -> 3.65e-7, 4.4e-7).
// Non-finite inputs give NaN (inf - inf in the split) where fp32 products may give inf.
//
// A workgroup (4 waves) owns 128 rows, each wave 32 rows (2 tiles of 16) x 64
// columns per pass.  Both operands go global -> registers -> LDS in
// slices of 32 k: the MFMA operand layout puts the 16 rows of a tile on 16
// adjacent lanes, so loading X straight into that layout makes every lane its
// own cache access; staged through LDS, adjacent lanes read adjacent addresses
// of a row.  X is staged as fp32 and split after the operand read (each value is
// consumed by exactly one lane); W is split when it is committed to LDS, as three
// [column][k] bf16 arrays, so an operand read is one 16-byte LDS read per piece.
// Loads go through buffer descriptors (fixed lane offsets, the slice as the scalar
// offset), so the loop has no address arithmetic.  Two register sets hold the slices
// one and two ahead of the one being multiplied.  Every wave stages the rows it
// multiplies itself, so the X tile needs one LDS buffer and no barrier (a wave's LDS
// accesses execute in order: the next slice is written after the current one has
// been read); the W pieces, shared by the four waves, have two buffers and cost the
// one barrier per slice.  The W operands of a column block are read while the block
// before it multiplies.  49 KB of LDS and under 168 registers: three workgroups per
// CU when the grid has at least one per CU; smaller grids are latency-bound and run
// the build with the two-per-CU register budget, which is faster there.
// Accumulators come out as D[row][col] with 16 adjacent lanes on 16 adjacent
// columns: Z stores coalesce, and the per-head dot products need one 16-lane DPP
// sum per row and head.
#include "common.h"

namespace ga {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kRT = 2;                                   // 16-row tiles per wave
constexpr int kWaveRows = kRT * 16;                      // 32
constexpr int kWgRows = kWaveRows * (kBlock / kWave);    // 128
constexpr int kCB = 4;                                   // 16-column blocks per pass
constexpr int kPassCols = kCB * 16;                      // 64
constexpr int kSliceK = 32;                              // k per LDS slice
constexpr int kXs = kSliceK + 4;                         // LDS row stride of the X tile
constexpr int kAhead = 2;                                // slices of X on their way (odd rows)
constexpr int kWb = kSliceK / 2 + 4;                      // LDS column stride of a W piece, in bf16 pairs

// The k of element j of lane group lk where X goes straight to its operand: 4 lk .. 4 lk + 3 and
// those 16 further on, so that the four lanes of a row read 64 bytes side by side.
__device__ __forceinline__ int k_of(int lk, int j) { return 4 * lk + (j & 3) + 4 * (j & 4); }

// What follows the k loop of a wavefront's 32 rows and NCB column blocks.
template <bool HAS_ATTN, int NCB>
__device__ __forceinline__ void store_tile(floatx4 (&acc)[kRT][NCB], const float *__restrict__ a_l,
                                           const float *__restrict__ a_r, float *__restrict__ Z,
                                           float *__restrict__ el, float *__restrict__ er,
                                           const float *__restrict__ row_scale, int64_t rows, int M,
                                           int heads, int ldz, int64_t wrow0, int col0) {
  const int lane = threadIdx.x & (kWave - 1), lr = lane & 15, lk = lane >> 4;
  // lane holds rows wrow0 + t*16 + 4*lk + r, column col0 + cb*16 + lr
  // the row factors of the plain projection, all requested before the first store
  float rsv[kRT][4];
  if (!HAS_ATTN) {
#pragma unroll
    for (int t = 0; t < kRT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t row = wrow0 + t * 16 + lk * 4 + r;
        rsv[t][r] = row_scale && row < rows ? row_scale[row] : 1.0f;
      }
  }
  float al[kCB], ar[kCB];
  const int dph = M / heads;
  const int bph = dph >> 4;                              // column blocks per head
  if constexpr (HAS_ATTN) {
#pragma unroll
    for (int cb = 0; cb < kCB; ++cb) {
      const int c = col0 + cb * 16 + lr;
      al[cb] = c < M ? a_l[c] : 0.0f;                    // (heads, dph) is (M,) flat
      ar[cb] = c < M ? a_r[c] : 0.0f;
    }
  }
#pragma unroll
  for (int t = 0; t < kRT; ++t) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t row = wrow0 + t * 16 + lk * 4 + r;
      const bool live = row < rows;
      if (!HAS_ATTN && row_scale) {                      // the plain projection only
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb) acc[t][cb][r] *= rsv[t][r];
      }
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb) {
        const int c = col0 + cb * 16 + lr;
        if (live && c < M) Z[row * ldz + c] = acc[t][cb][r];
      }
      if constexpr (HAS_ATTN) {
        // lane-local products, blocks of one head added, then one 16-lane tree
        float pl[kCB], pr[kCB];
#pragma unroll
        for (int cb = 0; cb < kCB; ++cb) {
          pl[cb] = acc[t][cb][r] * al[cb];
          pr[cb] = acc[t][cb][r] * ar[cb];
        }
        if (bph >= 2) {
          pl[0] += pl[1]; pr[0] += pr[1];
          pl[2] += pl[3]; pr[2] += pr[3];
        }
        if (bph == 4) { pl[0] += pl[2]; pr[0] += pr[2]; }
#pragma unroll
        for (int cb = 0; cb < kCB; ++cb) {
          if (cb % bph == 0) {                           // first block of a head
            const float sl_ = row16_sum(pl[cb]), sr_ = row16_sum(pr[cb]);
            const int head = (col0 + cb * 16) / dph;
            if (live && lr == 0 && head < heads) {
              el[row * heads + head] = sl_;
              er[row * heads + head] = sr_;
            }
          }
        }
      }
    }
  }
}

template <int VK> struct XVec;
template <> struct XVec<4> { using type = float4; };
template <> struct XVec<2> { using type = float2; };

// HAS_ATTN: also produce el / er; requires heads to tile a pass exactly
// (dph = M / heads in {16, 32, 64}).
// VK = widest aligned vector (floats) of a row of X: 4 when K % 4 == 0, 2 when
// K % 2 == 0.  K % VK == 0, so such a vector lies wholly inside or
// wholly outside a row: ragged edges clamp the address at fetch time (a valid
// one, the row's last vector) and zero by select at commit time, where the
// value is consumed anyway; no lane is ever predicated off in the k loop.
// WAVES: waves per SIMD the register allocation aims at (3 or 2)
// NCB: column blocks multiplied and stored, 4 or -- the plain projection onto at most 16
// columns (a GCN layer's hidden width) -- 1; the W tile is staged 64 columns wide either
// way, what shrinks is the matrix work and the operand reads.
template <bool HAS_ATTN, int VK, int WAVES, int NCB = kCB>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(WAVES, WAVES))) void
linear_attn_kernel(
    const float *__restrict__ X, const float *__restrict__ W,
    const float *__restrict__ a_l, const float *__restrict__ a_r,
    float *__restrict__ Z, float *__restrict__ el, float *__restrict__ er,
    const float *__restrict__ row_scale, int64_t rows, int K, int M, int heads, int ldz) {
  static_assert(NCB == kCB || !HAS_ATTN, "the attention epilogue pairs up all four column blocks");
  using xvec_t = typename XVec<VK>::type;
  __shared__ __attribute__((aligned(16))) float xs[kWgRows * kXs];   // wave-private rows, one buffer
  __shared__ __attribute__((aligned(16))) uint32_t wb[2][3][kPassCols * kWb];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);   // in a scalar register
  const int lr = lane & 15, lk = lane >> 4;
  const int col0 = blockIdx.y * kPassCols;               // first column of the pass
  const int64_t wg_row0 = (int64_t)blockIdx.x * kWgRows;
  const int64_t wrow0 = wg_row0 + wave * kWaveRows;
  const int n_slices = (K + kSliceK - 1) / kSliceK;

  // X slice of a wave: its 32 rows x 32 k in vectors of VK floats, kVpr per row; lane
  // i owns vectors i, i + 64, ...: a wave instruction reads 64 * VK * 4
  // contiguous-by-row bytes (2 * VK rows of 128 bytes).  Slices past the last
  // are fetched too (from the clamped address) and never multiplied.
  constexpr int kVpr = kSliceK / VK;                     // vectors per row and slice
  constexpr int kXPieces = kWaveRows * kVpr / kWave;     // 4 / 8 / 16 per thread
  constexpr int kRowStep = kWave / kVpr;                 // rows between a thread's vectors
  struct Stage {
    xvec_t x[kXPieces];
    float w[8];
  };
  // Lane offsets (bytes) never change; the slice / the row of W is the scalar offset.
  // Slices that lie wholly inside the rows (all but the last, and that one too when
  // K % 32 == 0) take paths without clamps and selects.
  const int wc = threadIdx.x & 63, wkg = wave;               // column, group of 8 k
  const int xr = wave * kWaveRows + lane / kVpr, xc = (lane % kVpr) * VK;   // each wave stages its own rows
  const rsrc_t xrs = make_rsrc(X + wg_row0 * K, (uint64_t)(rows - wg_row0) * K * 4);
  const rsrc_t wrs = make_rsrc(W, (uint64_t)K * M * 4);
  uint32_t xoff[kXPieces];                               // the piece in slice 0
#pragma unroll
  for (int j = 0; j < kXPieces; ++j)
    xoff[j] = (uint32_t)((min(wg_row0 + xr + j * kRowStep, rows - 1) - wg_row0) * K + xc) * 4u;
  const uint32_t woff = (uint32_t)min(col0 + wc, M - 1) * 4u;
  const bool w_cols_full = col0 + kPassCols <= M;        // uniform

  auto fetch = [&](int sl, Stage &st) {
    if (sl * kSliceK + kSliceK <= K) {
#pragma unroll
      for (int j = 0; j < kXPieces; ++j)
        st.x[j] = BufLoad<VK>::at(xrs, xoff[j], (uint32_t)sl * (kSliceK * 4));
    } else {
      // clamped to the row's last vector (a valid address); zeroed at commit
      const uint32_t dk = (uint32_t)(min(sl * kSliceK + xc, K - VK) - xc) * 4u;
#pragma unroll
      for (int j = 0; j < kXPieces; ++j) st.x[j] = BufLoad<VK>::at(xrs, xoff[j] + dk, 0);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j)
      st.w[j] = BufLoad<1>::at(wrs, woff, (uint32_t)min(sl * kSliceK + wkg * 8 + j, K - 1) * (uint32_t)M * 4u);
  };
  auto commit = [&](int sl, const Stage &st) {
    const int buf = sl & 1;
    const bool inside = sl * kSliceK + kSliceK <= K;     // uniform
    if (inside) {
#pragma unroll
      for (int j = 0; j < kXPieces; ++j)
        *reinterpret_cast<xvec_t *>(&xs[(xr + j * kRowStep) * kXs + xc]) = st.x[j];
    } else {
      const bool xin = sl * kSliceK + xc < K;
#pragma unroll
      for (int j = 0; j < kXPieces; ++j) {
        xvec_t v = st.x[j];
        if (!xin) v = xvec_t{};
        *reinterpret_cast<xvec_t *>(&xs[(xr + j * kRowStep) * kXs + xc]) = v;
      }
    }
    float wv[8];
    if (inside && w_cols_full) {
#pragma unroll
      for (int j = 0; j < 8; ++j) wv[j] = st.w[j];
    } else {
      const bool cin = col0 + wc < M;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        wv[j] = cin && sl * kSliceK + wkg * 8 + j < K ? st.w[j] : 0.0f;
    }
    uint4 p0, p1, p2;
    split8(wv, p0, p1, p2);
    *reinterpret_cast<uint4 *>(&wb[buf][0][wc * kWb + wkg * 4]) = p0;
    *reinterpret_cast<uint4 *>(&wb[buf][1][wc * kWb + wkg * 4]) = p1;
    *reinterpret_cast<uint4 *>(&wb[buf][2][wc * kWb + wkg * 4]) = p2;
  };

  floatx4 acc[kRT][NCB];
#pragma unroll
  for (int t = 0; t < kRT; ++t)
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) acc[t][cb] = floatx4{0, 0, 0, 0};

  const int xl_ofs = (wave * kWaveRows + lr) * kXs + lk * 8;
  const int wl_ofs = lr * kWb + lk * 4;                  // in uint32 (pairs of bf16)
  auto step = [&](int sl, Stage &next) {
    const int buf = sl & 1;
    float4 xa[kRT][2];
    uint4 wf[2][3];
#pragma unroll
    for (int t = 0; t < kRT; ++t) {
      xa[t][0] = *reinterpret_cast<const float4 *>(&xs[xl_ofs + t * 16 * kXs]);
      xa[t][1] = *reinterpret_cast<const float4 *>(&xs[xl_ofs + t * 16 * kXs + 4]);
    }
    auto read_w = [&](int cb, uint4 (&f)[3]) {
#pragma unroll
      for (int p = 0; p < 3; ++p)
        f[p] = *reinterpret_cast<const uint4 *>(&wb[buf][p][wl_ofs + cb * 16 * kWb]);
    };
    read_w(0, wf[0]);
    commit(sl + 1, next);
    fetch(sl + 3, next);
    uint4 xp[kRT][3];
#pragma unroll
    for (int t = 0; t < kRT; ++t) {
      const float v[8] = {xa[t][0].x, xa[t][0].y, xa[t][0].z, xa[t][0].w,
                          xa[t][1].x, xa[t][1].y, xa[t][1].z, xa[t][1].w};
      split8(v, xp[t][0], xp[t][1], xp[t][2]);
    }
    constexpr int px[6] = {2, 0, 1, 1, 0, 0}, pw[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) {
      if (cb + 1 < NCB) read_w(cb + 1, wf[(cb + 1) & 1]);
#pragma unroll
      for (int q = 0; q < 6; ++q)
#pragma unroll
        for (int t = 0; t < kRT; ++t)
          acc[t][cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8, xp[t][px[q]]), __builtin_bit_cast(bf16x8, wf[cb & 1][pw[q]]),
              acc[t][cb], 0, 0, 0);
    }
    __syncthreads();
  };

  Stage sa, sb;                                          // even / odd slices
  fetch(0, sa);
  fetch(1, sb);
  commit(0, sa);
  fetch(2, sa);
  __syncthreads();
  int sl = 0;
  for (; sl + 1 < n_slices; sl += 2) {
    step(sl, sb);
    step(sl + 1, sa);
  }
  if (sl < n_slices) step(sl, sb);

  store_tile<HAS_ATTN, NCB>(acc, a_l, a_r, Z, el, er, row_scale, rows, M, heads, ldz, wrow0, col0);
}

// Rows of an odd number of values, which only four-byte accesses tile: staged through LDS one
// float at a time they took 32 staged registers and two workgroups a CU.  Here the rows go
// straight to the operand of the matrix instruction with 16-byte loads of 4-byte alignment, 64
// bytes of a row side by side (few_rows' order of k); W as above.  Four workgroups per CU.  us:
// 300,000 x 37 -> 64 38.5 -> 27, 100,000 x 101 26.5 -> 21, 40,000 x 1433 94 -> 66, 60,000 x 1433
// 105 -> 93.  Rows that wider accesses tile are no faster this way (232,965 x 602 162 : 165,
// 1 M x 100 164 : 182).
template <bool HAS_ATTN, int WAVES, int NCB = kCB>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(WAVES, WAVES))) void
linear_odd_kernel(
    const float *__restrict__ X, const float *__restrict__ W,
    const float *__restrict__ a_l, const float *__restrict__ a_r,
    float *__restrict__ Z, float *__restrict__ el, float *__restrict__ er,
    const float *__restrict__ row_scale, int64_t rows, int K, int M, int heads, int ldz) {
  static_assert(NCB == kCB || !HAS_ATTN, "the attention epilogue pairs up all four column blocks");
  __shared__ __attribute__((aligned(16))) uint32_t wb[2][3][kPassCols * kWb];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);   // in a scalar register
  const int lr = lane & 15, lk = lane >> 4;
  const int col0 = blockIdx.y * kPassCols;               // first column of the pass
  const int64_t wg_row0 = (int64_t)blockIdx.x * kWgRows;
  const int64_t wrow0 = wg_row0 + wave * kWaveRows;
  const int n_slices = (K + kSliceK - 1) / kSliceK;

  struct Rows { float4 x[kRT][2]; };
  const rsrc_t xrs = make_rsrc(X + wg_row0 * K, (uint64_t)(rows - wg_row0) * K * 4);
  const rsrc_t wrs = make_rsrc(W, (uint64_t)K * M * 4);
  uint32_t xoff[kRT];                                    // byte offset in slice 0
#pragma unroll
  for (int t = 0; t < kRT; ++t)
    xoff[t] = (uint32_t)((min(wrow0 + t * 16 + lr, rows - 1) - wg_row0) * K + 4 * lk) * 4u;
  const int wc = threadIdx.x & 63, wkg = wave;           // column, lk of the eight k
  const uint32_t woff = (uint32_t)min(col0 + wc, M - 1) * 4u;
  const bool w_cols_full = col0 + kPassCols <= M;        // uniform

  // The last slice, if it is not whole, keeps its k together (8 lk .. 8 lk + 7): fewer of the
  // instruction's partial sums are rounded (error at K = 45 1.07e-7 -> 0.83e-7).
  auto k_in = [&](int sl, int lane_k, int j) __attribute__((always_inline)) {
    return sl * kSliceK + (sl * kSliceK + kSliceK <= K ? k_of(lane_k, j) : 8 * lane_k + j);
  };
  // What lies past the end of X reads as 0 (lane offsets are range-checked); what the last
  // slice reads of the row behind is cleared when it is multiplied.  Slices past the last are
  // fetched too and never multiplied.
  auto fetch_x = [&](int sl, Rows &r) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < kRT; ++t) {
      const bool whole = sl * kSliceK + kSliceK <= K;    // uniform
      const uint32_t at = xoff[t] + (uint32_t)sl * (kSliceK * 4) + (whole ? 0u : 16u * lk);
      r.x[t][0] = BufLoad<4>::at(xrs, at, 0);
      r.x[t][1] = BufLoad<4>::at(xrs, at + (whole ? 64u : 16u), 0);
    }
  };
  // the row of W is the scalar offset: no address arithmetic
  auto fetch_w = [&](int sl, float (&w)[8]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      w[j] = BufLoad<1>::at(wrs, woff, (uint32_t)min(k_in(sl, wkg, j), K - 1) * (uint32_t)M * 4u);
  };
  auto commit_w = [&](int sl, const float (&w)[8]) __attribute__((always_inline)) {
    const int buf = sl & 1;
    float wv[8];
    if (sl * kSliceK + kSliceK <= K && w_cols_full) {    // uniform
#pragma unroll
      for (int j = 0; j < 8; ++j) wv[j] = w[j];
    } else {
      const bool cin = col0 + wc < M;
#pragma unroll
      for (int j = 0; j < 8; ++j) wv[j] = cin && k_in(sl, wkg, j) < K ? w[j] : 0.0f;
    }
    uint4 p0, p1, p2;
    split8(wv, p0, p1, p2);
    *reinterpret_cast<uint4 *>(&wb[buf][0][wc * kWb + wkg * 4]) = p0;
    *reinterpret_cast<uint4 *>(&wb[buf][1][wc * kWb + wkg * 4]) = p1;
    *reinterpret_cast<uint4 *>(&wb[buf][2][wc * kWb + wkg * 4]) = p2;
  };

  floatx4 acc[kRT][NCB];
#pragma unroll
  for (int t = 0; t < kRT; ++t)
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) acc[t][cb] = floatx4{0, 0, 0, 0};

  const int wl_ofs = lr * kWb + lk * 4;                  // in uint32 (pairs of bf16)
  float wn[8];                                           // W of the next slice
  auto step = [&](int sl, Rows &now) __attribute__((always_inline)) {
    const int buf = sl & 1;
    uint4 wf[2][3];
    auto read_w = [&](int cb, uint4 (&f)[3]) {
#pragma unroll
      for (int p = 0; p < 3; ++p)
        f[p] = *reinterpret_cast<const uint4 *>(&wb[buf][p][wl_ofs + cb * 16 * kWb]);
    };
    read_w(0, wf[0]);
    commit_w(sl + 1, wn);
    fetch_w(sl + 2, wn);
    uint4 xp[kRT][3];
#pragma unroll
    for (int t = 0; t < kRT; ++t) {
      float v[8] = {now.x[t][0].x, now.x[t][0].y, now.x[t][0].z, now.x[t][0].w,
                    now.x[t][1].x, now.x[t][1].y, now.x[t][1].z, now.x[t][1].w};
      if (sl * kSliceK + kSliceK > K) {                  // uniform
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = k_in(sl, lk, j) < K ? v[j] : 0.0f;
      }
      split8(v, xp[t][0], xp[t][1], xp[t][2]);
    }
    fetch_x(sl + kAhead, now);
    constexpr int px[6] = {2, 0, 1, 1, 0, 0}, pw[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) {
      if (cb + 1 < NCB) read_w(cb + 1, wf[(cb + 1) & 1]);
#pragma unroll
      for (int q = 0; q < 6; ++q)
#pragma unroll
        for (int t = 0; t < kRT; ++t)
          acc[t][cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8, xp[t][px[q]]), __builtin_bit_cast(bf16x8, wf[cb & 1][pw[q]]),
              acc[t][cb], 0, 0, 0);
    }
    __syncthreads();
  };

  Rows x[kAhead];
#pragma unroll
  for (int i = 0; i < kAhead; ++i) fetch_x(i, x[i]);
  fetch_w(0, wn);
  commit_w(0, wn);
  fetch_w(1, wn);
  __syncthreads();
  for (int sl = 0; sl < n_slices; sl += kAhead) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i)
      if (i == 0 || sl + i < n_slices) step(sl + i, x[i]);
  }

  store_tile<HAS_ATTN, NCB>(acc, a_l, a_r, Z, el, er, row_scale, rows, M, heads, ldz, wrow0, col0);
}

// ---- few rows ------------------------------------------------------------------------------
// A grid of 128-row workgroups that leaves most CUs idle takes as long as one workgroup's chain
// of k slices.  Here a workgroup owns 16 rows and its KS wavefronts share out the slices: each
// loads its operands straight into the layout of the matrix instruction (two 16-byte loads of a
// row and eight of W per column block and slice, the next slice's behind this one's), and the
// partial tiles are added through LDS in the order of the wavefronts.
// The product is the fp32 instruction's: W is used for 16 rows only, so that splitting it, as
// above, takes as long as the matrix time it saves, and this form stands where a product of
// torch's would: infinities, products that overflow and operands near the end of the range come
// out as they do there.  Two or four sums a block, so that a chain of roundings is short: 2-norm
// against float64, values of both signs / of one, here, torch's product and the split: 2,708 x 1433
// -> 64 1.8e-7, 3.4e-7, 2.0e-7 / 0.6e-7, 1.5e-7, 0.8e-7; 16,000 x 16 0.6e-7, 0.7e-7, 0.4e-7.
// us, 128-row workgroups -> here (split: -): 2,708 x 1433 -> 64 50 -> 11.3 (11.8), 5,000 x 300 14.6
// -> 7.0 (7.2), 19,717 x 500 -> 16 17.2 -> 8.5 (8.7), 100,000 x 300 -> 32 39 -> 36 (33).
template <bool HAS_ATTN, int KS, int NCB>
__global__ __launch_bounds__(KS * kWave, NCB == 2 ? 3 : 2) void linear_few_rows_kernel(
    const float *__restrict__ X, const float *__restrict__ W, const float *__restrict__ a_l,
    const float *__restrict__ a_r, float *__restrict__ Z, float *__restrict__ el,
    float *__restrict__ er, const float *__restrict__ row_scale, int64_t rows, int K, int M,
    int heads, int ldz) {
  constexpr int kRows = 16, kCols = NCB * 16, kTile = kRows * kCols;
  __shared__ float part[KS][kTile];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int lr = lane & 15, lk = lane >> 4;
  const int col0 = blockIdx.y * kCols;
  const int64_t row0 = (int64_t)blockIdx.x * kRows;
  const int n_slices = (K + kSliceK - 1) / kSliceK;
  const rsrc_t xrs = make_rsrc(X + row0 * K, (uint64_t)min((int64_t)kRows, rows - row0) * K * 4);
  const rsrc_t wrs = make_rsrc(W, (uint64_t)K * M * 4);
  const uint32_t xoff = (uint32_t)((min(row0 + lr, rows - 1) - row0) * K + lk * 4) * 4u;
  uint32_t woff[NCB];
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb)
    woff[cb] = ((uint32_t)(lk * 4) * M + min(col0 + cb * 16 + lr, M - 1)) * 4u;
  constexpr int kSums = NCB == 4 ? 2 : 4;
  floatx4 acc[NCB][kSums];
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
    for (int i = 0; i < kSums; ++i) acc[cb][i] = floatx4{0, 0, 0, 0};
  struct Slice {
    float4 x[2];
    float w[NCB][8];
  };
  // Loads past the end of X and of W give 0 (the lane offsets are range-checked; W's columns are
  // clamped, so an offset past K rows is past its end); what the last slice reads of the row
  // behind it is cleared before it is multiplied.
  auto fetch = [&](int sl, Slice &s) __attribute__((always_inline)) {
    const uint32_t xs = xoff + (uint32_t)sl * (kSliceK * 4);
    const uint32_t ws = (uint32_t)sl * kSliceK * (uint32_t)M * 4u;
    s.x[0] = BufLoad<4>::at(xrs, xs, 0);
    s.x[1] = BufLoad<4>::at(xrs, xs + 64, 0);
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
      for (int j = 0; j < 8; ++j)
        s.w[cb][j] = BufLoad<1>::at(wrs, woff[cb] + ws + (uint32_t)(k_of(0, j) * M) * 4u, 0);
  };
  auto multiply = [&](int sl, const Slice &s) __attribute__((always_inline)) {
    float v[8] = {s.x[0].x, s.x[0].y, s.x[0].z, s.x[0].w, s.x[1].x, s.x[1].y, s.x[1].z, s.x[1].w};
    if (sl * kSliceK + kSliceK > K) {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = sl * kSliceK + k_of(lk, j) < K ? v[j] : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb)
        acc[cb][j % kSums] =
            __builtin_amdgcn_mfma_f32_16x16x4f32(v[j], s.w[cb][j], acc[cb][j % kSums], 0, 0, 0);
  };
  if (wave < n_slices) {
    Slice a, b;
    fetch(wave, a);
    for (int sl = wave; sl < n_slices; sl += 2 * KS) {
      if (sl + KS < n_slices) fetch(sl + KS, b);
      multiply(sl, a);
      if (sl + KS >= n_slices) break;
      if (sl + 2 * KS < n_slices) fetch(sl + 2 * KS, a);
      multiply(sl + KS, b);
    }
  }
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float z = acc[cb][0][r] + acc[cb][1][r];
      if constexpr (kSums == 4) z += acc[cb][2][r] + acc[cb][3][r];
      part[wave][(lk * 4 + r) * kCols + cb * 16 + lr] = z;
    }
  __syncthreads();
  const int dph = M / heads;
#pragma unroll
  for (int i = threadIdx.x; i < kTile; i += KS * kWave) {   // lane = column, or several rows of them
    float z = 0.0f;
#pragma unroll
    for (int w = 0; w < KS; ++w) z += part[w][i];
    const int64_t row = row0 + i / kCols;
    const int c = col0 + i % kCols;
    const bool live = row < rows && c < M;
    if (!HAS_ATTN && row_scale && live) z *= row_scale[row];
    if (live) Z[row * ldz + c] = z;
    if constexpr (HAS_ATTN) {             // a head's columns lie in one wavefront
      float l = row16_sum(c < M ? z * a_l[c] : 0.0f), r = row16_sum(c < M ? z * a_r[c] : 0.0f);
      if (dph >= 32) { l += __shfl_xor(l, 16); r += __shfl_xor(r, 16); }
      if (dph == 64) { l += __shfl_xor(l, 32); r += __shfl_xor(r, 32); }
      if (live && c % dph == 0) {
        el[row * heads + c / dph] = l;
        er[row * heads + c / dph] = r;
      }
    }
  }
}

// Where the form above is taken.  A plain product of a few thousand rows (`plain`, below kFewRows)
// stands where a product of torch's would: always, whatever the other form takes (16,000 x 16 -> 64
// 6.0 : 5.2 us).  Otherwise where it is the faster one, us here : there.  Up to 16 columns small
// grids and long rows (40,000 x 128 6.2 : 8.3, 100,000 x 300 23 : 31, 100,000 x 16 9.2 : 7.5, 150,000
// x 600 82 : 78), up to 32 with twice the matrix time a row (40,000 x 128 9.8 : 10.9, 70,000 x 128
// 15.8 : 14.8, 100,000 x 600 56 : 64, 150,000 x 300 52 : 47).  64 columns: two workgroups of tiles a
// CU at once (8,000 x 64 4.4 : 6.0, with attention terms 6.5 : 7.4; 10,000 x 64 with them 10.4 : 7.5),
// twice as many of long rows (with them 13,000 x 600 23 : 26, x 128 11.6 : 9.8; 20,000 x 600 33 : 26).
constexpr int64_t kFewRows = 16'384;
bool few_rows(int64_t rows, int64_t K, int64_t M, bool plain) {
  if ((K + kSliceK) * M >= ((int64_t)1 << 29)) return false;       // 32-bit offsets into W
  if (plain && M <= 64 && rows < kFewRows) return true;
  const int64_t slices = (K + kSliceK - 1) / kSliceK;
  if (M <= 32) {
    const int64_t most = M <= 16 ? 300'000 : slices >= 8 ? 100'000 : 40'000;
    return rows <= 20'000 || (slices >= 4 && rows <= most && rows * K <= ((int64_t)64 << 20));
  }
  const int64_t tiles = (rows + 15) / 16 * ((M + 63) / 64);
  return tiles <= 512 || (tiles <= 1024 && slices >= 10);
}

int launch_linear(const float *X, const float *W, const float *a_l, const float *a_r, float *Z,
                  float *el, float *er, const float *row_scale, int64_t rows, int64_t K,
                  int64_t M, int64_t heads, int64_t ldz, ga_stream_t stream) {
  if (rows < 0 || K <= 0 || M <= 0 || heads <= 0 || M % heads) return GA_EINVAL;
  if (rows > 0x7fffffff || K > 0x7fffffff || M > 0x7fffffff) return GA_EINVAL;
  if (ldz < M || ldz > 0x7fffffff) return GA_EINVAL;
  if (rows == 0) return GA_OK;
  if (!X || !W || !Z) return GA_EINVAL;
  // 32-bit byte offsets: 128 rows of K floats, and all of W
  if (K > (1 << 22) || K * M >= ((int64_t)1 << 30)) return GA_EUNSUPPORTED;
  const bool attn = el != nullptr || er != nullptr;
  if (attn && (!el || !er || !a_l || !a_r)) return GA_EINVAL;
  if (attn && row_scale) return GA_EINVAL;
  if (!aligned(X, 4) || !aligned(W, 4) || !aligned(Z, 4) || (row_scale && !aligned(row_scale, 4)))
    return GA_EALIGN;
  const int vk = (K % 4 == 0 && aligned(X, 16)) ? 4 : ((K % 2 == 0 && aligned(X, 8)) ? 2 : 1);
  const int64_t dph = M / heads;
  if (attn && !(dph == 16 || dph == 32 || dph == 64)) return GA_EUNSUPPORTED;
  const int64_t gx = (rows + kWgRows - 1) / kWgRows;
  const int64_t gy = (M + kPassCols - 1) / kPassCols;
  if (gx > 0x7fffffff || gy > 65535) return GA_EUNSUPPORTED;
  hipStream_t s = (hipStream_t)stream;
  if (few_rows(rows, K, M, !attn)) {
    const int ncb = M > 32 ? 4 : M > 16 ? 2 : 1;
    const dim3 grid((unsigned)((rows + 15) / 16), (unsigned)((M + 16 * ncb - 1) / (16 * ncb)));
#define GA_LAUNCH_FEW(ATTN, KS, NCB)                                                               \
  hipLaunchKernelGGL((linear_few_rows_kernel<ATTN, KS, NCB>), grid, dim3(KS * kWave), 0, s, X, W,  \
                     a_l, a_r, Z, el, er, row_scale, rows, (int)K, (int)M, (int)heads, (int)ldz)
#define GA_LAUNCH_FEW_NCB(ATTN, KS)                 \
  do {                                              \
    if (ncb == 4) GA_LAUNCH_FEW(ATTN, KS, 4);       \
    else if (ncb == 2) GA_LAUNCH_FEW(ATTN, KS, 2);  \
    else GA_LAUNCH_FEW(ATTN, KS, 1);                \
  } while (0)
    // at most a workgroup per CU: eight wavefronts halve the chain; with more they crowd each other
    const bool crowded = grid.x * grid.y > 256;
    if (attn && crowded) GA_LAUNCH_FEW_NCB(true, 4);
    else if (attn) GA_LAUNCH_FEW_NCB(true, 8);
    else if (crowded) GA_LAUNCH_FEW_NCB(false, 4);
    else GA_LAUNCH_FEW_NCB(false, 8);
#undef GA_LAUNCH_FEW_NCB
#undef GA_LAUNCH_FEW
    return launch_status();
  }
#define GA_LAUNCH_LINEAR_NCB(ATTN, VK, WAVES, NCB)                                  \
  hipLaunchKernelGGL((linear_attn_kernel<ATTN, VK, WAVES, NCB>),                   \
                     dim3((unsigned)gx, (unsigned)gy), dim3(kBlock), 0, s, X, W, a_l, a_r, Z, el, \
                     er, row_scale, rows, (int)K, (int)M, (int)heads, (int)ldz)
#define GA_LAUNCH_LINEAR(ATTN, VK, WAVES)                           \
  do {                                                              \
    if (!ATTN && M <= 16) GA_LAUNCH_LINEAR_NCB(false, VK, WAVES, 1); \
    else GA_LAUNCH_LINEAR_NCB(ATTN, VK, WAVES, kCB);                 \
  } while (0)
#define GA_LAUNCH_LINEAR_VK(ATTN, WAVES)                 \
  do {                                                   \
    if (vk == 4) GA_LAUNCH_LINEAR(ATTN, 4, WAVES);       \
    else GA_LAUNCH_LINEAR(ATTN, 2, WAVES);               \
  } while (0)
  // three workgroups per CU once there is at least one per CU to start with; below
  // that the kernel is latency-bound and the build with the larger register budget
  // (two per CU) has the shorter dependent chain per slice.
  constexpr int64_t kDeviceCUs = 256;                    // MI355X
  const bool dense_grid = gx * gy >= kDeviceCUs;
  if (vk == 1) {
#define GA_LAUNCH_ODD(ATTN, NCB)                                                                    \
  hipLaunchKernelGGL((linear_odd_kernel<ATTN, 4, NCB>), dim3((unsigned)gx, (unsigned)gy), dim3(kBlock), \
                     0, s, X, W, a_l, a_r, Z, el, er, row_scale, rows, (int)K, (int)M, (int)heads, (int)ldz)
    if (attn) GA_LAUNCH_ODD(true, kCB);
    else if (M <= 16) GA_LAUNCH_ODD(false, 1);
    else GA_LAUNCH_ODD(false, kCB);
#undef GA_LAUNCH_ODD
    return launch_status();
  }
  if (attn) {
    if (dense_grid) GA_LAUNCH_LINEAR_VK(true, 3);
    else GA_LAUNCH_LINEAR_VK(true, 2);
  } else {
    if (dense_grid) GA_LAUNCH_LINEAR_VK(false, 3);
    else GA_LAUNCH_LINEAR_VK(false, 2);
  }
#undef GA_LAUNCH_LINEAR_VK
#undef GA_LAUNCH_LINEAR
#undef GA_LAUNCH_LINEAR_NCB
  return launch_status();
}
}  // namespace
}  // namespace ga

extern "C" int ga_linear_attn(const float *X, const float *W, const float *a_l,
                              const float *a_r, float *Z, float *el, float *er,
                              int64_t rows, int64_t K, int64_t M, int64_t heads,
                              ga_stream_t stream) {
  return ga::launch_linear(X, W, a_l, a_r, Z, el, er, nullptr, rows, K, M, heads, M, stream);
}

extern "C" int ga_linear_attn_strided(const float *X, const float *W, const float *a_l,
                                      const float *a_r, float *Z, int64_t ldz, float *el,
                                      float *er, int64_t rows, int64_t K, int64_t M,
                                      int64_t heads, ga_stream_t stream) {
  return ga::launch_linear(X, W, a_l, a_r, Z, el, er, nullptr, rows, K, M, heads, ldz, stream);
}

extern "C" int ga_linear_rows_scaled(const float *X, const float *W, const float *row_scale,
                                     float *Z, int64_t rows, int64_t K, int64_t M,
                                     ga_stream_t stream) {
  return ga::launch_linear(X, W, nullptr, nullptr, Z, nullptr, nullptr, row_scale, rows, K, M, 1,
                           M, stream);
}
