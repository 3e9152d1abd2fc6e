// Matrix products of few rows: y[t][n] = sum_k x[t][k] w[n][k] (+ bias[n]), t < 32, bf16 with fp32 sums: the projections of a decode step.
//
// Bound by the weights' way from memory (below a few MB, by one trip to it; at 17 to 32 rows by the rows' image through the first cache).  Every
// weight is read once, straight into the registers of the lane that feeds it to the matrix cores: lane l holds output l % 16, channels
// 8 (l / 16) .. + 7 and the 8 that lie 32 further on, of blocks of 64 channels that the waves of a workgroup share out, so one load reads 64
// neighbouring bytes of each output.  All of a tile's blocks (at most four a wave) are in flight before its first product, the next tile's while the
// waves' sums meet in LDS, and the rows' image stays in registers from tile to tile.  A row's result does not depend on the other rows of the step.
// Measured against the library's product (us, weights cold, N x K): 1 row 1024 x 1024 5.8 -> 3.2, 2048 x 2048 11.1 -> 4.8, 2048 x 4096 14.6 -> 7.3,
// 16384 x 2048 17.5 -> 13.6, 151936 x 2048 204 -> 112 (5.5 TB/s); 16 rows 5120 x 2048 12.2 -> 8.0; 32 rows 2048 x 2048 11.2 -> 7.6.
#include "mixers_mfma.h"

namespace gbxm {
namespace {

constexpr int BK = 64;

// One product of a launch.
struct RowsProduct {
  const bf16_t* x;
  int64_t x_stride;
  const bf16_t *w, *bias;
  bf16_t* y;
  int64_t y_stride;
  int N;
};

// Workgroups walk over tiles of 16 outputs, from `block` on in steps of `step` (<= their number).  MT: tiles of 16 rows.  UNROLL: blocks a wave at most, K <= BK UNROLL WAVES.
template <int MT, int WAVES, int UNROLL>
__device__ __forceinline__ void linear_rows(const bf16_t* __restrict__ x, int64_t x_stride, const bf16_t* __restrict__ w, const bf16_t* __restrict__ bias,
                                            bf16_t* __restrict__ y, int64_t y_stride, int T, int N, int K, int block, int step) {
  __shared__ float part[2][WAVES][MT * 256];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r = lane & 15, q = lane >> 4;
  const int blocks = K / BK, tiles = (N + 15) / 16;
  u32x4 a[UNROLL][2], b[UNROLL][MT][2];
  int at[UNROLL];                            // (past the end: the last block, not added)
#pragma unroll
  for (int u = 0; u < UNROLL; ++u) at[u] = min(wave + u * WAVES, blocks - 1) * BK + 8 * q;
  auto load_w = [&](int tile) {
    const bf16_t* wp = w + static_cast<int64_t>(min(tile * 16 + r, N - 1)) * K;
#pragma unroll
    for (int u = 0; u < UNROLL; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) a[u][h] = *reinterpret_cast<const u32x4*>(wp + at[u] + 32 * h);
  };
  load_w(block);
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const bf16_t* xp = x + min(16 * m + r, T - 1) * x_stride;
#pragma unroll
    for (int u = 0; u < UNROLL; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) b[u][m][h] = *reinterpret_cast<const u32x4*>(xp + at[u] + 32 * h);
  }
  int which = 0;
  for (int tile = block; tile < tiles; tile += step, which ^= 1) {
    f32x4v acc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = f32x4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      if (wave + u * WAVES < blocks) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int m = 0; m < MT; ++m) acc[m] = mfma_bf16_16(a[u][h], b[u][m][h], acc[m]);
      }
    }
    if (tile + step < tiles) load_w(tile + step);
    float* mine = part[which][wave];         // two buffers: a tile's sums are read before the barrier of the next one's
#pragma unroll
    for (int m = 0; m < MT; ++m) *reinterpret_cast<f32x4v*>(&mine[(m * 16 + r) * 16 + 4 * q]) = acc[m];
    __syncthreads();
    for (int i = threadIdx.x; i < MT * 256; i += 64 * WAVES) {
      const int n = tile * 16 + (i & 15), t = i >> 4;
      float s = 0.f;
#pragma unroll
      for (int v = 0; v < WAVES; ++v) s += part[which][v][i];
      if (n < N && t < T) y[t * y_stride + n] = f32_to_bf16(bias ? s + to_f32(bias[n]) : s);
    }
  }
}

template <int MT, int WAVES, int UNROLL>
__global__ __launch_bounds__(64 * WAVES) void linear_rows_kernel(const bf16_t* __restrict__ x, int64_t x_stride, const bf16_t* __restrict__ w,
                                                                const bf16_t* __restrict__ bias, bf16_t* __restrict__ y, int64_t y_stride, int T, int N,
                                                                int K) {
  linear_rows<MT, WAVES, UNROLL>(x, x_stride, w, bias, y, y_stride, T, N, K, blockIdx.x, gridDim.x);
}
// Two products of one contraction length, of rows of their own, which alone are too few tiles for the chip and a launch each: workgroups [0, blocks) take the first.  The low-rank
// decay and gate of a recurrent mixer, 1 row of 512 x 64 and 1024 x 64: two launches | this, us 3.7 | 2.1.
template <int MT, int WAVES, int UNROLL>
__global__ __launch_bounds__(64 * WAVES) void linear_rows_pair_kernel(const RowsProduct a, const RowsProduct b, int T, int K, int blocks) {
  const bool second = static_cast<int>(blockIdx.x) >= blocks;
  const RowsProduct p = second ? b : a;
  linear_rows<MT, WAVES, UNROLL>(p.x, p.x_stride, p.w, p.bias, p.y, p.y_stride, T, p.N, K, second ? blockIdx.x - blocks : blockIdx.x, second ? gridDim.x - blocks : blocks);
}

// Waves: as many as give each of them at most four blocks of K; workgroups: what the chip holds at a time (8 waves a CU measured best, the 16-wave
// form needs 16), so that long outputs stream.  A form holds as many blocks a wave as there are (with four for all of them the missing ones were the
// last one's again, requests that nothing hides in long outputs; library | four | as many as there are, us: 1 row of 151936 x 64 12.2 | 19.9 | 9.1, 50304 x 2560
// 48.6 | 53.5 | 45.3, 16 rows of it 49.4 | 57.1 | 51.3, 32 rows of 50304 x 1152 24.8 | 38.6 | 32.0).
template <int WAVES, int UNROLL>
void launch_rows(hipStream_t s, const void* x, int64_t x_stride, const void* w, const void* bias, void* y, int64_t y_stride, int T, int N, int K) {
  const int grid = min((N + 15) / 16, 256 * (WAVES < 8 ? 8 / WAVES : 1));
#define GBXM_ROWS(MT)                                                                                                                                \
  linear_rows_kernel<MT, WAVES, UNROLL><<<grid, 64 * WAVES, 0, s>>>(static_cast<const bf16_t*>(x), x_stride, static_cast<const bf16_t*>(w),           \
                                                                    static_cast<const bf16_t*>(bias), static_cast<bf16_t*>(y), y_stride, T, N, K)
  if constexpr (WAVES <= 8) {
    if (T > 16) { GBXM_ROWS(2); return; }
  }
  GBXM_ROWS(1);
#undef GBXM_ROWS
}

}  // namespace
}  // namespace gbxm

using namespace gbxm;

extern "C" int gbxm_linear_rows(const void* x, int64_t x_stride, const void* w, const void* bias, void* y, int64_t y_stride, int64_t T_, int32_t N, int32_t K,
                                void* stream) {
  if (!x || !w || !y || T_ < 0 || N < 1 || K < 1 || x_stride < K || y_stride < N) return fail(GBXM_ERR_INVALID, "linear_rows: bad argument");
  if (T_ > 32 || K % BK || K > (T_ > 16 ? 2048 : 4096) || x_stride % 8 || !all_aligned(16, static_cast<const char*>(x), static_cast<const char*>(w)))
    return fail(GBXM_ERR_UNSUPPORTED, "linear_rows: 16 rows of up to 4096 channels or 32 of 2048, in multiples of %d, 16-byte aligned", BK);
  if (N > (1 << 26)) return fail(GBXM_ERR_UNSUPPORTED, "linear_rows: %d outputs", N);
  if (T_ == 0) return GBXM_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int T = static_cast<int>(T_);
#define GBXM_FORM(WAVES, UNROLL) if (K <= BK * WAVES * UNROLL) launch_rows<WAVES, UNROLL>(s, x, x_stride, w, bias, y, y_stride, T, N, K)
  GBXM_FORM(2, 1);
  else GBXM_FORM(2, 2);
  else GBXM_FORM(2, 3);
  else GBXM_FORM(2, 4);
  else GBXM_FORM(4, 3);
  else GBXM_FORM(4, 4);
  else GBXM_FORM(8, 3);
  else GBXM_FORM(8, 4);
  else GBXM_FORM(16, 3);
  else GBXM_FORM(16, 4);
#undef GBXM_FORM
  return after_launch("linear_rows");
}

// For this package's own Python layer; not part of the public header.  Neither product has a bias.
extern "C" int gbxm_linear_rows_pair(const void* x0, int64_t x0_stride, const void* w0, void* y0, int32_t N0, const void* x1, int64_t x1_stride, const void* w1, void* y1,
                                     int32_t N1, int64_t T_, int32_t K, void* stream) {
  if (!x0 || !w0 || !y0 || !x1 || !w1 || !y1 || T_ < 0 || N0 < 1 || N1 < 1 || K < 1 || x0_stride < K || x1_stride < K) return fail(GBXM_ERR_INVALID, "linear_rows_pair: bad argument");
  if (T_ > 32 || K % BK || K > 512 || x0_stride % 8 || x1_stride % 8 || N0 > (1 << 26) || N1 > (1 << 26) ||
      !all_aligned(16, static_cast<const char*>(x0), static_cast<const char*>(w0), static_cast<const char*>(x1), static_cast<const char*>(w1)))
    return fail(GBXM_ERR_UNSUPPORTED, "linear_rows_pair: 32 rows of up to 512 channels, in multiples of %d, 16-byte aligned", BK);
  if (T_ == 0) return GBXM_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int T = static_cast<int>(T_);
  const RowsProduct a{static_cast<const bf16_t*>(x0), x0_stride, static_cast<const bf16_t*>(w0), nullptr, static_cast<bf16_t*>(y0), N0, N0};
  const RowsProduct b{static_cast<const bf16_t*>(x1), x1_stride, static_cast<const bf16_t*>(w1), nullptr, static_cast<bf16_t*>(y1), N1, N1};
  const int g0 = min((N0 + 15) / 16, 512), g1 = min((N1 + 15) / 16, 512);
#define GBXM_FORM(UNROLL)                                                                                                \
  if (K <= BK * 2 * UNROLL) {                                                                                           \
    if (T > 16) linear_rows_pair_kernel<2, 2, UNROLL><<<g0 + g1, 128, 0, s>>>(a, b, T, K, g0);                           \
    else linear_rows_pair_kernel<1, 2, UNROLL><<<g0 + g1, 128, 0, s>>>(a, b, T, K, g0);                                  \
    return after_launch("linear_rows_pair");                                                                            \
  }
  GBXM_FORM(1)
  GBXM_FORM(2)
  GBXM_FORM(3)
  GBXM_FORM(4)
#undef GBXM_FORM
  return fail(GBXM_ERR_UNSUPPORTED, "linear_rows_pair: contraction of %d", K);
}
