// Router logits of prompt-sized steps: logits[t][e] = sum_k h[t][k] router[e][k], bf16 rows, fp32 router, fp32 sums on the matrix cores.
//
// An fp32 weight is the sum of three bf16 numbers (its upper eight bits, the next eight, the rest: both differences are exact), and a product of two bf16
// numbers is exact in fp32: three bf16 products a weight round less than one fp32 product does, at five times the rate of the fp32 instruction (which took
// 38 us for the first line below, the library beside its widened copy 47).
// Bound by the splitting, 5.5 instructions a weight and workgroup, with the router's way through the first cache beside it; a workgroup takes 32 rows x 64
// experts (32 where those are one round of the CUs).  Its eight waves share out the channels: lane l of a block of 32 holds expert (and row) l % 16, channels
// 4 (l / 16) .. + 3 of each half, so a load reads 64 neighbouring bytes of an expert; the next block's operands load under the products.  The waves' sums meet
// in LDS in a fixed order: a row's logits do not depend on the other rows.
// Logits that are not finite are summed again in fp32, on the matrix cores, by the workgroup that meets one: an infinity has no rest, and infinity times a rest
// of zero is no number.  A thread's own sum of K terms for each of them took 1 905 us where all of 3481 rows x 128 experts x 2048 are odd and 586 where one row is; 51
// and 49 here.
// Widened copy and library | this, us: 3481 rows x 128 experts x 2048 46.2 | 25.6, 8192 x 64 x 2048 38.5 | 25.7, 8192 x 32 x 1024 24.8 | 10.6 (error against 64 bits
// 8.1e-7 | 1.8e-7 of the logits' norm); the rule is where the rows are (mixer_ops.py: router_tiles_win).
#include "mixers_mfma.h"

namespace gbxm {
namespace {

constexpr int RW = 8;           // waves
constexpr int OUT = -16;        // byte offset (as unsigned) beyond every buffer: zeros

// NT: tiles of 16 experts.  LDS: a wave's sums, row r's quad q (four experts) at place q ^ r.
template <int NT>
__global__ __launch_bounds__(64 * RW) void router_tile_kernel(const bf16_t* __restrict__ h, const float* __restrict__ router, float* __restrict__ logits,
                                                            int T, int K, int E) {
  __shared__ __attribute__((aligned(16))) float part[RW][32][16 * NT];
  __shared__ int met;                                                   // a logit that is not finite (written before the sums' barrier, read after the next one)
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), fr = lane & 15, fk = lane >> 4;
  const int t0 = blockIdx.x * 32, e0 = blockIdx.y * 16 * NT, steps = (K + 31) / 32;
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(h + static_cast<int64_t>(t0) * K), 0, 0x7FFFFFFF, 0x00020000);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(router), 0, 0x7FFFFFFF, 0x00020000);
  int xo[2], wo[NT];
#pragma unroll
  for (int i = 0; i < 2; ++i) xo[i] = min(16 * i + fr, T - 1 - t0) * K * 2 + fk * 8;
#pragma unroll
  for (int j = 0; j < NT; ++j) wo[j] = min(e0 + 16 * j + fr, E - 1) * K * 4 + fk * 16;
  struct Block { u32x2 x[2][2]; u32x4 w[NT][2]; };
  auto load = [&](Block& b, int s) {                                    // (past the end, as past K: zeros)
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const bool in = s * 32 + q * 16 + fk * 4 < K;
#pragma unroll
      for (int i = 0; i < 2; ++i) b.x[i][q] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rx, in ? xo[i] + q * 32 : OUT, s * 64, 0));
#pragma unroll
      for (int j = 0; j < NT; ++j) b.w[j][q] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, in ? wo[j] + q * 64 : OUT, s * 128, 0));
    }
  };
  f32x4v acc[2][NT];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x4v{0};
  // the upper halves of two words as a bf16 pair; what is left of a word without its upper half
  auto upper = [](unsigned a, unsigned b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); };
  auto rest = [](unsigned a) { return __float_as_uint(__uint_as_float(a) - __uint_as_float(a & 0xFFFF0000u)); };
  auto mul = [&](const Block& b) {
    u32x4 x[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) x[i] = u32x4{b.x[i][0].x, b.x[i][0].y, b.x[i][1].x, b.x[i][1].y};
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      unsigned w[8] = {b.w[j][0].x, b.w[j][0].y, b.w[j][0].z, b.w[j][0].w, b.w[j][1].x, b.w[j][1].y, b.w[j][1].z, b.w[j][1].w};
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        const u32x4 f = u32x4{upper(w[0], w[1]), upper(w[2], w[3]), upper(w[4], w[5]), upper(w[6], w[7])};
#pragma unroll
        for (int i = 0; i < 2; ++i) acc[i][j] = mfma_bf16_16(f, x[i], acc[i][j]);
#pragma unroll
        for (int q = 0; q < 8; ++q) w[q] = rest(w[q]);
      }
    }
  };
  Block b0, b1;
  load(b0, wave);
  for (int s = wave; s < steps; s += 2 * RW) {
    load(b1, s + RW);
    __builtin_amdgcn_sched_barrier(0);                                  // (loads that move down to their use wait for themselves)
    mul(b0);
    __builtin_amdgcn_sched_barrier(0);
    load(b0, s + 2 * RW);
    __builtin_amdgcn_sched_barrier(0);
    mul(b1);
    __builtin_amdgcn_sched_barrier(0);
  }
  constexpr int SW = 4 * NT - 1 < 15 ? 4 * NT - 1 : 15;
  const int row = tid / (4 * NT), q = tid % (4 * NT), t = t0 + row, e = e0 + 4 * q;
  const bool live = row < 32 && t < T && e < E;
  auto meet = [&]() {                                                   // the waves' sums of this thread's four logits
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) *reinterpret_cast<f32x4v*>(&part[wave][16 * i + fr][((4 * j + fk) ^ (fr & SW)) * 4]) = acc[i][j];
    __syncthreads();
    f32x4v sum = f32x4v{0};
    if (live) {
#pragma unroll
      for (int w = 0; w < RW; ++w) sum += *reinterpret_cast<const f32x4v*>(&part[w][row][(q ^ (row & SW)) * 4]);
    }
    return sum;
  };
  auto leave = [&](const f32x4v& v) {
    float* out = logits + static_cast<int64_t>(t) * E + e;
    if (E % 4 == 0) *reinterpret_cast<f32x4v*>(out) = v;
    else
      for (int i = 0; i < 4 && e + i < E; ++i) out[i] = v[i];
  };
  if (tid == 0) met = 0;
  f32x4v v = meet();
  if (live) {
    bool odd = false;
    for (int i = 0; i < 4 && e + i < E; ++i) odd |= !(fabsf(v[i]) < INFINITY);
    if (odd) met = 1;
    leave(v);
  }
  __syncthreads();
  if (!met) return;                                                     // (the whole workgroup, past its last read of the sums)
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x4v{0};
#pragma unroll 1
  for (int s = wave; s < steps; s += RW) {
    load(b0, s);
#pragma unroll
    for (int h = 0; h < 8; ++h)                                         // channel h % 4 of the lane's four in half h / 4
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const unsigned pair = b0.x[i][h >> 2][(h & 3) >> 1];
        const float x = __uint_as_float(h & 1 ? pair & 0xFFFF0000u : pair << 16);
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(b0.w[j][h >> 2][h & 3]), x, acc[i][j], 0, 0, 0);
      }
  }
  const f32x4v whole = meet();
  if (!live) return;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (!(fabsf(v[i]) < INFINITY)) v[i] = whole[i];
  leave(v);
}

}  // namespace
}  // namespace gbxm

using namespace gbxm;

extern "C" int gbxm_router_tiles(const void* h, const float* router, float* logits, int64_t T, int32_t K, int32_t E, void* stream) {
  if (!h || !router || !logits || T < 0 || K < 1 || E < 1) return fail(GBXM_ERR_INVALID, "router_tiles: bad argument");
  if (K % 8 || (reinterpret_cast<uintptr_t>(h) | reinterpret_cast<uintptr_t>(router) | reinterpret_cast<uintptr_t>(logits)) % 16 || T > 0x3fffffff ||
      static_cast<int64_t>(E) * K >= (1 << 29) || E > 0x100000 || K > 0x100000)
    return fail(GBXM_ERR_UNSUPPORTED, "router_tiles: channels in multiples of 8, operands 16-byte aligned, a router under 2 GB");
  if (T == 0) return GBXM_OK;
  const int64_t rows = (T + 31) / 32;
  // 32 experts a workgroup where those fill one round of the CUs at most, else 64, whose rounds are half as many (us, 32 | 64: 2047 rows x 128 x 2048 17.6 | 24.6,
  // 1024 x 256 x 2048 17.5 | 24.6, 2500 x 128 x 2048 31.6 | 24.7, 4500 x 64 x 2048 31.7 | 25.0); a router of no more is not the wider one's (12000 x 32 x 2048 31.8 | 37.2)
  const bool wide = E > 32 && rows * ((E + 31) / 32) > 256;
  const dim3 grid(static_cast<unsigned>(rows), static_cast<unsigned>(wide ? (E + 63) / 64 : (E + 31) / 32));
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (wide) router_tile_kernel<4><<<grid, 64 * RW, 0, s>>>(static_cast<const bf16_t*>(h), router, logits, static_cast<int>(T), K, E);
  else router_tile_kernel<2><<<grid, 64 * RW, 0, s>>>(static_cast<const bf16_t*>(h), router, logits, static_cast<int>(T), K, E);
  return after_launch("router_tiles");
}
