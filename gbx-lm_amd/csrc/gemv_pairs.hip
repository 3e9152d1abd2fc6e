// Rows of experts for a few (token, slot) pairs (gbx_gather_qlinear_forward, gbx_gather_swiglu_forward): y[p, n] = sum_k x[p / div, k] (s q + z) of expert
// idx[p], and silu(gate) * up of two such matrices.  Same arithmetic as gemv_impl.h (fields as fp16 subnormals against pre-shifted activations, fp32 sums).
//
// What bounds it: one trip to memory behind another -- arguments, expert, rows, the store -- for 1 to 10 MB of weights in all.  The decode GEMV spends as long again
// on its activations, which a workgroup converts through LDS for the eight rows it then reads.  Here a lane reads its slot's 32 or 64 activations and forms
// their image in registers while the rows are on their way: no LDS, no barrier.  Rows of up to 32 slots lie two to a wave.  All of a wave's rows are asked for at once.
// Rows that take more than one slot a lane stay with gemv_impl.h.
// That GEMV | this, us, 8 pairs of 128 experts, bf16, weights from memory: gate and up of 768 x 2048 at 3 bits 6.5 | 5.0, down 8.5 | 3.9; 4 bits 5.9 | 5.1 and
// 7.6 | 4.0; 2 bits 7.6 | 5.6 and 10.0 | 4.4; 64 pairs at 3 bits 30.9 | 17.9 (3.6 TB/s) and 44.3 | 13.8; 6 pairs of 32, 1408 x 2048 at 4 bits 7.3 | 6.6 and 6.3 | 4.5.
#include "gbx_device.h"
#include "gemv_fmt.h"
#include "kernels.h"

namespace gbx {
namespace {

struct PairMatrix {
  const uint32_t* w;              // [E, N, K*bits/32]
  const unsigned short* scales;   // [E, N, K/g]
  const unsigned short* zeros;
};
struct PairArgs {
  const unsigned short* x;        // [pairs / div, K]
  PairMatrix m[2];                // SWIGLU: gate, up
  const int* idx;
  const unsigned short* bias;     // [E, N] or null
  unsigned short* y;              // [pairs, N]
  int N, K, log2g, div, E;
  // pair_mix_kernel: y [pairs / top, N] = residual + the sum of a token's slots by their weights
  const unsigned short *mix, *residual;
  int top;
};

// LPR: lanes a row.  B: batches of a wave from row `first` on, two accumulators each: a gate and an up row, or two plain rows.  The totals: with LPR 64 in every
// lane, with LPR 32 those of a half's row in its last lane.
template <int BITS, bool BF16, bool SPLIT, int LPR, bool SWIGLU, int B>
__device__ __forceinline__ void pair_totals(const PairArgs& a, int p, int e, int first, float (&t)[B][2]) {
  using F = Fmt<BITS>;
  using WT = typename SlotWords<BITS>::type;
  constexpr int NSUB = F::NSUB, PAIRS = F::VPL / 2, UP = F::UNIT_PAIRS, UPSUB = 32 / F::UNIT_VALS, NG = SPLIT ? 2 : 1;
  constexpr int RW = 64 / LPR, STEP = SWIGLU ? RW : 2 * RW;             // rows of y a batch
  const int lane = threadIdx.x & 63, N = a.N, K = a.K, nslots = K / F::VPL;
  const int half = lane / LPR, sub = lane % LPR, slot = min(sub, nslots - 1);
  const u32x4* xs4 = reinterpret_cast<const u32x4*>(a.x + static_cast<size_t>(p / a.div) * K + slot * F::VPL);
  u32x4 xr[F::VPL / 8];
#pragma unroll
  for (int i = 0; i < F::VPL / 8; ++i) xr[i] = xs4[i];
  const int W = K / 32 * BITS, G = K >> a.log2g;
  const int64_t ew = static_cast<int64_t>(e) * N * W, eg = static_cast<int64_t>(e) * N * G;
  const int gat = (slot * NSUB) >> (a.log2g - 5);
  WT w[B][2];
  unsigned short sc[B][2][NG], ze[B][2][NG];
  auto rsrc = [](const void* ptr) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(ptr), 0, 0x7FFFFFFF, 0x00020000); };
#pragma unroll
  for (int b = 0; b < B; ++b)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const PairMatrix& m = a.m[SWIGLU ? i : 0];
      const __amdgpu_buffer_rsrc_t wd = rsrc(m.w + ew), sd = rsrc(m.scales + eg), zd = rsrc(m.zeros + eg);
      const int row = min(first + b * STEP + half + (SWIGLU ? 0 : i * RW), N - 1);
      const int at = (row * W + slot * F::SLOT_WORDS) * 4, ga = (row * G + gat) * 2;
      if constexpr (BITS == 3) w[b][i] = __builtin_amdgcn_raw_buffer_load_b96(wd, at, 0, 2);      // nt
      else w[b][i] = __builtin_amdgcn_raw_buffer_load_b128(wd, at, 0, 2);
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        sc[b][i][g] = __builtin_amdgcn_raw_buffer_load_b16(sd, ga + 2 * g, 0, 0);
        ze[b][i][g] = __builtin_amdgcn_raw_buffer_load_b16(zd, ga + 2 * g, 0, 0);
      }
    }
  // the activations' image, one block exponent per 32 values (see gemv_impl.h); lanes past the row hold zeros
  const bool live = sub < nslots;
  h2 xv[PAIRS];
  float xsum[NSUB], cf[NSUB];
#pragma unroll
  for (int s = 0; s < NSUB; ++s) {
    float v[32];
    unsigned amax = 0;
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const unsigned u = live ? xr[s * 4 + i / 4][i % 4] : 0u;
      v[2 * i] = act_lo<BF16>(u);
      v[2 * i + 1] = act_hi<BF16>(u);
      amax = max(amax, max(__float_as_uint(v[2 * i]) & 0x7FFFFFFFu, __float_as_uint(v[2 * i + 1]) & 0x7FFFFFFFu));
      sum += v[2 * i] + v[2 * i + 1];
    }
    const int E = min(max(141 - static_cast<int>(amax >> 23), -100), 110);      // the largest |x| lands in [2^14, 2^15)
#pragma unroll
    for (int u = 0; u < UPSUB; ++u)
#pragma unroll
      for (int i = 0; i < UP; ++i) {
        const float m = exp2i(E - F::pos(i));
        h2 t;
        t.x = static_cast<_Float16>(v[u * F::UNIT_VALS + F::ka(i)] * m);
        t.y = static_cast<_Float16>(v[u * F::UNIT_VALS + F::kb(i)] * m);
        xv[(s * UPSUB + u) * UP + i] = t;
      }
    xsum[s] = sum;
    cf[s] = exp2i(24 - E);
  }
#pragma unroll
  for (int b = 0; b < B; ++b) {
    float acc[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      float d[NSUB];
      dot_slot<BITS>(w[b][i], xv, d);
      acc[i] = 0.f;
      if constexpr (NSUB == 2 && !SPLIT) {
        acc[i] = act_to_f32<BF16>(sc[b][i][0]) * fmaf(cf[1], d[1], cf[0] * d[0]);
        acc[i] = fmaf(act_to_f32<BF16>(ze[b][i][0]), xsum[0] + xsum[1], acc[i]);
      } else {
#pragma unroll
        for (int s = 0; s < NSUB; ++s) {
          acc[i] = fmaf(act_to_f32<BF16>(sc[b][i][s]) * cf[s], d[s], acc[i]);
          acc[i] = fmaf(act_to_f32<BF16>(ze[b][i][s]), xsum[s], acc[i]);
        }
      }
    }
    if constexpr (LPR == 64) {
      const float tot = wave_sum2(acc[0], acc[1]);
      t[b][0] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(tot), 31));
      t[b][1] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(tot), 63));
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        float v = acc[i];
        v += dpp_f32<0xB1>(v);
        v += dpp_f32<0x4E>(v);
        v += dpp_f32<0x141>(v);
        v += dpp_f32<0x140>(v);
        t[b][i] = v + dpp_f32<0x142, 0xA>(v);
      }
    }
  }
}

__device__ __forceinline__ int expert_of(const PairArgs& a, int p) { return min(max(a.idx[p], 0), a.E - 1); }      // (a bad index cannot leave the tensors)

template <int BITS, bool BF16, bool SPLIT, int LPR, bool SWIGLU, int B>
__global__ __launch_bounds__(256) void pair_rows_kernel(const PairArgs a) {
  constexpr int RW = 64 / LPR, STEP = SWIGLU ? RW : 2 * RW;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), p = blockIdx.y, e = expert_of(a, p), N = a.N;
  const int first = (blockIdx.x * 4 + wave) * B * STEP;                 // the wave's rows are neighbours
  float t[B][2];
  pair_totals<BITS, BF16, SPLIT, LPR, SWIGLU, B>(a, p, e, first, t);
  if (lane % LPR != LPR - 1) return;
  unsigned short* y = a.y + static_cast<size_t>(p) * N;
#pragma unroll
  for (int b = 0; b < B; ++b) {
    const int row = first + b * STEP + lane / LPR;
    if constexpr (SWIGLU) {                                             // every step rounded, as the three operations do
      const float g = round_bf16_or_f16(t[b][0], BF16), u = round_bf16_or_f16(t[b][1], BF16);
      const float sl = round_bf16_or_f16(g / (1.f + __expf(-g)), BF16);
      if (row < N) y[row] = f32_to_act<BF16>(sl * u);
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int r = row + i * RW;
        if (r < N) {
          unsigned short v = f32_to_act<BF16>(t[b][i]);
          if (a.bias) v = f32_to_act<BF16>(act_to_f32<BF16>(v) + act_to_f32<BF16>(a.bias[static_cast<int64_t>(e) * N + r]));
          y[r] = v;
        }
      }
    }
  }
}

// The last products of a token's up to eight experts with their weighted sum and the block's residual, every step rounded as moe_combine_kernel does: a wave a slot, the
// same few rows in each, which meet in LDS.  A launch less in a chain of launches that take one trip to memory each.  Two launches | this, us, 8 slots of 128
// experts, 2048 x 768 at 3 bits, 1 token 7.5 | 4.1, 8 tokens 17.0 | 15.0.
constexpr int MIX_ROWS = 8;
template <int BITS, bool BF16, bool SPLIT, int LPR>
__global__ __launch_bounds__(512) void pair_mix_kernel(const PairArgs a) {
  constexpr int RW = 64 / LPR, B = MIX_ROWS / (2 * RW);
  __shared__ float part[8][MIX_ROWS];
  const int lane = threadIdx.x & 63, slot = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), N = a.N, first = blockIdx.x * MIX_ROWS;
  const int64_t token = blockIdx.y;
  const int row = first + min(static_cast<int>(threadIdx.x), MIX_ROWS - 1);
  const float res = a.residual && threadIdx.x < MIX_ROWS ? act_to_f32<BF16>(a.residual[token * N + min(row, N - 1)]) : 0.f;
  if (slot < a.top) {
    const int p = blockIdx.y * a.top + slot;
    const float w = act_to_f32<BF16>(a.mix[p]);
    float t[B][2];
    pair_totals<BITS, BF16, SPLIT, LPR, false, B>(a, p, expert_of(a, p), first, t);
    if (lane % LPR == LPR - 1) {
#pragma unroll
      for (int b = 0; b < B; ++b)
#pragma unroll
        for (int i = 0; i < 2; ++i) part[slot][(b * 2 + i) * RW + lane / LPR] = round_bf16_or_f16(w * round_bf16_or_f16(t[b][i], BF16), BF16);
    }
  }
  __syncthreads();
  if (threadIdx.x >= MIX_ROWS || row >= N) return;
  float v = 0.f;
  for (int s = 0; s < a.top; ++s) v += part[s][threadIdx.x];
  if (a.residual) v = res + round_bf16_or_f16(v, BF16);
  a.y[token * N + row] = f32_to_act<BF16>(v);
}

template <int BITS, bool BF16, bool SPLIT, int LPR, bool SWIGLU>
void launch_pairs(const PairArgs& a, int pairs, hipStream_t s) {
  constexpr int STEP = (SWIGLU ? 1 : 2) * (64 / LPR);
  const int batches = (a.N + STEP - 1) / STEP;
  // Batches of a wave: what a lane does to its activations is shared by them, but a few thousand waves are wanted.  1 | 2 | 4, us: 6144 batches of 2048 at 3 bits 5.8 |
  // 5.0 | 5.4, 4096 of 768 4.3 | 3.9 | 4.8; 49 152 of 2048 27.5 | 20.5 | 17.9; 2 bits (64 activations a lane) 3072 of 2048 6.5 | 6.4 | 5.6, 4096 of 768 5.8 | 4.7 | 4.4.
  const bool four = BITS == 2 || static_cast<int64_t>(batches) * pairs >= 16384;
  const int B = four ? 4 : 2;
  const dim3 grid((batches + 4 * B - 1) / (4 * B), pairs);
  if (four) hipLaunchKernelGGL((pair_rows_kernel<BITS, BF16, SPLIT, LPR, SWIGLU, 4>), grid, dim3(256), 0, s, a);
  else if constexpr (BITS != 2) hipLaunchKernelGGL((pair_rows_kernel<BITS, BF16, SPLIT, LPR, SWIGLU, 2>), grid, dim3(256), 0, s, a);
}
template <int BITS, bool BF16, bool SPLIT>
void launch_pairs_rows(const PairArgs& a, int pairs, bool swiglu, hipStream_t s) {
  const bool two = a.K / Fmt<BITS>::VPL <= 32;
  if (a.mix) {
    const dim3 grid((a.N + MIX_ROWS - 1) / MIX_ROWS, pairs / a.top);
    if (two) hipLaunchKernelGGL((pair_mix_kernel<BITS, BF16, SPLIT, 32>), grid, dim3(512), 0, s, a);
    else hipLaunchKernelGGL((pair_mix_kernel<BITS, BF16, SPLIT, 64>), grid, dim3(512), 0, s, a);
    return;
  }
  if (swiglu) two ? launch_pairs<BITS, BF16, SPLIT, 32, true>(a, pairs, s) : launch_pairs<BITS, BF16, SPLIT, 64, true>(a, pairs, s);
  else two ? launch_pairs<BITS, BF16, SPLIT, 32, false>(a, pairs, s) : launch_pairs<BITS, BF16, SPLIT, 64, false>(a, pairs, s);
}
template <int BITS>
void launch_pairs_bits(const PairArgs& a, int pairs, bool swiglu, bool bf16, hipStream_t s) {
  if constexpr (BITS == 2) {
    if (a.log2g == 5) return bf16 ? launch_pairs_rows<2, true, true>(a, pairs, swiglu, s) : launch_pairs_rows<2, false, true>(a, pairs, swiglu, s);
  }
  bf16 ? launch_pairs_rows<BITS, true, false>(a, pairs, swiglu, s) : launch_pairs_rows<BITS, false, false>(a, pairs, swiglu, s);
}

}  // namespace

bool gemv_pairs_takes(int N, int K, int bits) {
  return K / (bits == 2 ? 64 : 32) <= 64 && static_cast<int64_t>(N) * (K / 32 * bits) * 4 <= INT32_MAX;      // (one slot a lane; 32-bit offsets in an expert)
}

static hipError_t launch_pairs_args(const PairArgs& a, int pairs, int bits, bool swiglu, bool bf16, hipStream_t s) {
  if (bits == 2) launch_pairs_bits<2>(a, pairs, swiglu, bf16, s);
  else if (bits == 3) launch_pairs_bits<3>(a, pairs, swiglu, bf16, s);
  else launch_pairs_bits<4>(a, pairs, swiglu, bf16, s);
  return hipGetLastError();
}

hipError_t launch_gemv_pairs(const void* x, const uint32_t* const* w, const void* const* scales, const void* const* zeros, int matrices, const void* bias,
                             const int32_t* idx, void* y, int pairs, int x_div, int E, int N, int K, int bits, int log2g, bool bf16, hipStream_t s) {
  PairArgs a{};
  a.x = static_cast<const unsigned short*>(x);
  for (int i = 0; i < matrices; ++i) a.m[i] = PairMatrix{w[i], static_cast<const unsigned short*>(scales[i]), static_cast<const unsigned short*>(zeros[i])};
  a.idx = idx;
  a.bias = static_cast<const unsigned short*>(bias);
  a.y = static_cast<unsigned short*>(y);
  a.N = N; a.K = K; a.log2g = log2g; a.div = x_div; a.E = E;
  return launch_pairs_args(a, pairs, bits, matrices == 2, bf16, s);
}

}  // namespace gbx

// y[t] = residual[t] (or nothing) + sum_s mix[t, s] * (expert idx[t, s] of the stacked [E, N, ...] matrices times x[t, s]), rounded like the product, the elementwise
// multiply, the sum and the add.  For this package's own Python layer; not part of the public header.  Non-zero: the caller runs the steps (nothing was launched).
extern "C" int gbx_gather_mix_forward(const void* x, const uint32_t* qweight, const void* scales, const void* zeros, const int32_t* indices, const void* mix,
                                      const void* residual, void* y, int32_t tokens, int32_t top, int32_t num_experts, int32_t N, int32_t K, int32_t bits,
                                      int32_t group_size, int32_t bf16, void* hip_stream) {
  const auto off = [](const void* p, unsigned n) { return reinterpret_cast<uintptr_t>(p) % n != 0; };
  if (!x || !qweight || !scales || !zeros || !indices || !mix || !y || tokens < 1 || tokens > 65535 || top < 1 || top > 8 || num_experts < 1 || N < 1) return 1;
  if (bits < 2 || bits > 4 || (group_size != 32 && group_size != 64 && group_size != 128) || K < 128 || K % 128 || !gbx::gemv_pairs_takes(N, K, bits)) return 1;
  if (off(x, 16) || off(qweight, 16) || (static_cast<int64_t>(N) * (K / 32 * bits) * 4) % 16) return 1;
  gbx::PairArgs a{};
  a.x = static_cast<const unsigned short*>(x);
  a.m[0] = gbx::PairMatrix{qweight, static_cast<const unsigned short*>(scales), static_cast<const unsigned short*>(zeros)};
  a.idx = indices;
  a.mix = static_cast<const unsigned short*>(mix);
  a.residual = static_cast<const unsigned short*>(residual);
  a.y = static_cast<unsigned short*>(y);
  a.N = N; a.K = K; a.log2g = group_size == 32 ? 5 : group_size == 64 ? 6 : 7; a.div = 1; a.E = num_experts; a.top = top;
  return gbx::launch_pairs_args(a, tokens * top, bits, false, bf16 != 0, static_cast<hipStream_t>(hip_stream)) == hipSuccess ? 0 : 2;
}
