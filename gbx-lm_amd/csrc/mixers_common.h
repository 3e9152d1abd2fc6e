// Device helpers shared by the translation units of libgbx_mixers.so.
#pragma once
#include <hip/hip_runtime.h>
#include <atomic>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <type_traits>
#include "gbx_mixers.h"

namespace gbxm {

typedef unsigned short bf16_t;          // storage type of a bf16 element

__device__ __forceinline__ float to_f32(float v) { return v; }
__device__ __forceinline__ float to_f32(bf16_t v) { return __uint_as_float(static_cast<unsigned>(v) << 16); }
// round to nearest even (values here are finite)
__device__ __forceinline__ bf16_t f32_to_bf16(float f) {
  const unsigned u = __float_as_uint(f);
  return static_cast<bf16_t>((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}
template <typename T> __device__ __forceinline__ T from_f32(float f);
template <> __device__ __forceinline__ float from_f32<float>(float f) { return f; }
template <> __device__ __forceinline__ bf16_t from_f32<bf16_t>(float f) { return f32_to_bf16(f); }

// V neighbouring elements of a row to and from fp32: one 8- or 16-byte access for V = 4 (aligned addresses).
template <typename T, int V> struct Lanes;
template <typename T> struct Lanes<T, 1> {
  static __device__ __forceinline__ void load(const T* p, float* v) { v[0] = to_f32(*p); }
  static __device__ __forceinline__ void store(T* p, const float* v) { *p = from_f32<T>(v[0]); }
};
template <> struct Lanes<float, 2> {
  static __device__ __forceinline__ void load(const float* p, float* v) {
    const float2 f = *reinterpret_cast<const float2*>(p);
    v[0] = f.x; v[1] = f.y;
  }
};
template <> struct Lanes<float, 4> {
  static __device__ __forceinline__ void load(const float* p, float* v) {
    const float4 f = *reinterpret_cast<const float4*>(p);
    v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
  }
  static __device__ __forceinline__ void store(float* p, const float* v) { *reinterpret_cast<float4*>(p) = float4{v[0], v[1], v[2], v[3]}; }
};
template <> struct Lanes<bf16_t, 4> {
  static __device__ __forceinline__ void load(const bf16_t* p, float* v) {
    const uint2 u = *reinterpret_cast<const uint2*>(p);
    v[0] = __uint_as_float(u.x << 16); v[1] = __uint_as_float(u.x & 0xFFFF0000u);
    v[2] = __uint_as_float(u.y << 16); v[3] = __uint_as_float(u.y & 0xFFFF0000u);
  }
  static __device__ __forceinline__ void store(bf16_t* p, const float* v) {
    *reinterpret_cast<uint2*>(p) = uint2{static_cast<unsigned>(f32_to_bf16(v[0])) | (static_cast<unsigned>(f32_to_bf16(v[1])) << 16),
                                         static_cast<unsigned>(f32_to_bf16(v[2])) | (static_cast<unsigned>(f32_to_bf16(v[3])) << 16)};
  }
};

// One step of a sum over a wave, every lane: v of this lane plus that of the lane 2^k away.  Register moves: a trip through LDS (__shfl_xor) is what a row kernel
// of a decode step waits for otherwise (by __shfl_xor | this, the same bits, us a token: 1 row of 4 streams x 1024 over 4 layers 197.5 | 192.0, 2 rows of 2048 over 4
// 332.6 | 329.6).  FROM 32, 16: halves and rows of 16 trade places; 8: any values; 4: values that step 8 has made alike.
template <int FROM> __device__ __forceinline__ float lanes_apart_sum(float v) {
  if constexpr (FROM >= 16) {
    const unsigned b = __float_as_uint(v);
    if constexpr (FROM == 32) {
      const auto r = __builtin_amdgcn_permlane32_swap(b, b, false, false);
      return __uint_as_float(r[0]) + __uint_as_float(r[1]);
    } else {
      const auto r = __builtin_amdgcn_permlane16_swap(b, b, false, false);
      return __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
  } else {
    constexpr int MOVE = FROM == 8 ? 0x128 : FROM == 4 ? 0x124 : FROM == 2 ? 0x4E : 0xB1;       // row_ror:8, row_ror:4, quad_perm [2,3,0,1], [1,0,3,2]
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), MOVE, 0xf, 0xf, false));
  }
}
// The sum of a wave's values, the same bits in every lane: halves first, neighbours last.
__device__ __forceinline__ float wave_sum(float v) {
  v = lanes_apart_sum<16>(lanes_apart_sum<32>(v));
  v = lanes_apart_sum<4>(lanes_apart_sum<8>(v));
  return lanes_apart_sum<1>(lanes_apart_sum<2>(v));
}
// The same over aligned groups of `lanes` (a power of two, the same for a whole wave), neighbours first.
__device__ __forceinline__ float group_sum(float v, int lanes) {
  const auto plus = [&](auto move) { v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), decltype(move)::value, 0xf, 0xf, false)); };
  if (lanes > 1) plus(std::integral_constant<int, 0xB1>{});          // quad_perm [1,0,3,2]
  if (lanes > 2) plus(std::integral_constant<int, 0x4E>{});          // quad_perm [2,3,0,1]
  if (lanes > 4) plus(std::integral_constant<int, 0x141>{});         // row_half_mirror
  if (lanes > 8) plus(std::integral_constant<int, 0x140>{});         // row_mirror
  if (lanes > 16) v = lanes_apart_sum<16>(v);
  if (lanes > 32) v = lanes_apart_sum<32>(v);
  return v;
}
// Sum over the 16 lanes of a row; every lane of the row gets the same bits (each step adds the two halves of a mirrored pair).
__device__ __forceinline__ float row16_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, false));    // quad_perm [1,0,3,2]
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, false));    // quad_perm [2,3,0,1]
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, false));   // row_half_mirror
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xf, 0xf, false));   // row_mirror
  return v;
}

// sum over a workgroup of NW waves; every thread gets the result; `red` is NW floats of LDS.  Fixed order: deterministic.
template <int NW>
__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  __syncthreads();                       // red may still be read from an earlier call
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < NW; ++i) s += red[i];
  return s;
}

// The same over the workgroup of a row of `width` channels (row_threads); `red` is 16 floats of LDS that no earlier call used.
__device__ __forceinline__ float row_sum(float v, float* red, int width) {
  const int waves = (width / 4 + 63) >> 6;
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 16; i += 4)                  // (four at a time: a loop waits for LDS once a wave)
    if (i < waves) {
      const float r[4] = {red[i], red[i + 1], red[i + 2], red[i + 3]};
      s += r[0];
#pragma unroll
      for (int k = 1; k < 4; ++k)
        if (i + k < waves) s += r[k];
    }
  return s;
}

// Row kernels that give every thread one group of four neighbouring channels (rows of up to 4 * 1024): every operand of a row is in flight
// at once, where a loop over channels whose stores may alias its loads pays a trip to memory per pass.  Threads of a workgroup for `width`
// channels; 0: the row is too wide or not in groups of four.
inline int row_threads(int width) { return width % 4 == 0 && width <= 4096 ? (width / 4 + 63) / 64 * 64 : 0; }
template <typename... P>
inline bool all_aligned(size_t bytes, const P*... p) { return ((reinterpret_cast<uintptr_t>(p) | ...) & (bytes - 1)) == 0; }

// Candidates in front of candidate e of value x among 4 n4 values: larger ones, and equal ones of a lower index.
__device__ __forceinline__ int rank_of(const float* v, int n4, int e, float x) {
  int rank = 0;
#pragma unroll 8
  for (int j = 0; j < n4; ++j) {
    const float4 u = *reinterpret_cast<const float4*>(v + 4 * j);
    const float w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) rank += (w[k] > x || (w[k] == x && 4 * j + k < e)) ? 1 : 0;
  }
  return rank;
}

// The largest of a wave's values, the same in every lane: within rows of 16 lanes by DPP, then the four rows' by scalar reads (a number beside
// values that are none).
template <typename T, typename Max> __device__ __forceinline__ T wave_most(T x, Max most) {
  const auto moved = [&](auto dpp) { return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(dpp)::value, 0xf, 0xf, false)); };
  x = most(x, moved(std::integral_constant<int, 0xB1>{}));           // quad_perm [1,0,3,2]
  x = most(x, moved(std::integral_constant<int, 0x4E>{}));           // quad_perm [2,3,0,1]
  x = most(x, moved(std::integral_constant<int, 0x141>{}));          // row_half_mirror
  x = most(x, moved(std::integral_constant<int, 0x140>{}));          // row_mirror
  const auto row = [&](int lane) { return __builtin_bit_cast(T, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), lane)); };
  return most(most(row(0), row(16)), most(row(32), row(48)));
}
__device__ __forceinline__ float wave_max(float x) { return wave_most(x, [](float a, float b) { return fmaxf(a, b); }); }

// Floats (numbers and infinities) as unsigned keys of the same order; 0 lies below all of them.
__device__ __forceinline__ unsigned order_key(float x) {
  const unsigned b = __float_as_uint(x + 0.f);                       // (-0 is 0)
  return b ^ (b >> 31 ? 0xFFFFFFFFu : 0x80000000u);
}
__device__ __forceinline__ float key_value(unsigned k) { return __uint_as_float(k ^ (k >> 31 ? 0x80000000u : 0xFFFFFFFFu)); }

// Rounds of arg-max over up to 64 PER candidates that one wave holds, candidate 64 i + lane in key[i] (0: none, or taken), of equal ones the
// lowest first: take(round, candidate, its key), all uniform.  A round is some 40 instructions without a barrier or a trip to LDS.
template <int PER, typename Take> __device__ __forceinline__ void wave_choose(unsigned (&key)[PER], int rounds, Take take) {
  const int lane = threadIdx.x & 63;
  for (int k = 0; k < rounds; ++k) {
    unsigned m = key[0];
#pragma unroll
    for (int i = 1; i < PER; ++i) m = max(m, key[i]);
    m = wave_most(m, [](unsigned a, unsigned b) { return max(a, b); });
    int e = 0;
#pragma unroll
    for (int i = PER - 1; i >= 0; --i) {
      const unsigned long long here = __builtin_amdgcn_ballot_w64(key[i] == m);
      if (here) e = 64 * i + __builtin_ctzll(here);
    }
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (64 * i + lane == e) key[i] = 0;
    take(k, e, m);
  }
}
// Which form a router's choice takes: rounds of a wave, or by rank, where every expert counts those in front of it in LDS, whatever their number.  The line is each
// kernel's own (`most` choices; the softmax kernel's ranks cost more: it takes probabilities in 256 threads), a row's form does not depend on the other rows.  Rank | wave, us,
// 1 row / 3 481 rows.  Softmax: 8 of 16 3.4 | 2.8 / 6.6 | 4.1, 16 of 16 3.5 | 3.5 / 6.7 | 5.4; 28 of 32 4.4 | 4.6 / 8.6 | 7.4; 8 of 64 5.6 | 2.8 / 11.4 | 4.1, 36 of 64 5.9 | 5.3 / 11.8 |
// 8.6, 52 of 64 6.0 | 6.8 / 12.0 | 11.2, 64 of 64 5.9 | 7.9 / 11.8 | 13.2; 8 of 128 8.5 | 3.1 / 19.8 | 4.7, 64 of 128 9.0 | 9.8 / 20.2 | 15.9; 64 of 256 15.1 | 13.2 / 43.5 | 21.6.
// Sigmoid: 12 of 16 2.9 | 3.3 / 4.2 | 4.6; 12 of 32 3.7 | 3.3 / 5.0 | 4.6, 20 of 32 3.7 | 4.1 / 5.1 | 6.0; 28 of 64 5.2 | 5.0 / 7.1 | 7.3, 36 of 64 5.3 | 5.9 / 7.2 | 8.7; 36 of 128 8.3 | 6.8 /
// 16.0 | 10.3, 52 of 128 8.4 | 9.0 / 16.3 | 13.6; 64 of 256 14.6 | 13.8 / 42.9 | 21.2; softmax over the logits' order: 28 of 64 5.3 | 4.7 / 7.3 | 7.2, 36 of 64 5.4 | 5.4 / 7.3 | 8.5, 52 of 128
// 8.6 | 8.3 / 16.4 | 13.1.  Sigmoid, groups kept of all + choices of experts: 4 of 8 + 8 of 128 9.0 | 3.8 / 17.4 | 6.0, 32 of 64 + 8 of 128 11.5 | 6.0 / 22.8 | 9.3, 16 of 32 + 16 of 64
// 7.0 | 5.2 / 9.5 | 8.0, 40 of 64 + 40 of 64 8.5 | 9.7 / 11.8 | 15.6.  A lane holds a choice and a group: 64 of either at most.
constexpr int most_of_softmax(int E) { return 6 + 5 * E / 8; }
constexpr int most_of_logits(int E) { return 4 + 3 * E / 8; }
inline bool choice_by_wave(int E, int top, int most, int groups = 0, int keep = 0) {
  return E <= 256 && top <= 64 && groups <= 64 && top <= most && (groups == 0 || top + keep <= 16 + E / 2);
}
// Beyond that few choices with many groups remain, whose rounds of arg-max (per choice and kept group) a workgroup makes in about the time of 11 experts' ranks.
constexpr int RANK_EXPERTS = 256;
inline bool choice_by_rank(int E, int rounds) { return E <= RANK_EXPERTS && E <= 11 * rounds; }
// a wave per row: one a workgroup while rows are few
inline unsigned choice_threads(int64_t rows) { return rows > 1024 ? 256 : 64; }
inline unsigned choice_blocks(int64_t rows) { return static_cast<unsigned>(rows > 1024 ? (rows + 3) / 4 : rows); }

// Four neighbouring elements as they lie in memory, so that a load in a branch does not wait there for its own conversion.
template <typename T> struct Raw4;
template <> struct Raw4<float> {
  float4 r;
  __device__ __forceinline__ void load(const float* p) { r = *reinterpret_cast<const float4*>(p); }
  __device__ __forceinline__ void get(float* v) const { v[0] = r.x; v[1] = r.y; v[2] = r.z; v[3] = r.w; }
};
template <> struct Raw4<bf16_t> {
  uint2 r;
  __device__ __forceinline__ void load(const bf16_t* p) { r = *reinterpret_cast<const uint2*>(p); }
  __device__ __forceinline__ void get(float* v) const {
    v[0] = __uint_as_float(r.x << 16); v[1] = __uint_as_float(r.x & 0xFFFF0000u);
    v[2] = __uint_as_float(r.y << 16); v[3] = __uint_as_float(r.y & 0xFFFF0000u);
  }
};
// Numbers that are the same for a whole wave, here and now: left to itself the compiler asks for each where it is first used, behind the trip of the rows.
__device__ __forceinline__ void at_hand(float& x) { asm volatile("" : "+v"(x)); }
template <typename P> __device__ __forceinline__ void at_hand(P* p) { asm volatile("" ::"s"(p)); }
template <typename P, typename... Q> __device__ __forceinline__ void at_hand(P* p, Q*... q) { at_hand(p); at_hand(q...); }

// z = a row of a sublayer's output, or sum_k mix[k] (candidate row k) (mix null: the sum alone where `sum` says so), at channels c .. c + 3; eight candidates in
// flight at a time, the first ones (FEW: and their weights) from ask() on.
template <typename T, bool FEW = false> struct Candidates {
  Raw4<T> u[8];
  float m[8];
  __device__ __forceinline__ void ask(const T* __restrict__ y, const float* __restrict__ mix, int first, int top, int width, int c) {
#pragma unroll
    for (int k = 0; k < 8; ++k) u[k].load(y + static_cast<int64_t>(min(first + k, top - 1)) * width + c);
#pragma unroll
    for (int k = 0; k < 8; ++k) m[k] = mix ? mix[min(first + k, top - 1)] : 1.f;
  }
  __device__ __forceinline__ void add(int first, int top, float* z) {
    if constexpr (FEW) {
#pragma unroll
      for (int k = 0; k < 8; ++k) at_hand(m[k]);
    }
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (first + k < top) {
        float v[4];
        u[k].get(v);
#pragma unroll
        for (int i = 0; i < 4; ++i) z[i] += m[k] * v[i];
      }
  }
  __device__ __forceinline__ void rest(const T* __restrict__ y, const float* __restrict__ mix, int top, int width, int c, float* z) {
    for (int k0 = 8; k0 < top; k0 += 8) {
      ask(y, mix, k0, top, width, c);
      add(k0, top, z);
    }
  }
};
template <typename T, bool FEW = false> struct Branch : Candidates<T, FEW> {
  using Candidates<T, FEW>::u;
  __device__ __forceinline__ void ask(const T* __restrict__ y, const float* __restrict__ mix, int top, int width, int c) {
    if (mix) Candidates<T, FEW>::ask(y, mix, 0, top, width, c);
    else u[0].load(y + c);
  }
  __device__ __forceinline__ void sum(const T* __restrict__ y, const float* __restrict__ mix, int top, int width, int c, float* z) {
    if (!mix) { u[0].get(z); return; }
#pragma unroll
    for (int i = 0; i < 4; ++i) z[i] = 0.f;
    this->add(0, top, z);
    this->rest(y, mix, top, width, c, z);
  }
};

// Transcendentals: exact library forms for fp32 models, hardware approximations (a few ulp) where activations are bf16.
template <bool FAST> __device__ __forceinline__ float exp_(float x) { if constexpr (FAST) return __expf(x); else return expf(x); }
template <bool FAST> __device__ __forceinline__ float sigmoid_(float x) {
  if constexpr (FAST) return __fdividef(1.f, 1.f + __expf(-x)); else return 1.f / (1.f + expf(-x));
}
template <bool FAST> __device__ __forceinline__ float tanh_(float x) {
  if constexpr (FAST) { const float e = __expf(2.f * x); return 1.f - __fdividef(2.f, e + 1.f); } else return tanhf(x);
}
// Gated activations of feed-forwards (GBXM_GLU_*): silu(g) u, gelu(g) u in the tanh form, sigmoid(g) u, or the clamped form
// g' sigmoid(alpha g') (u' + 1) with g' = min(g, limit), u' = clamp(u, -limit, limit).
template <bool FAST> __device__ __forceinline__ float glu_act(float g, float u, int kind, float limit, float alpha) {
  if (kind == GBXM_GLU_CLAMPED_SWISH) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    return g * sigmoid_<FAST>(alpha * g) * (u + 1.f);
  }
  if (kind == GBXM_GLU_GELU_TANH) return 0.5f * g * (1.f + tanh_<FAST>(0.7978845608028654f * (g + 0.044715f * g * g * g))) * u;
  if (kind == GBXM_GLU_SIGMOID) return sigmoid_<FAST>(g) * u;
  return g * sigmoid_<FAST>(g) * u;
}
template <bool FAST> __device__ __forceinline__ float log1p_(float x) { if constexpr (FAST) return __logf(1.f + x); else return log1pf(x); }

// First position the row at `pos` sees: its chunk's start (chunks of `chunk` tokens counted from position 0), or the window's, or 0.
// Never falls as pos grows.
__host__ __device__ __forceinline__ int first_seen(int pos, int window, int chunk) {
  if (chunk > 0) return pos - pos % chunk;
  return window > 0 && pos >= window ? pos - window + 1 : 0;
}

// floats per (split, row, head) of the key-split partial sums of softmax attention: dv sums padded to a multiple of four (rows stay
// 16-byte aligned), then two more pairs of which the last holds (running maximum, denominator)
__host__ __device__ __forceinline__ int partial_width(int dv) { return (dv + 3) / 4 * 4 + 4; }

// First use of something on each device (a kernel's attributes belong to the device that is current when they are set).
struct OncePerDevice {
  std::atomic<unsigned long long> seen{0};
  unsigned long long bit() const { int d = 0; (void)hipGetDevice(&d); return 1ull << (d & 63); }
  bool pending() const { return (seen.load(std::memory_order_acquire) & bit()) == 0; }
  void done() { seen.fetch_or(bit(), std::memory_order_release); }
};

extern thread_local char g_err[512];
int fail(int code, const char* fmt, ...);
int hip_fail(hipError_t e, const char* what);
inline int after_launch(const char* what) {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? GBXM_OK : hip_fail(e, what);
}

}  // namespace gbxm
