// Device helpers shared by the translation units of libgbx_mixers.so.
#pragma once
#include <hip/hip_runtime.h>
#include <atomic>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
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

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
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

// The same over a workgroup of blockDim.x threads (whole waves, at most 16 of them); `red` is 16 floats of LDS that no earlier call used.
__device__ __forceinline__ float row_sum(float v, float* red) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float s = 0.f;
  for (int i = 0; i < static_cast<int>(blockDim.x >> 6); ++i) s += red[i];
  return s;
}

// Row kernels that give every thread one group of four neighbouring channels (rows of up to 4 * 1024): every operand of a row is in flight
// at once, where a loop over channels whose stores may alias its loads pays a trip to memory per pass.  Threads of a workgroup for `width`
// channels; 0: the row is too wide or not in groups of four.
inline int row_threads(int width) { return width % 4 == 0 && width <= 4096 ? (width / 4 + 63) / 64 * 64 : 0; }
template <typename... P>
inline bool all_aligned(size_t bytes, const P*... p) { return ((reinterpret_cast<uintptr_t>(p) | ...) & (bytes - 1)) == 0; }

// Candidates in front of candidate e of value x among 4 n4 values: larger ones, and equal ones of a lower index.  Every candidate's rank is
// taken at once, where rounds of arg-max wait for one another.
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
// Where a router's choice goes by rank: every expert reads all scores, E / 16 steps of a wave, where each of the `rounds` of arg-max (one per choice and per
// kept group) is a chain of its own; `per_round` steps cost what one of them does.  Measured, rounds | rank, us: softmax, top 8, 1 row: 64 experts
// 9.7 | 5.2, 128 9.6 | 8.1, 256 9.5 | 14.1, 512 10.3 | 49; 4000 rows: 64 29.6 | 11.5, 128 30.0 | 20.8, 256 30.6 | 47; top 2, 1 row: 64 4.1 | 5.2.
// Sigmoid, top 8, 1 row: 64 6.8 | 5.1, 128 7.4 | 7.9, 256 8.6 | 14.1; in 8 groups of which 4 stay 64 10.4 | 5.9, 128 11.9 | 9.0, 256 14.9 | 15.6, 4000 rows
// 64 15.4 | 8.1, 128 17.0 | 17.5, 160 18.1 | 29.4; top 2 in groups 64 6.5 | 5.9, 96 7.2 | 7.5.
constexpr int RANK_EXPERTS = 256;
inline bool choice_by_rank(int E, int rounds, int per_round) { return E <= RANK_EXPERTS && E <= per_round * rounds; }
constexpr int RANK_PER_SOFTMAX_ROUND = 16, RANK_PER_SIGMOID_ROUND = 11;

// z = a row of a sublayer's output, or sum_k mix[k] (candidate row k), at channels c .. c + 3; eight candidates in flight at a time.
template <typename T>
__device__ __forceinline__ void candidate_sum(const T* __restrict__ y, const float* __restrict__ mix, int top, int width, int c, float* z) {
  if (!mix) { Lanes<T, 4>::load(y + c, z); return; }
#pragma unroll
  for (int i = 0; i < 4; ++i) z[i] = 0.f;
  for (int k0 = 0; k0 < top; k0 += 8) {
    float u[8][4];
#pragma unroll
    for (int k = 0; k < 8; ++k) Lanes<T, 4>::load(y + static_cast<int64_t>(min(k0 + k, top - 1)) * width + c, u[k]);
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (k0 + k < top) {
        const float m = mix[k0 + k];
#pragma unroll
        for (int i = 0; i < 4; ++i) z[i] += m * u[k][i];
      }
  }
}

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
