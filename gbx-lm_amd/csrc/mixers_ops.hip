// Row kernels of ragged steps: embedding, segment norms, the branch-norm residual update, the last norm, the router and the
// append to the window rings.  One workgroup per row; statistics in fp32 with a fixed summation order, so a row's result does
// not depend on which other rows share the step.
#include <type_traits>
#include "mixers_common.h"

namespace gbxm {

thread_local char g_err[512] = "";
int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}
int hip_fail(hipError_t e, const char* what) { return fail(GBXM_ERR_HIP, "%s: %s", what, hipGetErrorString(e)); }

namespace {

constexpr int NT = 256, NW = NT / 64;

template <typename T>
__global__ __launch_bounds__(NT) void embed_kernel(const T* __restrict__ table, const int64_t* __restrict__ tokens, float* __restrict__ x,
                                                   T* __restrict__ h, int64_t h_row, int width, float scale, int copies) {
  const int64_t t = blockIdx.x;
  const T* row = table + tokens[t] * width;
  for (int c = threadIdx.x; c < width; c += NT) {
    const float v = to_f32(row[c]) * scale;
    for (int i = 0; i < copies; ++i) x[(t * copies + i) * width + c] = v;
    if (h) h[t * h_row + c] = from_f32<T>(v);
  }
}

// Rows in groups of four neighbouring channels, one a thread (row_threads; T: 8 bytes of bf16, 16 of fp32): all of a row's operands are in flight at once.
// Bound by memory.  A channel a thread and pass | this, us: 3 481 rows of 2048 embedded 12.0 | 10.4, added behind a norm 24.0 | 15.2, the same of eight
// candidates 35.6 | 27.6; segments of 4096 and 512 channels normed 21.6 | 15.9; 8 192 rows normed 26.2 | 18.9; 1 row: 3.1 | 2.6, 4.8 | 2.9, 7.4 | 3.6, 5.9 | 3.4,
// 4.0 | 2.7.
template <typename T>
__global__ __launch_bounds__(1024) void embed_row_kernel(const T* __restrict__ table, const int64_t* __restrict__ tokens, float* __restrict__ x, T* __restrict__ h,
                                                         int64_t h_row, int width, float scale, int copies) {
  const int64_t t = blockIdx.x;
  const int c = threadIdx.x * 4;
  if (c >= width) return;
  float v[4];
  Lanes<T, 4>::load(table + tokens[t] * width + c, v);
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] *= scale;
  for (int i = 0; i < copies; ++i) Lanes<float, 4>::store(x + (t * copies + i) * width + c, v);
  if (h) Lanes<T, 4>::store(h + t * h_row + c, v);
}

// Logits -> log-probabilities: out = x - lse, lse = log sum exp x in fp32, rounded to the row's type before the subtraction.  A workgroup of 16
// waves per row; a row's first 128 KB stay in registers between the three passes (maximum, sum, result), what lies beyond is read again
// from the L2 that the first pass filled.  Rows with an infinite maximum are summed unshifted, so that they come out as the definition has it.
// A few long rows are bound by the vector instructions of the few CUs that hold them (one row of 128 256 bf16 logits: 22 us): slices of a row are
// then workgroups of their own that leave (maximum, sum) in the first of two launches and write their slice in the second.
// Replaces torch's logsumexp and subtraction, some ten launches: 1 x 32 000 fp32 40 -> 5.5 us, 32 x 32 000 fp32 40 -> 8, 1 x 128 256 bf16 62 -> 5.6.
constexpr int LSM_NT = 1024, LSM_VR = 8;

template <typename T> __device__ __forceinline__ float lsm_get(const uint4& v, int j) {
  const unsigned w[4] = {v.x, v.y, v.z, v.w};
  if constexpr (sizeof(T) == 4) return __uint_as_float(w[j]);
  else {
    const unsigned short h = static_cast<unsigned short>(w[j >> 1] >> (16 * (j & 1)));
    if constexpr (std::is_same<T, _Float16>::value) return static_cast<float>(__builtin_bit_cast(_Float16, h));
    else return to_f32(static_cast<bf16_t>(h));
  }
}
// (a plain cast: rounds to nearest even and keeps NaN and infinities)
template <typename T> __device__ __forceinline__ unsigned short lsm_bits(float f) {
  if constexpr (std::is_same<T, _Float16>::value) return __builtin_bit_cast(unsigned short, static_cast<_Float16>(f));
  else return __builtin_bit_cast(unsigned short, static_cast<__bf16>(f));
}
template <typename T> __device__ __forceinline__ float lsm_round(float f) {
  if constexpr (sizeof(T) == 4) return f;
  else {
    const unsigned short h = lsm_bits<T>(f);
    if constexpr (std::is_same<T, _Float16>::value) return static_cast<float>(__builtin_bit_cast(_Float16, h));
    else return to_f32(static_cast<bf16_t>(h));
  }
}

// Few long rows: 8 logits a thread, as many workgroups as that makes, whose (maximum, sum) pairs the second launch puts together.  Slices of 8192 in loads of one
// logit left 19 workgroups with 32 round trips' worth of requests each: 1 x 151 936 bf16 12.4 -> 5.6 us, 8 x 128 256 12.1 -> 6.2, and 1 x 32 000 fp32 7.1 (one workgroup) -> 5.5; 20 000 5.4 in one launch, 5.5 in two.
constexpr int LSM_SLICE = 2048;

// A thread's logits are k + j `step`: neighbours where 16-byte accesses reach them and in 16 bits, whose eight are 16 bytes anyway; 32-bit ones off that grid lie
// beside those of the neighbouring threads (neighbours | beside, us: 1 x 24 577 7.9 | 6.4, 15 x 50 257 10.5 | 7.4, 15 x 151 935 19.4 | 9.3; 1 x 24 577 bf16 6.9 | 7.1).
template <typename T> __device__ __forceinline__ int lsm_step(int vec) { return vec || sizeof(T) == 2 ? 1 : 256; }
template <typename T> __device__ __forceinline__ int lsm_first(int vec) { return blockIdx.x * LSM_SLICE + threadIdx.x * (lsm_step<T>(vec) == 1 ? 8 : 1); }

template <typename T>
__device__ __forceinline__ void lsm_load8(const T* __restrict__ row, int k, int n, int vec, float scale, float* v) {
  if (vec) {                                                  // (n is a multiple of 8: all of them are in the row, or none)
    constexpr int PER = 16 / sizeof(T);
    uint4 u[8 / PER];
#pragma unroll
    for (int i = 0; i < 8 / PER; ++i) u[i] = *reinterpret_cast<const uint4*>(row + min(k, n - 8) + i * PER);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = k < n ? lsm_get<T>(u[j / PER], j % PER) * scale : -INFINITY;
  } else {
    const int step = lsm_step<T>(0);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = k + j * step < n ? static_cast<float>(row[k + j * step]) * scale : -INFINITY;
  }
}

// (maximum, sum of exponentials against it or against 0 where it is infinite) of one slice
template <typename T>
__global__ __launch_bounds__(256) void log_softmax_slice_kernel(const T* __restrict__ x, float2* __restrict__ part, int n, int vec, float scale) {
  __shared__ float top[4], red[4];
  const int k = lsm_first<T>(vec), step = lsm_step<T>(vec);
  float v[8], m = -INFINITY, s = 0.f;
  lsm_load8(x + static_cast<int64_t>(blockIdx.y) * n, k, n, vec, scale, v);
#pragma unroll
  for (int j = 0; j < 8; ++j) m = fmaxf(m, v[j]);
  m = wave_max(m);
  if ((threadIdx.x & 63) == 0) top[threadIdx.x >> 6] = m;
  __syncthreads();
  m = fmaxf(fmaxf(top[0], top[1]), fmaxf(top[2], top[3]));
  const float shift = isinf(m) ? 0.f : m;
#pragma unroll
  for (int j = 0; j < 8; ++j) s += k + j * step < n ? expf(v[j] - shift) : 0.f;
  s = block_sum<4>(s, red);
  if (threadIdx.x == 0) part[blockIdx.y * gridDim.x + blockIdx.x] = float2{m, s};
}

template <typename T, typename O>
__global__ __launch_bounds__(256) void log_softmax_write_kernel(const T* __restrict__ x, const float2* __restrict__ part, O* __restrict__ out, int n, int vec, float scale) {
  __shared__ float top[4], red[4];
  const float2* p = part + blockIdx.y * gridDim.x;
  const int parts = gridDim.x, k = lsm_first<T>(vec);
  const int64_t base = static_cast<int64_t>(blockIdx.y) * n;
  float v[8], m = -INFINITY, s = 0.f;
  lsm_load8(x + base, k, n, vec, scale, v);
  for (int i = threadIdx.x; i < parts; i += 256) m = fmaxf(m, p[i].x);
  m = wave_max(m);
  if ((threadIdx.x & 63) == 0) top[threadIdx.x >> 6] = m;
  __syncthreads();
  m = fmaxf(fmaxf(top[0], top[1]), fmaxf(top[2], top[3]));
  const float shift = isinf(m) ? 0.f : m;
  // (an infinite maximum: the slice's sum is 0, infinite or no number against any shift -- the shift's own exponential may be infinite, and 0 times that is
  // no number)
  for (int i = threadIdx.x; i < parts; i += 256) s += isinf(p[i].x) ? p[i].y : p[i].y * expf(p[i].x - shift);
  const float lse = lsm_round<O>(logf(block_sum<4>(s, red)) + shift);
  if (vec) {
    if (k >= n) return;
    if constexpr (sizeof(O) == 4) {
      float* o = reinterpret_cast<float*>(out) + base + k;
#pragma unroll
      for (int i = 0; i < 2; ++i) *reinterpret_cast<float4*>(o + 4 * i) = float4{v[4 * i] - lse, v[4 * i + 1] - lse, v[4 * i + 2] - lse, v[4 * i + 3] - lse};
    } else {
      unsigned w[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) w[j] = static_cast<unsigned>(lsm_bits<O>(v[2 * j] - lse)) | (static_cast<unsigned>(lsm_bits<O>(v[2 * j + 1] - lse)) << 16);
      *reinterpret_cast<uint4*>(out + base + k) = uint4{w[0], w[1], w[2], w[3]};
    }
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (k + j * lsm_step<T>(0) < n) out[base + k + j * lsm_step<T>(0)] = static_cast<O>(v[j] - lse);
  }
}

template <typename T, typename O>
__global__ __launch_bounds__(LSM_NT) void log_softmax_kernel(const T* __restrict__ x, O* __restrict__ out, int n, int vec, float scale) {
  constexpr int PER = 16 / sizeof(T), NWV = LSM_NT / 64;
  __shared__ float red[NWV];
  const T* row = x + static_cast<int64_t>(blockIdx.x) * n;
  O* orow = out + static_cast<int64_t>(blockIdx.x) * n;
  const int nv = vec ? n / PER : 0;                          // whole 16-byte pieces; the rest (all of it where rows are not aligned) one by one
  const uint4* rv = reinterpret_cast<const uint4*>(row);
  const int tid = threadIdx.x;
  uint4 v[LSM_VR];
  float m = -INFINITY;
#pragma unroll
  for (int i = 0; i < LSM_VR; ++i) {
    const int k = tid + i * LSM_NT;
    if (k < nv) {
      v[i] = rv[k];
#pragma unroll
      for (int j = 0; j < PER; ++j) m = fmaxf(m, lsm_get<T>(v[i], j) * scale);
    }
  }
  for (int k = tid + LSM_VR * LSM_NT; k < nv; k += LSM_NT) {
    const uint4 u = rv[k];
#pragma unroll
    for (int j = 0; j < PER; ++j) m = fmaxf(m, lsm_get<T>(u, j) * scale);
  }
  for (int k = nv * PER + tid; k < n; k += LSM_NT) m = fmaxf(m, static_cast<float>(row[k]) * scale);
  m = wave_max(m);
  if ((tid & 63) == 0) red[tid >> 6] = m;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NWV; ++i) m = fmaxf(m, red[i]);
  if (isinf(m)) m = 0.f;
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < LSM_VR; ++i)
    if (tid + i * LSM_NT < nv) {
#pragma unroll
      for (int j = 0; j < PER; ++j) s += expf(lsm_get<T>(v[i], j) * scale - m);
    }
  for (int k = tid + LSM_VR * LSM_NT; k < nv; k += LSM_NT) {
    const uint4 u = rv[k];
#pragma unroll
    for (int j = 0; j < PER; ++j) s += expf(lsm_get<T>(u, j) * scale - m);
  }
  for (int k = nv * PER + tid; k < n; k += LSM_NT) s += expf(static_cast<float>(row[k]) * scale - m);
  s = block_sum<NWV>(s, red);
  const float lse = lsm_round<O>(logf(s) + m);
  auto put = [&](int k, const uint4& u) {
    if constexpr (sizeof(O) == 4) {
#pragma unroll
      for (int i = 0; i < PER; i += 4)
        reinterpret_cast<float4*>(orow)[(k * PER + i) / 4] = float4{lsm_get<T>(u, i) * scale - lse, lsm_get<T>(u, i + 1) * scale - lse, lsm_get<T>(u, i + 2) * scale - lse,
                                                                    lsm_get<T>(u, i + 3) * scale - lse};
    } else {
      uint4 r;
      unsigned* w = &r.x;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        w[j] = static_cast<unsigned>(lsm_bits<O>(lsm_get<T>(u, 2 * j) * scale - lse)) | (static_cast<unsigned>(lsm_bits<O>(lsm_get<T>(u, 2 * j + 1) * scale - lse)) << 16);
      reinterpret_cast<uint4*>(orow)[k] = r;
    }
  };
#pragma unroll
  for (int i = 0; i < LSM_VR; ++i)
    if (tid + i * LSM_NT < nv) put(tid + i * LSM_NT, v[i]);
  for (int k = tid + LSM_VR * LSM_NT; k < nv; k += LSM_NT) put(k, rv[k]);
  for (int k = nv * PER + tid; k < n; k += LSM_NT) orow[k] = static_cast<O>(static_cast<float>(row[k]) * scale - lse);
}

// The tables of a step's rows and query tiles, from its sequences' (slot, first position, rows, first row) and first tiles.  Written on the host, entry by entry, they kept the
// chip waiting: 8 192 rows 1.2 ms, here 3 us.
__device__ __forceinline__ int step_sequence(const int* __restrict__ first, int stride, int B, int i) {      // the last one that starts at or before i
  int lo = 0, hi = B - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (first[static_cast<int64_t>(mid) * stride] <= i) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}
__global__ __launch_bounds__(256) void step_tables_kernel(const int* __restrict__ seq, const int* __restrict__ tile0, int2* __restrict__ tok, int2* __restrict__ tiles, int B, int T,
                                                         int n_tiles, int q_tile) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < T) {
    const int b = step_sequence(seq + 3, 4, B, i);
    tok[i] = int2{b, seq[4 * b + 1] + i - seq[4 * b + 3]};
  }
  if (i < n_tiles) {
    const int b = step_sequence(tile0, 1, B, i);
    tiles[i] = int2{b, (i - tile0[b]) * q_tile};
  }
}

// The tokens of the next step of the same sequences, from where they were chosen, and every position one further: what a step needs that is enqueued before the host has
// read them.  A step of the 4-layer models in batching.py's loop, us, tokens through the host | ahead of it: one sequence, several streams of 1024 244 | 219; two, latent attention 387 |
// 362; 32, sandwich norms 1124 | 1080 (a replay of the step alone: 200, 332 and 1043).
// The host has not yet looked at the tokens: one that is no row of the embedding (a sampler's end mark) goes on as token 0, in a step whose row the host then drops.
template <typename I>
__global__ __launch_bounds__(256) void step_advance_kernel(const I* __restrict__ from, int64_t rows, int64_t* __restrict__ tokens, int* __restrict__ seq, int* __restrict__ tok,
                                                           int B) {
  const int b = threadIdx.x;
  if (b >= B) return;
  const int64_t v = from[b];
  tokens[b] = v >= 0 && v < rows ? v : 0;
  seq[4 * b + 1] += 1;
  tok[2 * b + 1] += 1;
}

template <typename T, typename O = T>
void launch_log_softmax(const void* x, void* out, int64_t rows, int n, float* part, float scale, hipStream_t s) {
  constexpr int PER = 16 / sizeof(T);
  const T* xt = static_cast<const T*>(x);
  O* ot = static_cast<O*>(out);
  const bool aligned = (reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out)) % 16 == 0;
  if (part) {
    const dim3 grid((n + LSM_SLICE - 1) / LSM_SLICE, static_cast<unsigned>(rows));
    const int vec = aligned && n % 8 == 0;
    log_softmax_slice_kernel<T><<<grid, 256, 0, s>>>(xt, reinterpret_cast<float2*>(part), n, vec, scale);
    log_softmax_write_kernel<T, O><<<grid, 256, 0, s>>>(xt, reinterpret_cast<const float2*>(part), ot, n, vec, scale);
    return;
  }
  const int vec = aligned && (rows == 1 || n % PER == 0);
  log_softmax_kernel<T, O><<<static_cast<unsigned>(rows), LSM_NT, 0, s>>>(xt, ot, n, vec, scale);
}

template <typename T>
__global__ __launch_bounds__(NT) void segment_rmsnorm_kernel(T* __restrict__ rows, int64_t stride, int n0, int n1, const float* __restrict__ w0,
                                                            const float* __restrict__ w1, float eps) {
  constexpr int VR = 16;                   // values a thread keeps between the two passes
  __shared__ float red[NW];
  const int seg = blockIdx.y;
  T* p = rows + blockIdx.x * stride + (seg ? n0 : 0);
  const int n = seg ? n1 : n0;
  const float* w = seg ? w1 : w0;
  float vr[VR];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < VR; ++i) {
    const int c = threadIdx.x + i * NT;
    vr[i] = c < n ? to_f32(p[c]) : 0.f;
    ss += vr[i] * vr[i];
  }
  for (int c = threadIdx.x + VR * NT; c < n; c += NT) { const float v = to_f32(p[c]); ss += v * v; }
  ss = block_sum<NW>(ss, red);
  const float r = 1.f / sqrtf(ss / n + eps);
#pragma unroll
  for (int i = 0; i < VR; ++i) {
    const int c = threadIdx.x + i * NT;
    if (c < n) p[c] = from_f32<T>(vr[i] * r * w[c]);
  }
  for (int c = threadIdx.x + VR * NT; c < n; c += NT) p[c] = from_f32<T>(to_f32(p[c]) * r * w[c]);
}

// G groups of four channels a thread; the waves of either segment sum their own squares.
template <typename T, int G>
__global__ __launch_bounds__(1024) void segment_rmsnorm_row_kernel(T* __restrict__ rows, int64_t stride, int n0, int n1, int waves0, const float* __restrict__ w0,
                                                                   const float* __restrict__ w1, float eps) {
  __shared__ float red[16];
  const int wave = threadIdx.x >> 6, seg = wave >= waves0, first = seg ? waves0 : 0, last = seg ? static_cast<int>(blockDim.x >> 6) : waves0;
  const int n = seg ? n1 : n0, lanes = (last - first) * 64, c0 = static_cast<int>(threadIdx.x - first * 64) * 4;
  const float* w = seg ? w1 : w0;
  T* p = rows + blockIdx.x * stride + (seg ? n0 : 0);
  float v[G][4], f[G][4];
  float ss = 0.f;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int c = c0 + g * lanes * 4;
    if (c >= n) continue;
    Lanes<T, 4>::load(p + c, v[g]);
    Lanes<float, 4>::load(w + c, f[g]);
#pragma unroll
    for (int i = 0; i < 4; ++i) ss += v[g][i] * v[g][i];
  }
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) red[wave] = ss;
  __syncthreads();
  ss = 0.f;
  for (int i = first; i < last; ++i) ss += red[i];
  const float r = 1.f / sqrtf(ss / n + eps);
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int c = c0 + g * lanes * 4;
    if (c >= n) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[g][i] = v[g][i] * r * f[g][i];
    Lanes<T, 4>::store(p + c, v[g]);
  }
}

template <typename T>
void launch_segment_rmsnorm(T* rows, int64_t T_, int64_t stride, int n0, int n1, const float* w0, const float* w1, float eps, hipStream_t s) {
  const bool fours = stride % 4 == 0 && n0 % 4 == 0 && n1 % 4 == 0 && all_aligned(4 * sizeof(T), rows) && all_aligned(16, w0, w1);
  for (int g = 1; fours && g <= 2; ++g) {
    const int waves0 = (n0 + 256 * g - 1) / (256 * g), waves1 = (n1 + 256 * g - 1) / (256 * g);
    if (waves0 + waves1 > 16) continue;
    const int threads = (waves0 + waves1) * 64;
    if (g == 1) segment_rmsnorm_row_kernel<T, 1><<<static_cast<unsigned>(T_), threads, 0, s>>>(rows, stride, n0, n1, waves0, w0, w1, eps);
    else segment_rmsnorm_row_kernel<T, 2><<<static_cast<unsigned>(T_), threads, 0, s>>>(rows, stride, n0, n1, waves0, w0, w1, eps);
    return;
  }
  segment_rmsnorm_kernel<T><<<dim3(T_, 2), NT, 0, s>>>(rows, stride, n0, n1, w0, w1, eps);
}

constexpr int ZR = 16;             // branch values a thread keeps between the statistic and the update (rows up to ZR * NT wide)

template <typename T>
__global__ __launch_bounds__(NT) void residual_norm_add_kernel(float* __restrict__ x, const T* __restrict__ branch, const float* __restrict__ mix,
                                                              const float* __restrict__ w, T* __restrict__ h, int width, int top, float eps,
                                                              float mult) {
  __shared__ float red[NW];
  __shared__ float ml[64];
  const int64_t t = blockIdx.x;
  const T* b = branch + t * top * width;
  const bool mixed = mix != nullptr;
  if (mixed && threadIdx.x < min(top, 64)) ml[threadIdx.x] = mix[t * top + threadIdx.x];
  __syncthreads();
  auto z_at = [&](int c) {
    if (!mixed) return to_f32(b[c]);
    float z = 0.f;
    for (int s = 0; s < top; ++s) z += (s < 64 ? ml[s] : mix[t * top + s]) * to_f32(b[s * width + c]);
    return z;
  };
  float zr[ZR];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < ZR; ++i) {
    const int c = threadIdx.x + i * NT;
    zr[i] = c < width ? z_at(c) : 0.f;
    ss += zr[i] * zr[i];
  }
  for (int c = threadIdx.x + ZR * NT; c < width; c += NT) { const float z = z_at(c); ss += z * z; }
  ss = block_sum<NW>(ss, red);
  const float r = 1.f / sqrtf(ss / width + eps);
#pragma unroll
  for (int i = 0; i < ZR; ++i) {
    const int c = threadIdx.x + i * NT;
    if (c < width) {
      const float v = x[t * width + c] + mult * (zr[i] * r * w[c]);
      x[t * width + c] = v;
      if (h) h[t * width + c] = from_f32<T>(v);
    }
  }
  for (int c = threadIdx.x + ZR * NT; c < width; c += NT) {
    const float v = x[t * width + c] + mult * (z_at(c) * r * w[c]);
    x[t * width + c] = v;
    if (h) h[t * width + c] = from_f32<T>(v);
  }
}

template <typename T>
__global__ __launch_bounds__(NT) void stream_rmsnorm_kernel(const float* __restrict__ x, const float* __restrict__ w, T* __restrict__ out, int width,
                                                           float eps) {
  __shared__ float red[NW];
  const int64_t t = blockIdx.x;
  float ss = 0.f;
  for (int c = threadIdx.x; c < width; c += NT) { const float v = x[t * width + c]; ss += v * v; }
  ss = block_sum<NW>(ss, red);
  const float r = 1.f / sqrtf(ss / width + eps);
  for (int c = threadIdx.x; c < width; c += NT) out[t * width + c] = from_f32<T>(x[t * width + c] * r * w[c]);
}

template <typename T>
__global__ __launch_bounds__(1024) void residual_norm_add_row_kernel(float* __restrict__ x, const T* __restrict__ branch, const float* __restrict__ mix,
                                                                     const float* __restrict__ w, T* __restrict__ h, int width, int top, float eps, float mult) {
  __shared__ float red[16];
  const int64_t t = blockIdx.x;
  const int c = threadIdx.x * 4;
  const bool on = c < width;
  const T* y = branch + t * top * width;
  const float* m = mix ? mix + t * top : nullptr;
  float z[4] = {0.f, 0.f, 0.f, 0.f}, v[4], f[4];
  if (on) {
    Branch<T> b;
    Lanes<float, 4>::load(x + t * width + c, v);
    Lanes<float, 4>::load(w + c, f);
    b.ask(y, m, top, width, c);
    b.sum(y, m, top, width, c, z);
  }
  const float r = 1.f / sqrtf(row_sum(z[0] * z[0] + z[1] * z[1] + z[2] * z[2] + z[3] * z[3], red, width) / width + eps);
  if (!on) return;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] += mult * (z[i] * r * f[i]);
  Lanes<float, 4>::store(x + t * width + c, v);
  if (h) Lanes<T, 4>::store(h + t * width + c, v);
}

template <typename T>
__global__ __launch_bounds__(1024) void stream_rmsnorm_row_kernel(const float* __restrict__ x, const float* __restrict__ w, T* __restrict__ out, int width, float eps) {
  __shared__ float red[16];
  const int64_t t = blockIdx.x;
  const int c = threadIdx.x * 4;
  const bool on = c < width;
  float v[4] = {0.f, 0.f, 0.f, 0.f}, f[4];
  if (on) {
    Lanes<float, 4>::load(x + t * width + c, v);
    Lanes<float, 4>::load(w + c, f);
  }
  const float r = 1.f / sqrtf(row_sum(v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3], red, width) / width + eps);
  if (!on) return;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = v[i] * r * f[i];
  Lanes<T, 4>::store(out + t * width + c, v);
}

// Softmax over all experts and `top` rounds of arg-max on a row of fp32 router logits (the logits are a plain fp32 matrix product:
// the vendor library's); one workgroup per row.
__global__ __launch_bounds__(NT) void route_topk_kernel(const float* __restrict__ logits, int* __restrict__ idx, float* __restrict__ weight, int E,
                                                       int top, int renorm) {
  extern __shared__ float lg[];            // [E] logits, then probabilities
  __shared__ float red[NW];
  __shared__ float bestv[NW];
  __shared__ int besti[NW];
  const int64_t t = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int e = threadIdx.x; e < E; e += NT) lg[e] = logits[t * E + e];
  __syncthreads();
  float mx = -INFINITY;
  for (int e = threadIdx.x; e < E; e += NT) mx = fmaxf(mx, lg[e]);
  mx = wave_max(mx);
  if (lane == 0) red[wave] = mx;
  __syncthreads();
  mx = red[0];
#pragma unroll
  for (int i = 1; i < NW; ++i) mx = fmaxf(mx, red[i]);
  float sum = 0.f;
  for (int e = threadIdx.x; e < E; e += NT) { const float p = expf(lg[e] - mx); lg[e] = p; sum += p; }
  sum = block_sum<NW>(sum, red);
  for (int e = threadIdx.x; e < E; e += NT) {
    const float p = lg[e] / sum;
    lg[e] = p == p ? p : -1.f;                                 // (not a number: behind every probability, but still an expert)
  }
  __syncthreads();
  float chosen_sum = 0.f;
  for (int s = 0; s < top; ++s) {
    float bv = -1.5f;                                          // (-2: taken)
    int bi = 0x7fffffff;
    for (int e = threadIdx.x; e < E; e += NT)
      if (lg[e] > bv) { bv = lg[e]; bi = e; }                  // ascending e per thread: the first of equals stays
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(bv, o, 64);
      const int oi = __shfl_xor(bi, o, 64);
      if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
    }
    if (lane == 0) { bestv[wave] = bv; besti[wave] = bi; }
    __syncthreads();
    bv = bestv[0]; bi = besti[0];
#pragma unroll
    for (int i = 1; i < NW; ++i)
      if (bestv[i] > bv || (bestv[i] == bv && besti[i] < bi)) { bv = bestv[i]; bi = besti[i]; }
    __syncthreads();
    if (threadIdx.x == 0) { idx[t * top + s] = bi; weight[t * top + s] = bv; lg[bi] = -2.f; }
    chosen_sum += bv;
    __syncthreads();
  }
  if (renorm && threadIdx.x < top) weight[t * top + threadIdx.x] /= chosen_sum;
}

// The same by rank: probabilities and their order as above, no round waits for another.
__global__ __launch_bounds__(NT) void route_topk_rank_kernel(const float* __restrict__ logits, int* __restrict__ idx, float* __restrict__ weight, int E,
                                                            int top, int renorm) {
  __shared__ __attribute__((aligned(16))) float pl[RANK_EXPERTS];
  __shared__ float sel[NT];
  __shared__ float red[NW], mxs[NW];
  const int64_t t = blockIdx.x;
  constexpr int PER = RANK_EXPERTS / NT;
  float v[PER];
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = threadIdx.x + i * NT;
    v[i] = e < E ? logits[t * E + e] : -INFINITY;
    mx = fmaxf(mx, v[i]);
  }
  mx = wave_max(mx);
  if ((threadIdx.x & 63) == 0) mxs[threadIdx.x >> 6] = mx;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NW; ++i) mx = fmaxf(mx, mxs[i]);
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const bool live = static_cast<int>(threadIdx.x) + i * NT < E;
    v[i] = live ? expf(v[i] - mx) : 0.f;
    sum += v[i];
  }
  sum = block_sum<NW>(sum, red);
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const bool live = static_cast<int>(threadIdx.x) + i * NT < E;
    v[i] = live ? v[i] / sum : -1.f;
    if (!(v[i] == v[i])) v[i] = -1.f;            // (not a number: behind every probability)
    pl[threadIdx.x + i * NT] = v[i];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = threadIdx.x + i * NT;
    if (e < E) {
      const int rank = rank_of(pl, (E + 3) / 4, e, v[i]);
      if (rank < top) {
        idx[t * top + rank] = e;
        if (renorm) sel[rank] = v[i]; else weight[t * top + rank] = v[i];
      }
    }
  }
  if (!renorm) return;
  __syncthreads();
  if (static_cast<int>(threadIdx.x) < top) {
    float chosen = 0.f;
    for (int k = 0; k < top; ++k) chosen += sel[k];
    weight[t * top + threadIdx.x] = sel[threadIdx.x] / chosen;
  }
}

// The same for up to 64 PER experts, a wave per row.
template <int PER>
__global__ __launch_bounds__(256) void route_topk_wave_kernel(const float* __restrict__ logits, int* __restrict__ idx, float* __restrict__ weight, int64_t rows, int E,
                                                              int top, int renorm) {
  const int lane = threadIdx.x & 63;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (t >= rows) return;
  float v[PER], mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < PER; ++i) v[i] = lane + 64 * i < E ? logits[t * E + lane + 64 * i] : -INFINITY;
#pragma unroll
  for (int i = 0; i < PER; ++i) mx = fmaxf(mx, v[i]);
  mx = wave_max(mx);
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    v[i] = lane + 64 * i < E ? expf(v[i] - mx) : 0.f;
    sum += wave_sum(v[i]);
  }
  unsigned key[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const float p = v[i] / sum;
    key[i] = lane + 64 * i < E ? order_key(p == p ? p : -1.f) : 0u;      // (not a number: behind every probability, but still an expert)
  }
  float chosen = 0.f, p = 0.f;                                           // lane k holds choice k
  int mine = 0;
  wave_choose(key, top, [&](int k, int e, unsigned m) {
    const float v = key_value(m);
    chosen += v;
    if (lane == k) { mine = e; p = v; }
  });
  if (lane >= top) return;
  idx[t * top + lane] = mine;
  weight[t * top + lane] = renorm ? p / chosen : p;
}

// V: channels a thread copies at a time (4: rows, rings and their starts in groups of four)
template <typename T, int V>
__global__ __launch_bounds__(NT) void window_append_kernel(const T* __restrict__ qkv, int64_t stride, int nq, int nk, int nv, T* __restrict__ kc,
                                                          T* __restrict__ vc, const int* __restrict__ seq, const int* __restrict__ tok, int window) {
  const int64_t t = blockIdx.x;
  const int b = tok[2 * t], pos = tok[2 * t + 1];
  const int slot = seq[4 * b], pos0 = seq[4 * b + 1], n = seq[4 * b + 2];
  if (pos < pos0 + n - window) return;          // a later row of this step takes the same ring row
  const T* src = qkv + t * stride + nq;
  const int64_t row = static_cast<int64_t>(slot) * window + pos % window;
  struct alignas(V * sizeof(T)) Group { T v[V]; };
  for (int c = threadIdx.x * V; c < nk + nv; c += NT * V)
    *reinterpret_cast<Group*>(c < nk ? kc + row * nk + c : vc + row * nv + (c - nk)) = *reinterpret_cast<const Group*>(src + c);
}

bool act_ok(int act) { return act == GBXM_BF16 || act == GBXM_F32; }

}  // namespace
}  // namespace gbxm

using namespace gbxm;

extern "C" {

int gbxm_version(void) { return 100; }
const char* gbxm_last_error(void) { return g_err; }

#define GBXM_DISPATCH(act, CALL)              \
  do {                                        \
    if ((act) == GBXM_BF16) { using T = bf16_t; CALL; } else { using T = float; CALL; } \
  } while (0)

static int embed_rows(const void* table, const int64_t* tokens, float* x, void* h, int64_t h_row, int64_t T_, int32_t width, float scale, int32_t copies, int32_t act,
                      void* stream) {
  if (!act_ok(act) || !table || !tokens || !x || width <= 0 || T_ < 0 || (h && h_row < width)) return fail(GBXM_ERR_INVALID, "embed_scaled: bad argument");
  if (T_ == 0) return GBXM_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int threads = row_threads(width);
  const size_t group = act == GBXM_BF16 ? 8 : 16;
  if (threads && all_aligned(16, x) && all_aligned(group, static_cast<const char*>(table)) && (!h || (h_row % 4 == 0 && all_aligned(group, static_cast<const char*>(h)))))
    GBXM_DISPATCH(act, (embed_row_kernel<T><<<dim3(T_), threads, 0, s>>>(static_cast<const T*>(table), tokens, x, static_cast<T*>(h), h_row, width, scale, copies)));
  else
    GBXM_DISPATCH(act, (embed_kernel<T><<<dim3(T_), NT, 0, s>>>(static_cast<const T*>(table), tokens, x, static_cast<T*>(h), h_row, width, scale, copies)));
  return after_launch("embed_scaled");
}

int gbxm_embed_scaled(const void* table, const int64_t* tokens, float* x, void* h, int64_t h_row, int64_t T_, int32_t width, float scale, int32_t act,
                      void* stream) {
  return embed_rows(table, tokens, x, h, h_row, T_, width, scale, 1, act, stream);
}

// x [T, copies, width]: the embedding in every residual stream (a launch to spread it: 3 us and a row).  For this package's own Python layer; not part of the public header.
extern "C" int gbxm_embed_streams(const void* table, const int64_t* tokens, float* x, int64_t T_, int32_t width, int32_t copies, int32_t act, void* stream) {
  if (copies < 1 || copies > 64) return fail(GBXM_ERR_INVALID, "embed_streams: %d streams", copies);
  return embed_rows(table, tokens, x, nullptr, 0, T_, width, 1.f, copies, act, stream);
}

extern "C" int gbxm_step_tables(const int32_t* seq, const int32_t* tile0, int32_t* tok, int32_t* tiles, int32_t B, int32_t T_, int32_t n_tiles, int32_t q_tile, void* stream) {
  if (!seq || !tile0 || !tok || !tiles || B < 1 || T_ < 1 || n_tiles < 1 || n_tiles > T_ || q_tile < 1 || ((reinterpret_cast<uintptr_t>(tok) | reinterpret_cast<uintptr_t>(tiles)) & 7))
    return fail(GBXM_ERR_INVALID, "step_tables: bad argument");
  step_tables_kernel<<<(T_ + 255) / 256, 256, 0, static_cast<hipStream_t>(stream)>>>(seq, tile0, reinterpret_cast<int2*>(tok), reinterpret_cast<int2*>(tiles), B, T_, n_tiles, q_tile);
  return after_launch("step_tables");
}

extern "C" size_t gbxm_log_softmax_workspace(int64_t rows, int32_t n) {
  // few rows that are long: sixteen and more keep that many CUs busy in the one-launch form, shorter ones are done there before a second launch would start; one row
  // off the grid of eight takes wide accesses there and none in slices (one launch | two, us, bf16: 24 577 6.2 | 6.9, 28 001 6.7 | 7.0, 30 001 6.9 both, 32 769 9.9 | 6.9)
  return rows > 0 && rows < 16 && n > (rows == 1 && n % 8 ? 14 : 12) * LSM_SLICE ? static_cast<size_t>(rows) * ((n + LSM_SLICE - 1) / LSM_SLICE) * 8 : 0;
}

extern "C" int gbxm_log_softmax(const void* x, void* out, int64_t rows, int32_t n, int32_t type, void* ws, size_t ws_bytes, void* stream) {
  return gbxm_log_softmax_scaled(x, out, rows, n, type, type, 1.f, ws, ws_bytes, stream);
}

extern "C" int gbxm_log_softmax_scaled(const void* x, void* out, int64_t rows, int32_t n, int32_t type, int32_t out_type, float scale, void* ws, size_t ws_bytes, void* stream) {
  if (rows < 0 || n <= 0 || (type != GBXM_BF16 && type != GBXM_F32 && type != GBXM_F16) || (out_type != type && out_type != GBXM_F32) || rows > 0x7fffffff)
    return fail(GBXM_ERR_INVALID, "log_softmax: bad argument");
  if (rows == 0) return GBXM_OK;
  const size_t need = gbxm_log_softmax_workspace(rows, n);
  if (!x || !out || (need && (!ws || ws_bytes < need || reinterpret_cast<uintptr_t>(ws) % 8))) return fail(GBXM_ERR_INVALID, "log_softmax: null pointer or workspace");
  hipStream_t s = static_cast<hipStream_t>(stream);
  float* part = need ? static_cast<float*>(ws) : nullptr;
  if (type == GBXM_F32) launch_log_softmax<float>(x, out, rows, n, part, scale, s);
  else if (type == GBXM_BF16 && out_type == GBXM_F32) launch_log_softmax<__bf16, float>(x, out, rows, n, part, scale, s);
  else if (type == GBXM_BF16) launch_log_softmax<__bf16>(x, out, rows, n, part, scale, s);
  else if (out_type == GBXM_F32) launch_log_softmax<_Float16, float>(x, out, rows, n, part, scale, s);
  else launch_log_softmax<_Float16>(x, out, rows, n, part, scale, s);
  return after_launch("log_softmax");
}

extern "C" int gbxm_step_advance(const void* from, int32_t from_bytes, int64_t rows, int64_t* tokens, int32_t* seq, int32_t* tok, int32_t B, void* stream) {
  if (!from || rows < 1 || !tokens || !seq || !tok || B < 1 || B > 256 || (from_bytes != 4 && from_bytes != 8) || reinterpret_cast<uintptr_t>(from) % from_bytes ||
      reinterpret_cast<uintptr_t>(tokens) % 8 || (reinterpret_cast<uintptr_t>(seq) | reinterpret_cast<uintptr_t>(tok)) % 4)
    return fail(GBXM_ERR_INVALID, "step_advance: bad argument");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (from_bytes == 8) step_advance_kernel<int64_t><<<1, 256, 0, s>>>(static_cast<const int64_t*>(from), rows, tokens, seq, tok, B);
  else step_advance_kernel<int><<<1, 256, 0, s>>>(static_cast<const int*>(from), rows, tokens, seq, tok, B);
  return after_launch("step_advance");
}

int gbxm_segment_rmsnorm(void* rows, int64_t T_, int64_t row_stride, int32_t n0, int32_t n1, const float* w0, const float* w1, float eps,
                         int32_t act, void* stream) {
  if (!act_ok(act) || !rows || !w0 || !w1 || n0 <= 0 || n1 <= 0 || row_stride < n0 + n1 || T_ < 0)
    return fail(GBXM_ERR_INVALID, "segment_rmsnorm: bad argument");
  if (T_ == 0) return GBXM_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  GBXM_DISPATCH(act, (launch_segment_rmsnorm<T>(static_cast<T*>(rows), T_, row_stride, n0, n1, w0, w1, eps, s)));
  return after_launch("segment_rmsnorm");
}

int gbxm_residual_norm_add(float* x, const void* branch, const float* mix, const float* w, void* h, int64_t T_, int32_t width, int32_t top,
                           float eps, float mult, int32_t act, void* stream) {
  if (!act_ok(act) || !x || !branch || !w || width <= 0 || top < 1 || T_ < 0 || (top > 1 && !mix))
    return fail(GBXM_ERR_INVALID, "residual_norm_add: bad argument");
  if (act == GBXM_BF16 && !h) return fail(GBXM_ERR_INVALID, "residual_norm_add: bf16 needs the image buffer");
  if (T_ == 0) return GBXM_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int threads = row_threads(width);
  if (threads && all_aligned(16, x, w) && all_aligned(act == GBXM_BF16 ? 8 : 16, static_cast<const char*>(branch), static_cast<const char*>(h)))
    GBXM_DISPATCH(act, (residual_norm_add_row_kernel<T><<<dim3(T_), threads, 0, s>>>(x, static_cast<const T*>(branch), mix, w, static_cast<T*>(h), width, top, eps, mult)));
  else
    GBXM_DISPATCH(act, (residual_norm_add_kernel<T><<<dim3(T_), NT, 0, s>>>(x, static_cast<const T*>(branch), mix, w, static_cast<T*>(h), width, top, eps, mult)));
  return after_launch("residual_norm_add");
}

int gbxm_stream_rmsnorm(const float* x, const float* w, void* out, int64_t T_, int32_t width, float eps, int32_t act, void* stream) {
  if (!act_ok(act) || !x || !w || !out || width <= 0 || T_ < 0) return fail(GBXM_ERR_INVALID, "stream_rmsnorm: bad argument");
  if (T_ == 0) return GBXM_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int threads = row_threads(width);
  if (threads && all_aligned(16, x, w) && all_aligned(act == GBXM_BF16 ? 8 : 16, static_cast<const char*>(out)))
    GBXM_DISPATCH(act, (stream_rmsnorm_row_kernel<T><<<dim3(T_), threads, 0, s>>>(x, w, static_cast<T*>(out), width, eps)));
  else
    GBXM_DISPATCH(act, (stream_rmsnorm_kernel<T><<<dim3(T_), NT, 0, s>>>(x, w, static_cast<T*>(out), width, eps)));
  return after_launch("stream_rmsnorm");
}

int gbxm_route_topk(const float* logits, int32_t* idx, float* weight, int64_t T_, int32_t E, int32_t top, int32_t renorm, void* stream) {
  if (!logits || !idx || !weight || E <= 0 || top < 1 || top > E || T_ < 0) return fail(GBXM_ERR_INVALID, "route_topk: bad argument");
  if (E > 8192) return fail(GBXM_ERR_UNSUPPORTED, "route_topk: more than 8192 experts");
  if (top > NT) return fail(GBXM_ERR_UNSUPPORTED, "route_topk: top > %d", NT);
  if (T_ == 0) return GBXM_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (choice_by_wave(E, top, most_of_softmax(E))) {
    const unsigned blocks = choice_blocks(T_), threads = choice_threads(T_);
    if (E <= 64) route_topk_wave_kernel<1><<<blocks, threads, 0, s>>>(logits, idx, weight, T_, E, top, renorm);
    else if (E <= 128) route_topk_wave_kernel<2><<<blocks, threads, 0, s>>>(logits, idx, weight, T_, E, top, renorm);
    else route_topk_wave_kernel<4><<<blocks, threads, 0, s>>>(logits, idx, weight, T_, E, top, renorm);
  } else if (choice_by_rank(E, top)) route_topk_rank_kernel<<<dim3(T_), NT, 0, s>>>(logits, idx, weight, E, top, renorm);
  else route_topk_kernel<<<dim3(T_), NT, E * sizeof(float), s>>>(logits, idx, weight, E, top, renorm);
  return after_launch("route_topk");
}

int gbxm_window_append(const void* qkv, int64_t row_stride, int32_t nq, int32_t nk, int32_t nv, void* kcache, void* vcache, const int32_t* seq,
                       const int32_t* tok, int64_t T_, int32_t window, int32_t act, void* stream) {
  if (!act_ok(act) || !qkv || !kcache || !vcache || !seq || !tok || nq < 0 || nk <= 0 || nv <= 0 || row_stride < nq + nk + nv || window < 1 ||
      T_ < 0)
    return fail(GBXM_ERR_INVALID, "window_append: bad argument");
  if (T_ == 0) return GBXM_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool fours = row_stride % 4 == 0 && (nq | nk | nv) % 4 == 0 &&
                     all_aligned(act == GBXM_BF16 ? 8 : 16, static_cast<const char*>(qkv), static_cast<const char*>(kcache), static_cast<const char*>(vcache));
#define GBXM_APPEND(V_) window_append_kernel<T, V_><<<dim3(T_), NT, 0, s>>>(static_cast<const T*>(qkv), row_stride, nq, nk, nv, static_cast<T*>(kcache), \
                                                                           static_cast<T*>(vcache), seq, tok, window)
  if (fours) GBXM_DISPATCH(act, GBXM_APPEND(4));
  else GBXM_DISPATCH(act, GBXM_APPEND(1));
#undef GBXM_APPEND
  return after_launch("window_append");
}

}  // extern "C"
