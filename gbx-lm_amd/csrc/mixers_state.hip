// Recurrent mixers: a decayed matrix state per head.
//
//   recurrent_prep_kernel   short causal convolution + silu on q | k | v, unit q / k heads (a wave per head), q scale, the decay
//                           exp(-rate_h softplus(sign (a + bias))) and beta = sigmoid(b), all in fp32, into one fp32 row.
//   conv_tail_kernel        the last taps-1 convolution inputs of every sequence into its slot.
//   state_scan_kernel<R>    the scan token by token (mixers_state_scan.h; steps with longer portions: mixers_state_mfma.hip).  The columns of a head's state (one per value channel) never meet: a wave takes four columns, 16
//                           lanes per column, a lane holds R key channels of its column in registers; per token the two dot products
//                           over key channels are R multiply-adds and four cross-lane adds inside a 16-lane row (all 16 lanes end
//                           with the same bits).  Operands come through LDS in chunks of tokens, the next chunk fetched while the
//                           current one is computed.  Sums run in a fixed order: a sequence's result does not depend on what else is
//                           in the step, nor on how many columns a workgroup takes.
//   head_norm_gate_kernel   per-head RMS norm of the read-out, weight and gate, one wave per (row, head).
#include "mixers_mfma.h"
#include "mixers_state_scan.h"

namespace gbxm {
namespace {

constexpr int NT = 256, NW = NT / 64;

// grid (rows, splits): the splits of a row share out its q / k heads (a wave per head, up to MAXD channels a lane in registers),
// its value channels, its decays and betas; a step of few rows takes more splits.  Loads are issued unconditionally (a tap before
// the sequence's start reads a clamped address and counts as zero).
constexpr int MAXD = 4;                     // head channels per lane: heads of up to 256 channels

template <typename T, bool FAST>
__global__ __launch_bounds__(NT) void recurrent_prep_kernel(gbxm_recurrent_prep_args p) {
  const int64_t t = blockIdx.x;
  const int b = p.tok[2 * t], pos = p.tok[2 * t + 1];
  const int slot = p.seq[4 * b], pos0 = p.seq[4 * b + 1], row0 = p.seq[4 * b + 3];
  const int nq = p.G * p.dk, nv = p.H * p.dv, nd = p.H * p.dk;
  const int C = 2 * nq + nv;
  const T* y = static_cast<const T*>(p.y);
  const T* yr = y + t * p.y_stride;
  const T* cw = static_cast<const T*>(p.conv);
  const T* tail = p.taps > 1 ? static_cast<const T*>(p.tail) + static_cast<int64_t>(slot) * (p.taps - 1) * C : nullptr;
  float* out = p.out + t * p.out_stride;
  // channel c of q | k | v after the convolution and silu (or as projected, without a convolution; `plain`: its offset in the row)
  auto value = [&](int c, int plain) {
    if (!cw) { const float x = to_f32(yr[plain]); return p.qkv_silu ? x * sigmoid_<FAST>(x) : x; }
    float acc = 0.f;
    for (int j = 0; j < p.taps; ++j) {
      const int src = pos - (p.taps - 1) + j;
      const bool own = src >= pos0;
      const T* sp = own ? y + (row0 + (src - pos0)) * p.y_stride + p.off_q + c
                        : (tail ? tail + static_cast<int64_t>(max(src, pos0 - (p.taps - 1)) - pos0 + p.taps - 1) * C + c : yr + p.off_q + c);
      const float x = to_f32(*sp);
      acc += src >= 0 ? to_f32(cw[c * p.taps + j]) * x : 0.f;
    }
    return acc * sigmoid_<FAST>(acc);
  };
  const int lane = threadIdx.x & 63;
  const int gwave = blockIdx.y * NW + (threadIdx.x >> 6), n_waves = gridDim.y * NW;
  const int gthread = blockIdx.y * NT + threadIdx.x, n_threads = gridDim.y * NT;
  for (int hd = gwave; hd < 2 * p.G; hd += n_waves) {                  // q heads, then k heads
    const int first = hd * p.dk, plain = (hd < p.G ? p.off_q + first : p.off_k + first - nq);
    float v[MAXD];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < MAXD; ++i) {
      const int c = lane + 64 * i;
      const bool live = c < p.dk;
      const float x = value(first + (live ? c : 0), plain + (live ? c : 0));
      v[i] = live ? x : 0.f;
      ss += v[i] * v[i];
    }
    float mul = hd < p.G ? p.q_scale : 1.f;
    if (p.unit) mul *= 1.f / sqrtf(wave_sum(ss) + 1e-6f);
#pragma unroll
    for (int i = 0; i < MAXD; ++i)
      if (lane + 64 * i < p.dk) out[first + lane + 64 * i] = v[i] * mul;
  }
  for (int c = gthread; c < nv; c += n_threads) out[2 * nq + c] = value(2 * nq + c, p.off_v + c);
  const T* ar = static_cast<const T*>(p.a) + t * p.a_stride;
  if (!p.a) {                               // no decay projection: the head's constant
    for (int c = gthread; c < nd; c += n_threads) out[2 * nq + nv + c] = p.decay_rate[c / p.dk];
  } else for (int c = gthread; c < nd; c += n_threads) {
    const float z = p.sign * (to_f32(ar[c]) + p.decay_bias[c]);
    const float sp = z > 20.f ? z : log1p_<FAST>(exp_<FAST>(z));
    out[2 * nq + nv + c] = exp_<FAST>(-p.decay_rate[c / p.dk] * sp);
  }
  if (p.off_beta >= 0)
    for (int c = gthread; c < p.H; c += n_threads) out[2 * nq + nv + nd + c] = sigmoid_<FAST>(to_f32(yr[p.off_beta + c]));
}

// The same for rows in groups of four channels: a thread takes four neighbouring channels of R neighbouring rows of the step, so that every input is read once and
// not once per tap, in 8-byte pieces, and its taps once; a head's norm is a sum over the dk / 4 lanes that hold it.  The convolution's sum runs as above.
// Bound by the fp32 rows it writes (12 320 numbers a token in the first line) and the decays' logarithms and exponentials.  Measured, us: 2 266 rows, 32 heads of 128 with 16
// of q / k and a convolution 184 -> 67; without one, 8 heads of 128 x 256 29 -> 27; one row of the former kind, 8 heads of 64 x 128 6.4 -> 3.5.
template <typename T, bool CONV, int R>
__global__ __launch_bounds__(NT) void recurrent_prep_rows_kernel(gbxm_recurrent_prep_args p, T* tails) {
  const int nq = p.G * p.dk, nv = p.H * p.dv, nd = p.H * p.dk, C = 2 * nq + nv;
  const int c = (blockIdx.y * NT + threadIdx.x) * 4;
  const int64_t t0 = static_cast<int64_t>(blockIdx.x) * R;
  const int n = static_cast<int>(min(static_cast<int64_t>(R), p.T - t0));
  const T* __restrict__ y = static_cast<const T*>(p.y);
  float* __restrict__ out = p.out + t0 * p.out_stride;
  if (c < C) {
    const int place = c < nq ? p.off_q + c : c < 2 * nq ? p.off_k + c - nq : p.off_v + c - 2 * nq;
    float x[R][4], w[4][4], h[3][4];
#pragma unroll
    for (int i = 0; i < R; ++i) Lanes<T, 4>::load(y + (t0 + min(i, n - 1)) * p.y_stride + place, x[i]);
    if constexpr (CONV) {
#pragma unroll
      for (int k = 0; k < 4; ++k) Lanes<T, 4>::load(static_cast<const T*>(p.conv) + (c + k) * 4, w[k]);
    }
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if (i >= n) break;
      float v[4];
      if constexpr (CONV) {
        const int b = p.tok[2 * (t0 + i)], pos = p.tok[2 * (t0 + i) + 1], pos0 = p.seq[4 * b + 1];
        if (i == 0 || pos == pos0) {                         // the three inputs before this row: of the step, of the slot, or none
          const int64_t row0 = p.seq[4 * b + 3];
          const T* tail = static_cast<const T*>(p.tail) + static_cast<int64_t>(p.seq[4 * b]) * 3 * C;
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            const int src = pos - 3 + j;
            Lanes<T, 4>::load(src >= pos0 ? y + (row0 + (src - pos0)) * p.y_stride + place : tail + static_cast<int64_t>(max(src - pos0 + 3, 0)) * C + c, h[j]);
            if (src < 0) {
#pragma unroll
              for (int k = 0; k < 4; ++k) h[j][k] = 0.f;
            }
          }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          float acc = w[k][0] * h[0][k];
          acc += w[k][1] * h[1][k];
          acc += w[k][2] * h[2][k];
          acc += w[k][3] * x[i][k];
          v[k] = acc * sigmoid_<false>(acc);
          h[0][k] = h[1][k]; h[1][k] = h[2][k]; h[2][k] = x[i][k];
        }
        if (tails && pos == pos0 + p.seq[4 * b + 2] - 1) {   // (every sequence brings one row: nobody else reads these channels of the slot)
          T* to = tails + static_cast<int64_t>(p.seq[4 * b]) * 3 * C + c;
#pragma unroll
          for (int j = 0; j < 3; ++j) Lanes<T, 4>::store(to + static_cast<int64_t>(j) * C, h[j]);
        }
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = p.qkv_silu ? x[i][k] * sigmoid_<false>(x[i][k]) : x[i][k];
      }
      if (c < 2 * nq) {
        float mul = c < nq ? p.q_scale : 1.f;
        if (p.unit) {
          float ss = v[0] * v[0] + v[1] * v[1] + (v[2] * v[2] + v[3] * v[3]);
          mul *= 1.f / sqrtf(group_sum(ss, p.dk / 4) + 1e-6f);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] *= mul;
      }
      *reinterpret_cast<float4*>(out + i * p.out_stride + c) = float4{v[0], v[1], v[2], v[3]};
    }
  } else if (c < C + nd) {
    const int d = c - C;
    const float rate = p.decay_rate[d / p.dk];
    float z[R][4], bias[4];
    if (p.a) {
#pragma unroll
      for (int i = 0; i < R; ++i) Lanes<T, 4>::load(static_cast<const T*>(p.a) + (t0 + min(i, n - 1)) * p.a_stride + d, z[i]);
#pragma unroll
      for (int k = 0; k < 4; ++k) bias[k] = p.decay_bias[d + k];
    }
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if (i >= n) break;
      float v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        v[k] = rate;                                         // no decay projection: the head's constant
        if (p.a) {
          const float u = p.sign * (z[i][k] + bias[k]);
          v[k] = exp_<false>(-rate * (u > 20.f ? u : log1p_<false>(exp_<false>(u))));
        }
      }
      *reinterpret_cast<float4*>(out + i * p.out_stride + c) = float4{v[0], v[1], v[2], v[3]};
    }
  }
  if (p.off_beta >= 0 && blockIdx.y == gridDim.y - 1)
    for (int i = threadIdx.x; i < n * p.H; i += NT)
      out[(i / p.H) * p.out_stride + C + nd + i % p.H] = sigmoid_<false>(to_f32(y[(t0 + i / p.H) * p.y_stride + p.off_beta + i % p.H]));
}

// What that kernel takes: heads of 4, 8, .. 256 channels, everything in groups of four on the grid of their loads, four taps or no convolution.  Without one, rows
// of few numbers leave most of its lanes idle (one number a lane | this, us: 500 rows of 128 numbers 4.4 | 5.1, 8 192 16.0 | 29; of 256 4.4 | 4.9, 8 192 16.2 | 16.3,
// 16 000 30.8 | 21.5; of 512 4.6 | 3.9, 8 192 20.3 | 16.9).
template <typename T>
bool prep_rows_shape(const gbxm_recurrent_prep_args& a) {
  const int C = 2 * a.G * a.dk + a.H * a.dv;
  if (a.dk < 4 || a.dk > 256 || (a.dk & (a.dk - 1)) || a.H * a.dv % 4 || a.off_q % 4 || a.off_k % 4 || a.off_v % 4 || a.y_stride % 4 || a.out_stride % 4 || (a.conv && a.taps != 4) ||
      (a.a && a.a_stride % 4) || (!a.conv && C + a.H * a.dk < 256))
    return false;
  const T* none = nullptr;
  return all_aligned(4 * sizeof(T), static_cast<const T*>(a.y), a.a ? static_cast<const T*>(a.a) : none, a.conv ? static_cast<const T*>(a.conv) : none,
                     a.conv ? static_cast<const T*>(a.tail) : none) && all_aligned(16, a.out) && (C + a.H * a.dk + 4 * NT - 1) / (4 * NT) <= 65535;
}

template <typename T, bool CONV>
void launch_prep_rows(const gbxm_recurrent_prep_args& a, bool keep, hipStream_t s) {
  T* tails = keep ? static_cast<T*>(const_cast<void*>(a.tail)) : nullptr;
  const unsigned cols = (2 * a.G * a.dk + a.H * a.dv + a.H * a.dk + 4 * NT - 1) / (4 * NT);
  // eight rows a thread where that leaves the chip full, else one
  if (a.T * cols >= 8 * 1024) recurrent_prep_rows_kernel<T, CONV, 8><<<dim3((a.T + 7) / 8, cols), NT, 0, s>>>(a, tails);
  else recurrent_prep_rows_kernel<T, CONV, 1><<<dim3(a.T, cols), NT, 0, s>>>(a, tails);
}

template <typename T>
__global__ __launch_bounds__(NT) void conv_tail_kernel(const T* __restrict__ y, int64_t y_stride, T* __restrict__ tail, const int* __restrict__ seq,
                                                      int C, int taps) {
  const int b = blockIdx.y;
  const int slot = seq[4 * b], pos0 = seq[4 * b + 1], n = seq[4 * b + 2], row0 = seq[4 * b + 3];
  const int keep = taps - 1;
  T* tl = tail + static_cast<int64_t>(slot) * keep * C;
  for (int c = blockIdx.x * NT + threadIdx.x; c < C; c += gridDim.x * NT) {
    // entry i afterwards holds position pos0 + n - keep + i: ascending i reads entries above the ones already written
    for (int i = 0; i < keep; ++i) {
      const int pos = pos0 + n - keep + i;
      T v;
      if (pos >= pos0) v = y[(row0 + (pos - pos0)) * y_stride + c];
      else if (pos >= 0) v = tl[static_cast<int64_t>(i + n) * C + c];
      else v = from_f32<T>(0.f);
      tl[static_cast<int64_t>(i) * C + c] = v;
    }
  }
}

template <int R, bool DELTA, int NW, int V>
__global__ __launch_bounds__(64 * NW) void state_scan_kernel(const StateArgs a, const StateChunks made) {
  __shared__ __attribute__((aligned(16))) float lds[ScanShape<R, NW, scan_tokens(R, NW)>::FLOATS];
  const int b = blockIdx.z;
  if (made.flags && state_by_chunks(made, b, blockIdx.y, a.seq[4 * b + 2], a.seq[4 * b + 3])) return;
  scan_columns<R, DELTA, NW, V>(a, b, blockIdx.y, blockIdx.x * 4 * NW, lds);
}

template <typename T, bool FAST>
__global__ __launch_bounds__(NT) void head_norm_gate_kernel(const float* __restrict__ o, const T* __restrict__ gate, int64_t gate_stride,
                                                           const float* __restrict__ w, T* __restrict__ out, int64_t out_row, int H, int dv, float eps,
                                                           int kind) {
  const int64_t t = blockIdx.x;
  const int lane = threadIdx.x & 63;
  const int h = blockIdx.y * NW + (threadIdx.x >> 6);
  if (h >= H) return;
  const float* x = o + (t * H + h) * dv;
  float ss = 0.f;
  for (int c = lane; c < dv; c += 64) ss += x[c] * x[c];
  const float r = 1.f / sqrtf(wave_sum(ss) / dv + eps);
  const T* g = gate + t * gate_stride + h * dv;
  T* y = out + t * out_row + h * dv;
  for (int c = lane; c < dv; c += 64) {
    const float z = to_f32(g[c]);
    const float s = sigmoid_<FAST>(z);
    y[c] = from_f32<T>(x[c] * r * (w ? w[c] : 1.f) * (kind == 1 ? z * s : s));
  }
}

// The same in groups of four channels: dv / 4 neighbouring lanes hold a head (dv a power of two, 4 to 256), so that a wave takes 256 channels of a row whatever the
// head's size.  Bound by its traffic.  Measured, us: 2 266 rows, 32 heads of 128 26 -> 15, 8 heads of 256 12.5 -> 9.2.
template <typename T, bool FAST>
__global__ __launch_bounds__(NT) void head_norm_gate_vec_kernel(const float* __restrict__ o, const T* __restrict__ gate, int64_t gate_stride,
                                                               const float* __restrict__ w, T* __restrict__ out, int64_t out_row, int width, int dv, float eps,
                                                               int kind) {
  const int64_t t = blockIdx.x;
  const int c = (blockIdx.y * NT + threadIdx.x) * 4;
  if (c >= width) return;
  float x[4], g[4], m[4] = {1.f, 1.f, 1.f, 1.f};
  Lanes<float, 4>::load(o + t * width + c, x);
  Lanes<T, 4>::load(gate + t * gate_stride + c, g);
  if (w) {
#pragma unroll
    for (int k = 0; k < 4; ++k) m[k] = w[(c & (dv - 1)) + k];
  }
  float ss = x[0] * x[0] + x[1] * x[1] + (x[2] * x[2] + x[3] * x[3]);
  const float r = 1.f / sqrtf(group_sum(ss, dv / 4) / dv + eps);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float s = sigmoid_<FAST>(g[k]);
    x[k] = x[k] * r * m[k] * (kind == 1 ? g[k] * s : s);
  }
  Lanes<T, 4>::store(out + t * out_row + c, x);
}

// The same for heads of more channels (all heads normalised together): a workgroup a head, GROUPS times four channels a thread, all of a row in flight.  Bound by the
// trip to memory and the sum across waves.  Measured, us, one wave a head | this: 32 rows of 2 048 channels 11.5 | 3.8 (23 | 4 among other kernels, code and rows cold), 2 736
// 25.7 | 12.2, 32 rows of 512 4.7 | 3.0, 300 of 300 4.1 | 3.3.
template <typename T, int GROUPS>
__global__ __launch_bounds__(NT) void head_norm_gate_wide_kernel(const float* __restrict__ o, const T* __restrict__ gate, int64_t gate_stride,
                                                                const float* __restrict__ w, T* __restrict__ out, int64_t out_row, int dv, float eps, int kind) {
  __shared__ float red[NW];
  const int64_t t = blockIdx.x;
  const int h = blockIdx.y;
  const float* orow = o + (t * gridDim.y + h) * dv;
  const T* grow = gate + t * gate_stride + h * dv;
  float x[GROUPS][4], g[GROUPS][4], m[GROUPS][4];
#pragma unroll
  for (int i = 0; i < GROUPS; ++i) {                                    // (loads past the end repeat the last group)
    const int c = min((static_cast<int>(threadIdx.x) + NT * i) * 4, dv - 4);
    Lanes<float, 4>::load(orow + c, x[i]);
    Lanes<T, 4>::load(grow + c, g[i]);
#pragma unroll
    for (int k = 0; k < 4; ++k) m[i][k] = w ? w[c + k] : 1.f;
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < GROUPS; ++i) {
    const float q = x[i][0] * x[i][0] + x[i][1] * x[i][1] + (x[i][2] * x[i][2] + x[i][3] * x[i][3]);
    ss += (static_cast<int>(threadIdx.x) + NT * i) * 4 < dv ? q : 0.f;
  }
  const float r = 1.f / sqrtf(block_sum<NW>(ss, red) / dv + eps);
#pragma unroll
  for (int i = 0; i < GROUPS; ++i) {
    const int c = (static_cast<int>(threadIdx.x) + NT * i) * 4;
    if (c >= dv) break;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float s = sigmoid_<false>(g[i][k]);
      x[i][k] = x[i][k] * r * m[i][k] * (kind == 1 ? g[i][k] * s : s);
    }
    Lanes<T, 4>::store(out + t * out_row + h * dv + c, x[i]);
  }
}

template <typename T>
void launch_head_norm_gate(const float* o, const void* gate, int64_t gate_stride, const float* w, void* out, int64_t out_row, int64_t T_, int H, int dv, float eps,
                           int kind, hipStream_t s) {
  const T* g = static_cast<const T*>(gate);
  T* y = static_cast<T*>(out);
  const int64_t blocks = (static_cast<int64_t>(H) * dv / 4 + NT - 1) / NT;
  // (rows of less than 64 channels are a few lanes of a workgroup: 1 000 rows of one head of 16 2.6 us | 3.4, 629 of one of 32 2.5 | 3.2)
  if (H * dv >= 64 && dv >= 4 && dv <= 256 && !(dv & (dv - 1)) && gate_stride % 4 == 0 && out_row % 4 == 0 && all_aligned(4 * sizeof(T), g, static_cast<const T*>(y)) && all_aligned(16, o) &&
      blocks <= 65535)
    head_norm_gate_vec_kernel<T, false><<<dim3(T_, static_cast<unsigned>(blocks)), NT, 0, s>>>(o, g, gate_stride, w, y, out_row, H * dv, dv, eps, kind);
  else if (dv > 256 && dv <= 16 * NT && dv % 4 == 0 && H <= 65535 && gate_stride % 4 == 0 && out_row % 4 == 0 && all_aligned(4 * sizeof(T), g, static_cast<const T*>(y)) &&
           all_aligned(16, o)) {
    const dim3 grid(T_, H);
    if (dv <= 4 * NT) head_norm_gate_wide_kernel<T, 1><<<grid, NT, 0, s>>>(o, g, gate_stride, w, y, out_row, dv, eps, kind);
    else if (dv <= 8 * NT) head_norm_gate_wide_kernel<T, 2><<<grid, NT, 0, s>>>(o, g, gate_stride, w, y, out_row, dv, eps, kind);
    else head_norm_gate_wide_kernel<T, 4><<<grid, NT, 0, s>>>(o, g, gate_stride, w, y, out_row, dv, eps, kind);
  } else
    head_norm_gate_kernel<T, false><<<dim3(T_, (H + NW - 1) / NW), NT, 0, s>>>(o, g, gate_stride, w, y, out_row, H, dv, eps, kind);
}

template <bool DELTA, int NW>
int launch_scan(const StateArgs& a, const StateChunks& made, bool vec, hipStream_t s) {
  const int R = (a.dk + 15) / 16;
  const dim3 grid((a.dv + 4 * NW - 1) / (4 * NW), a.H, a.B);
#define GBXM_SCAN(N)                                                        \
  do {                                                                      \
    if (vec) state_scan_kernel<N, DELTA, NW, 4><<<grid, 64 * NW, 0, s>>>(a, made); \
    else state_scan_kernel<N, DELTA, NW, 1><<<grid, 64 * NW, 0, s>>>(a, made);     \
  } while (0)
  if (R <= 1) GBXM_SCAN(1);
  else if (R <= 2) GBXM_SCAN(2);
  else if (R <= 4) GBXM_SCAN(4);
  else if (R <= 6 && !vec) state_scan_kernel<6, DELTA, NW, 1><<<grid, 64 * NW, 0, s>>>(a, made);
  else if (R <= 8) GBXM_SCAN(8);
  else if (R <= 12) GBXM_SCAN(12);
  else GBXM_SCAN(16);
#undef GBXM_SCAN
  return after_launch("state_scan");
}

bool act_ok(int act) { return act == GBXM_BF16 || act == GBXM_F32; }

}  // namespace
}  // namespace gbxm

using namespace gbxm;

static int prepare(const gbxm_recurrent_prep_args* a, bool keep, void* stream) {
  if (!a || !act_ok(a->act) || !a->y || (a->a && !a->decay_bias) || !a->decay_rate || !a->seq || !a->tok || !a->out || a->T < 0 || a->H < 1 || a->G < 1 ||
      a->H % a->G || a->dk < 1 || a->dv < 1 || a->off_q < 0 || a->off_k < 0 || a->off_v < 0)
    return fail(GBXM_ERR_INVALID, "recurrent_prepare: bad argument");
  const int nq = a->G * a->dk, nv = a->H * a->dv, C = 2 * nq + nv;
  if (a->conv && (a->taps < 1 || (a->taps > 1 && !a->tail) || a->off_k != a->off_q + nq || a->off_v != a->off_k + nq))
    return fail(GBXM_ERR_INVALID, "recurrent_prepare: a convolution needs q | k | v side by side and the slots' tails");
  if (a->out_stride < C + a->H * a->dk + (a->off_beta >= 0 ? a->H : 0)) return fail(GBXM_ERR_INVALID, "recurrent_prepare: output rows too short");
  if (a->dk > 64 * MAXD) return fail(GBXM_ERR_UNSUPPORTED, "recurrent_prepare: heads of %d channels (at most %d)", a->dk, 64 * MAXD);
  if (a->T == 0) return GBXM_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool bf = a->act == GBXM_BF16;
  if (bf ? prep_rows_shape<bf16_t>(*a) : prep_rows_shape<float>(*a)) {
    if (bf && a->conv) launch_prep_rows<bf16_t, true>(*a, keep, s);
    else if (bf) launch_prep_rows<bf16_t, false>(*a, keep, s);
    else if (a->conv) launch_prep_rows<float, true>(*a, keep, s);
    else launch_prep_rows<float, false>(*a, keep, s);
    return after_launch("recurrent_prepare");
  }
  // splits of a row: enough workgroups for the chip when the step has few rows, never more than the row has work for
  int64_t splits = (1024 + a->T - 1) / a->T;
  const int64_t most = (C + a->H * a->dk + 4 * NT - 1) / (4 * NT);
  if (splits > most) splits = most;
  if (splits > 64) splits = 64;
  if (splits < 1) splits = 1;
  const dim3 grid(a->T, static_cast<unsigned>(splits));
  if (a->act == GBXM_BF16) recurrent_prep_kernel<bf16_t, false><<<grid, NT, 0, s>>>(*a);
  else recurrent_prep_kernel<float, false><<<grid, NT, 0, s>>>(*a);
  if (keep) {
    const dim3 grid((C + NT - 1) / NT, static_cast<unsigned>(a->T));
    if (bf) conv_tail_kernel<bf16_t><<<grid, NT, 0, s>>>(static_cast<const bf16_t*>(a->y) + a->off_q, a->y_stride, static_cast<bf16_t*>(const_cast<void*>(a->tail)), a->seq, C, a->taps);
    else conv_tail_kernel<float><<<grid, NT, 0, s>>>(static_cast<const float*>(a->y) + a->off_q, a->y_stride, static_cast<float*>(const_cast<void*>(a->tail)), a->seq, C, a->taps);
  }
  return after_launch("recurrent_prepare");
}

extern "C" {

int gbxm_recurrent_prepare(const gbxm_recurrent_prep_args* a, void* stream) { return prepare(a, false, stream); }

// The same and gbxm_conv_tail_update behind it, for a step whose every sequence brings one row (T sequences): the convolution's inputs go on into the slots from the registers that
// hold them (a launch of its own: 3.3 us).  For this package's own Python layer; not part of the public header.
int gbxm_recurrent_prepare_keep(const gbxm_recurrent_prep_args* a, void* stream) {
  if (!a || !a->conv || a->taps < 2 || a->T > 65535) return fail(GBXM_ERR_INVALID, "recurrent_prepare_keep: a convolution of two taps at least");
  return prepare(a, true, stream);
}

int gbxm_conv_tail_update(const void* y, int64_t y_stride, void* tail, const int32_t* seq, int32_t B, int32_t C, int32_t taps, int32_t act,
                          void* stream) {
  if (!act_ok(act) || !y || !tail || !seq || B < 0 || C < 1 || taps < 2 || y_stride < C) return fail(GBXM_ERR_INVALID, "conv_tail_update: bad argument");
  if (B == 0) return GBXM_OK;
  if (B > 65535) return fail(GBXM_ERR_UNSUPPORTED, "conv_tail_update: more than 65535 sequences in a step");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 grid((C + NT - 1) / NT, B);
  if (act == GBXM_BF16) conv_tail_kernel<bf16_t><<<grid, NT, 0, s>>>(static_cast<const bf16_t*>(y), y_stride, static_cast<bf16_t*>(tail), seq, C, taps);
  else conv_tail_kernel<float><<<grid, NT, 0, s>>>(static_cast<const float*>(y), y_stride, static_cast<float*>(tail), seq, C, taps);
  return after_launch("conv_tail_update");
}

size_t gbxm_state_scan_workspace(int32_t B, int64_t T_, int64_t longest, int32_t H, int32_t dk, int32_t dv) {
  return longest < STATE_CHUNKS_FROM || B < 1 || T_ < longest || H < 1 ? 0 : state_chunks_workspace(T_, B, H, dk, dv);
}

int gbxm_state_scan(const float* r, int64_t r_stride, float* state, float* out, const int32_t* seq, int32_t B, int64_t T_, int32_t H, int32_t G,
                    int32_t dk, int32_t dv, int32_t delta, void* stream) {
  return gbxm_state_scan_ws(r, r_stride, state, out, seq, B, T_, H, G, dk, dv, delta, nullptr, 0, stream);
}

int gbxm_state_scan_ws(const float* r, int64_t r_stride, float* state, float* out, const int32_t* seq, int32_t B, int64_t T_, int32_t H, int32_t G,
                       int32_t dk, int32_t dv, int32_t delta, void* ws, size_t ws_bytes, void* stream) {
  if (!r || !state || !out || !seq || B < 0 || H < 1 || G < 1 || H % G || dk < 1 || dv < 1 ||
      r_stride < 2 * G * dk + H * dv + H * dk + (delta ? H : 0))
    return fail(GBXM_ERR_INVALID, "state_scan: bad argument");
  if (dk > 256) return fail(GBXM_ERR_UNSUPPORTED, "state_scan: %d key channels per head (at most 256)", dk);
  if (B == 0) return GBXM_OK;
  if (B > 65535 || H > 65535) return fail(GBXM_ERR_UNSUPPORTED, "state_scan: grid");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const StateArgs a{r, r_stride, state, out, seq, B, H, G, dk, dv};
  const bool vec = dk % 4 == 0 && dv % 4 == 0 && r_stride % 4 == 0 && all_aligned(16, r, state);
  const size_t need = ws && vec ? state_chunks_workspace(T_, B, H, dk, dv) : 0;
  StateChunks made{nullptr, 0};
  if (need && ws_bytes >= need && r_stride <= (1 << 22) && all_aligned(16, static_cast<const char*>(ws))) {
    const int rc = launch_state_chunks(a, T_, delta, ws, s, &made);
    if (rc != GBXM_OK || !made.flags) return rc;
  }
  // long rows (prompts): 16 columns per workgroup share the staged operands; a few rows per sequence: 4 columns, four times the
  // workgroups for the state's traffic.  A column's arithmetic is the same in both.
  if (T_ >= 8 * static_cast<int64_t>(B)) return delta ? launch_scan<true, 4>(a, made, vec, s) : launch_scan<false, 4>(a, made, vec, s);
  return delta ? launch_scan<true, 1>(a, made, vec, s) : launch_scan<false, 1>(a, made, vec, s);
}

int gbxm_head_norm_gate(const float* o, const void* gate, int64_t gate_stride, const float* w, void* out, int64_t out_row, int64_t T_, int32_t H, int32_t dv,
                        float eps, int32_t kind, int32_t act, void* stream) {
  if (!act_ok(act) || !o || !gate || !out || T_ < 0 || H < 1 || dv < 1 || gate_stride < H * dv || out_row < H * dv || (kind != 1 && kind != 2))
    return fail(GBXM_ERR_INVALID, "head_norm_gate: bad argument");
  if (T_ == 0) return GBXM_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (act == GBXM_BF16) launch_head_norm_gate<bf16_t>(o, gate, gate_stride, w, out, out_row, T_, H, dv, eps, kind, s);
  else launch_head_norm_gate<float>(o, gate, gate_stride, w, out, out_row, T_, H, dv, eps, kind, s);
  return after_launch("head_norm_gate");
}

}  // extern "C"
