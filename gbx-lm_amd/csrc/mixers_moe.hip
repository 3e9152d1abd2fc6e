// Routed MLPs over dense stacked experts:  y[t][s] = down_e (silu(gate_e h_t) * (up_e h_t)),  e = idx[t][s] -- or another gated
// activation, or experts without a gate, down_e relu(up_e h_t)^2.  With a factor per (row, choice) an expert reads the scaled row: the
// factor meets the fp32 sums of its first products.
//
//   * row kernels -- weight-bandwidth bound: the kernels of decode steps, of fp32 models and of shapes the grouped kernel does not
//     take.  Two launches so that even ONE row spreads over the chip: the first (a workgroup = one (row, choice) pair x some hidden
//     channels, lanes across the contraction, fp32 sums in a fixed order) leaves the hidden row in the workspace, the second (a pair x 16
//     output channels) consumes it.  expert_up_vec / expert_down_vec where rows are whole 16-byte vectors, else expert_up_rows / _down_rows.
//   * grouped matrix-core products for bf16 prompt portions (rows sorted by expert on the device, no host round trip).
#include "mixers_common.h"

namespace gbxm {
namespace {

constexpr int NT = 256, NW = NT / 64;
constexpr int FC = 8;             // hidden channels per workgroup of expert_up_rows
constexpr int KC = 16;            // output channels per workgroup of expert_down_rows

// The vector form.  Four rows of weights per wave, 16 lanes a row: a row's whole sum is four cross-lane adds, the four rows' at once, and the row that
// they meet is read as it is, from the first cache: nothing is staged and no barrier stands before the weights.  UN steps of 16 lanes x 16 bytes are in
// flight per matrix.  Bound by the weights' way from memory (16 pairs of 768 x 2048) or one trip to it (4 pairs of 512 x 1024).
// (Rows staged in LDS, one wave per channel -> now, us: 16 pairs, 768 x 2048, first and second product 17.4 + 17.9 -> 13.1 + 12.3 (4.1 TB/s); 4 gated
// pairs, 512 x 1024, 7.2 + 5.3 -> 5.9 + 3.8.)
constexpr int UN = 4;

// s0 = sum_k w0[k] x[k], s1 = sum_k w1[k] x[k] (PAIR), every lane of the 16 gets them; n a multiple of the vector
template <typename T, bool PAIR>
__device__ __forceinline__ void rows_dot(const T* __restrict__ w0, const T* __restrict__ w1, const T* __restrict__ x, int n, int l16, float& s0, float& s1) {
  constexpr int PER = 16 / sizeof(T), STEP = 16 * PER;
  float a0[2] = {0.f, 0.f}, a1[2] = {0.f, 0.f};
  for (int k0 = 0; k0 < n; k0 += UN * STEP) {
    uint4 u[UN], v[UN], y[UN];
#pragma unroll
    for (int i = 0; i < UN; ++i) {
      const int k = min(k0 + i * STEP + l16 * PER, n - PER);
      u[i] = *reinterpret_cast<const uint4*>(w0 + k);
      if (PAIR) v[i] = *reinterpret_cast<const uint4*>(w1 + k);
      y[i] = *reinterpret_cast<const uint4*>(x + k);
    }
#pragma unroll
    for (int i = 0; i < UN; ++i) {
      if (k0 + i * STEP + l16 * PER < n) {
        const unsigned uu[4] = {u[i].x, u[i].y, u[i].z, u[i].w}, yy[4] = {y[i].x, y[i].y, y[i].z, y[i].w};
        const unsigned vv[4] = {PAIR ? v[i].x : 0, PAIR ? v[i].y : 0, PAIR ? v[i].z : 0, PAIR ? v[i].w : 0};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if constexpr (sizeof(T) == 2) {
            const float lo = __uint_as_float(yy[j] << 16), hi = __uint_as_float(yy[j] & 0xFFFF0000u);
            a0[0] += __uint_as_float(uu[j] << 16) * lo;
            a0[1] += __uint_as_float(uu[j] & 0xFFFF0000u) * hi;
            if (PAIR) {
              a1[0] += __uint_as_float(vv[j] << 16) * lo;
              a1[1] += __uint_as_float(vv[j] & 0xFFFF0000u) * hi;
            }
          } else {
            a0[j & 1] += __uint_as_float(uu[j]) * __uint_as_float(yy[j]);
            if (PAIR) a1[j & 1] += __uint_as_float(vv[j]) * __uint_as_float(yy[j]);
          }
        }
      }
    }
  }
  s0 = row16_sum(a0[0] + a0[1]);
  if (PAIR) s1 = row16_sum(a1[0] + a1[1]);
}

constexpr int VC = 4 * NW;        // channels per workgroup of the vector form

// A workgroup's pair and block of VC channels, from a grid of pairs x blocks, or (RUNS) from one dimension of workgroups, which go round-robin over the 8
// XCDs -- each gets a run of units, blocks one after another and all pairs of a block together, so that the pairs of one expert read its rows from one L2.
struct PairUnit { int64_t pair; int block; };
template <bool RUNS> __device__ __forceinline__ PairUnit pair_unit(unsigned pairs, int blocks) {
  if constexpr (!RUNS) return {blockIdx.x, static_cast<int>(blockIdx.y)};
  const unsigned units = pairs * blocks, per = (units + 7) / 8, j = blockIdx.x >> 3, u = (blockIdx.x & 7) * per + j;
  if (j >= per || u >= units) return {0, -1};
  return {u % pairs, static_cast<int>(u / pairs)};
}

template <typename T, bool FAST, bool GATED, bool RUNS>
__global__ __launch_bounds__(NT) void expert_up_vec(const T* __restrict__ h, const T* __restrict__ first, const int* __restrict__ idx,
                                                   const float* __restrict__ scale, T* __restrict__ act, int K, int F, int top, int kind, float limit,
                                                   unsigned pairs) {
  const PairUnit at = pair_unit<RUNS>(pairs, (F + VC - 1) / VC);
  if (at.block < 0) return;
  const int64_t pair = at.pair;
  const int lane = threadIdx.x & 63, f = at.block * VC + 4 * (threadIdx.x >> 6) + (lane >> 4), fc = min(f, F - 1);
  const T* w = first + (static_cast<int64_t>(idx[pair]) * (GATED ? 2 : 1) * F + fc) * K;
  float a, u;
  rows_dot<T, GATED>(w, w + static_cast<int64_t>(F) * K, h + (pair / top) * K, K, lane & 15, a, u);
  const float sc = scale ? scale[pair] : 1.f;
  if ((lane & 15) == 0 && f < F) {
    if constexpr (GATED) a = glu_act<FAST>(sc * a, sc * u, kind, limit, 1.702f);
    else { a = fmaxf(sc * a, 0.f); a *= a; }
    act[pair * F + f] = from_f32<T>(a);
  }
}

template <typename T, bool RUNS>
__global__ __launch_bounds__(NT) void expert_down_vec(const T* __restrict__ act, const T* __restrict__ down, const int* __restrict__ idx, T* __restrict__ y,
                                                     int K, int F, unsigned pairs) {
  const PairUnit at = pair_unit<RUNS>(pairs, (K + VC - 1) / VC);
  if (at.block < 0) return;
  const int64_t pair = at.pair;
  const int lane = threadIdx.x & 63, c = at.block * VC + 4 * (threadIdx.x >> 6) + (lane >> 4), cc = min(c, K - 1);
  float a, unused;
  const T* w = down + (static_cast<int64_t>(idx[pair]) * K + cc) * F;
  rows_dot<T, false>(w, w, act + pair * F, F, lane & 15, a, unused);
  if ((lane & 15) == 0 && c < K) y[pair * K + c] = from_f32<T>(a);
}

// sum_k w[k] * x[k] over this lane's share of n elements; x in LDS (fp32)
template <typename T>
__device__ __forceinline__ float lane_dot(const T* __restrict__ w, const float* __restrict__ x, int n, int lane) {
  float acc = 0.f;
  for (int k = lane; k < n; k += 64) acc += to_f32(w[k]) * x[k];
  return acc;
}

// GATED: first = gate rows over up rows, a wave takes one hidden channel at a time; else first = up rows, a wave takes its two channels of
// the workgroup's FC = 2 NW together.
template <typename T, bool FAST, bool GATED>
__global__ __launch_bounds__(NT) void expert_up_rows(const T* __restrict__ h, const T* __restrict__ first, const int* __restrict__ idx,
                                                    const float* __restrict__ scale, T* __restrict__ act, int K, int F, int top, int kind, float limit) {
  static_assert(FC == 2 * NW, "two hidden channels per wave");
  extern __shared__ float hl[];                     // the row [K]
  const int64_t pair = blockIdx.x;
  const int e = idx[pair];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const T* hr = h + (pair / top) * K;
  for (int k = threadIdx.x; k < K; k += NT) hl[k] = to_f32(hr[k]);
  __syncthreads();
  const T* wg = first + static_cast<int64_t>(e) * (GATED ? 2 : 1) * F * K;
  const float sc = scale ? scale[pair] : 1.f;
  if constexpr (!GATED) {
    const int fa = blockIdx.y * FC + wave, fb = fa + NW;
    if (fa >= F) return;
    float a = lane_dot<T>(wg + static_cast<int64_t>(fa) * K, hl, K, lane);
    float b = lane_dot<T>(wg + static_cast<int64_t>(min(fb, F - 1)) * K, hl, K, lane);
    a = fmaxf(sc * wave_sum(a), 0.f);
    b = fmaxf(sc * wave_sum(b), 0.f);
    if (lane == 0) {
      act[pair * F + fa] = from_f32<T>(a * a);
      if (fb < F) act[pair * F + fb] = from_f32<T>(b * b);
    }
    return;
  }
  const T* wu = wg + static_cast<int64_t>(F) * K;
  const int f_end = min(F, (static_cast<int>(blockIdx.y) + 1) * FC);
  for (int f = blockIdx.y * FC + wave; f < f_end; f += NW) {
    const float ag = sc * wave_sum(lane_dot<T>(wg + static_cast<int64_t>(f) * K, hl, K, lane));
    const float au = sc * wave_sum(lane_dot<T>(wu + static_cast<int64_t>(f) * K, hl, K, lane));
    if (lane == 0) act[pair * F + f] = from_f32<T>(glu_act<FAST>(ag, au, kind, limit, 1.702f));
  }
}

template <typename T>
__global__ __launch_bounds__(NT) void expert_down_rows(const T* __restrict__ act, const T* __restrict__ down, const int* __restrict__ idx,
                                                      T* __restrict__ y, int K, int F) {
  extern __shared__ float al[];                     // the hidden row [F]
  const int64_t pair = blockIdx.x;
  const int e = idx[pair];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int f = threadIdx.x; f < F; f += NT) al[f] = to_f32(act[pair * F + f]);
  __syncthreads();
  const T* wd = down + static_cast<int64_t>(e) * K * F;
  const int c_end = min(K, (static_cast<int>(blockIdx.y) + 1) * KC);
  for (int c = blockIdx.y * KC + wave; c < c_end; c += NW) {
    const float acc = wave_sum(lane_dot<T>(wd + static_cast<int64_t>(c) * F, al, F, lane));
    if (lane == 0) y[pair * K + c] = from_f32<T>(acc);
  }
}

// Where enough pairs meet in an expert for the runs of `pair_unit` to pay.  Grid of pairs x blocks | runs, us: fp32, 8 experts of 3 x 4096 x 2048, 16 pairs 233 | 166, 128
// 1 061 | 698 (an earlier form 945); 128 of 3 x 2048 x 768, 64 pairs 191 | 168, 512 1 170 | 1 060, but 16 49 | 51; 64 of 2 x 2048 x 2048, 16 pairs 89 | 99, 32 180 | 171; bf16, 16 of
// 3 x 1024 x 512, 8 pairs 6.6 | 8.2, 16 12.9 | 9.0, 48 26 | 15; 4 of 3 x 512 x 2048, 4 pairs 9.7 | 9.0, 8 14.3 | 10.2; 64 of 3 x 1024 x 256, 16 pairs 7.1 | 7.6, 32 12.7 | 10.5.
bool pairs_share(int64_t P, int E) { return P >= 2 * static_cast<int64_t>(E) || (P >= 16 && 2 * P >= E); }

template <typename T, bool FAST, bool GATED>
int launch_rows(const gbxm_expert_args& a, hipStream_t s) {
  constexpr int PER = 16 / sizeof(T);
  const bool vec = a.K % PER == 0 && a.F % PER == 0 &&
                   all_aligned(16, static_cast<const T*>(a.first), static_cast<const T*>(a.down), static_cast<const T*>(a.h), static_cast<const T*>(a.ws));
  const int64_t P = a.T * a.top;
  const dim3 gu(P, (a.F + (vec ? VC : FC) - 1) / (vec ? VC : FC)), gd(P, (a.K + KC - 1) / KC);
  static_assert(VC == KC, "one grid for both forms of the second product");
  T* act = static_cast<T*>(a.ws);
  const T *h = static_cast<const T*>(a.h), *first = static_cast<const T*>(a.first), *down = static_cast<const T*>(a.down);
  T* y = static_cast<T*>(a.y);
  if (vec) {
    const auto grid = [](const dim3& g) { return dim3((g.x * g.y + 7) / 8 * 8); };
    if (pairs_share(P, a.E) && P * gu.y < 0x7ffffff0 && P * gd.y < 0x7ffffff0) {
      const unsigned pairs = static_cast<unsigned>(P);
      expert_up_vec<T, FAST, GATED, true><<<grid(gu), NT, 0, s>>>(h, first, a.idx, a.scale, act, a.K, a.F, a.top, a.kind, a.limit, pairs);
      expert_down_vec<T, true><<<grid(gd), NT, 0, s>>>(act, down, a.idx, y, a.K, a.F, pairs);
    } else {
      expert_up_vec<T, FAST, GATED, false><<<gu, NT, 0, s>>>(h, first, a.idx, a.scale, act, a.K, a.F, a.top, a.kind, a.limit, 0);
      expert_down_vec<T, false><<<gd, NT, 0, s>>>(act, down, a.idx, y, a.K, a.F, 0);
    }
  } else {
    expert_up_rows<T, FAST, GATED><<<gu, NT, a.K * sizeof(float), s>>>(h, first, a.idx, a.scale, act, a.K, a.F, a.top, a.kind, a.limit);
    expert_down_rows<T><<<gd, NT, a.F * sizeof(float), s>>>(act, down, a.idx, y, a.K, a.F);
  }
  return after_launch("expert_ff (rows)");
}

template <typename T, bool FAST>
int launch_rows(const gbxm_expert_args& a, hipStream_t s) {
  return a.kind == GBXM_EXPERT_RELU2 ? launch_rows<T, FAST, false>(a, s) : launch_rows<T, FAST, true>(a, s);
}

}  // namespace

int launch_expert_grouped(const gbxm_expert_args& a, hipStream_t s);   // mixers_moe_mfma.hip
size_t expert_grouped_workspace(int64_t T, int K, int F, int E, int top);

}  // namespace gbxm

using namespace gbxm;

extern "C" size_t gbxm_expert_glu_workspace(int64_t T_, int32_t K, int32_t F, int32_t E, int32_t top, int32_t act) {
  const size_t rows = static_cast<size_t>(T_) * top * F * (act == GBXM_BF16 ? 2 : 4);      // the hidden rows of the row kernels
  const size_t grouped = act == GBXM_BF16 ? expert_grouped_workspace(T_, K, F, E, top) : 0;
  return grouped > rows ? grouped : rows;
}

extern "C" int gbxm_expert_glu_grouped(int64_t T_, int32_t K, int32_t F, int32_t E, int32_t top, int32_t act) {
  return act == GBXM_BF16 && expert_grouped_workspace(T_, K, F, E, top) > 0;
}

extern "C" int gbxm_expert_ff(const gbxm_expert_args* a, void* stream) {
  if (!a || !a->h || !a->first || !a->down || !a->idx || !a->y || a->K <= 0 || a->F <= 0 || a->E <= 0 || a->top < 1 || a->top > a->E || a->T < 0 ||
      (a->act != GBXM_BF16 && a->act != GBXM_F32) || (a->kind != GBXM_GLU_SILU && a->kind != GBXM_GLU_CLAMPED_SWISH && a->kind != GBXM_EXPERT_RELU2))
    return fail(GBXM_ERR_INVALID, "expert_ff: bad argument");
  if (a->T == 0) return GBXM_OK;
  if (!a->ws || a->ws_bytes < gbxm_expert_glu_workspace(a->T, a->K, a->F, a->E, a->top, a->act)) return fail(GBXM_ERR_INVALID, "expert_ff: workspace too small");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (a->act == GBXM_BF16) {
    const int rc = launch_expert_grouped(*a, s);
    if (rc != GBXM_ERR_UNSUPPORTED) return rc;
  }
  const int longest = a->K > a->F ? a->K : a->F;
  if (static_cast<size_t>(longest) * sizeof(float) > 64 * 1024) return fail(GBXM_ERR_UNSUPPORTED, "expert_ff: rows of %d channels beyond the row kernels' LDS", longest);
  if (a->T * a->top > 0x7fffffffLL || (a->F + FC - 1) / FC > 65535 || (a->K + KC - 1) / KC > 65535) return fail(GBXM_ERR_UNSUPPORTED, "expert_ff: grid");
  return a->act == GBXM_BF16 ? launch_rows<bf16_t, true>(*a, s) : launch_rows<float, false>(*a, s);
}

extern "C" int gbxm_expert_glu_act(const void* h, const void* gate_up, const void* down, const int32_t* idx, void* y, int64_t T_, int32_t K,
                                   int32_t F, int32_t E, int32_t top, int32_t act, int32_t kind, float limit, void* ws, size_t ws_bytes,
                                   void* stream) {
  if (kind == GBXM_EXPERT_RELU2) return fail(GBXM_ERR_INVALID, "expert_glu: gated experts only");
  const gbxm_expert_args a{h, gate_up, down, idx, nullptr, y, T_, K, F, E, top, act, kind, limit, ws, ws_bytes};
  return gbxm_expert_ff(&a, stream);
}

extern "C" int gbxm_expert_glu(const void* h, const void* gate_up, const void* down, const int32_t* idx, void* y, int64_t T_, int32_t K, int32_t F,
                               int32_t E, int32_t top, int32_t act, void* ws, size_t ws_bytes, void* stream) {
  return gbxm_expert_glu_act(h, gate_up, down, idx, y, T_, K, F, E, top, act, GBXM_GLU_SILU, 0.f, ws, ws_bytes, stream);
}
