// Softmax attention with a sink over a ragged step, and the row kernels around it: head rotations / norms, the append to slot
// tables, the parallel-layer stream update and the feed-forward activation.
//
//   out[t][h] = gate[t][h] * sum_j p_j v_j,   p_j = exp(s_j) / (exp(sink_h) + sum_j exp(s_j)),   s_j = scale <q[t][h], k_j>
// over the keys j <= i of the row's sequence with i - j < window (or, with chunks instead of a window, j in the same chunk of
// positions as i) or j < keep; s_j may carry a factor per query head.  The keys a row sees are two runs of positions,
// [0, min(keep, lo)) and [lo, i] with lo = first_seen(i); the kernels walk them as ONE run of indices (no masked key is
// ever loaded).  Position j of a sequence is read from its slot's table (row j if j < keep, else keep + (j - keep) % ring) when it
// lies before the step, and from the step's own rows otherwise.
//
// sink_rows_kernel: any head sizes, fp32 or bf16, all arithmetic fp32 -- one workgroup per (row, kv head, chunk of its query
// heads, share of the key tiles); scores by a thread per (head, key) of a 64-key tile, running maximum / sum per head in LDS, the
// value sum with a wave per key and the lanes across channels.  A step of few rows splits the key tiles over workgroups; each
// leaves (sum, maximum, denominator) and sink_reduce_kernel joins them in a fixed order, adds the sink and applies the gate.
// The matrix-core kernel for bf16 prompt portions is in mixers_sink_mfma.hip.
#include <algorithm>
#include <climits>
#include <utility>
#include "mixers_mfma.h"

namespace gbxm {
namespace {

constexpr int NT = 256, NW = NT / 64;
constexpr int KT = 64;            // keys per tile
constexpr int RC = 8;             // query heads a workgroup takes at most
constexpr int DCH = 128;          // value channels per lane pass (two per lane)
constexpr int NCH_MAX = 8;        // lane passes: value sizes up to NCH_MAX * DCH (a kernel is compiled for 4 and for 8)

struct SinkGeo {
  int H, G, dk, dv, window, keep, ring, chunk, gate_channels;
  float scale;
  const float* head_scale;
  int64_t out_row;
  int64_t q_row, q_head, k_row, k_head, v_row, v_head, kc_slot, kc_row, kc_head, vc_slot, vc_row, vc_head, gate_row;
};

template <typename T, bool VEC>
__device__ __forceinline__ float dot_row(const float* __restrict__ q, const T* __restrict__ k, int dk) {
  float dot = 0.f;
  if constexpr (VEC) {
    constexpr int PER = 16 / sizeof(T);
    for (int d = 0; d < dk; d += PER) {
      const uint4 raw = *reinterpret_cast<const uint4*>(k + d);
      if constexpr (sizeof(T) == 2) {
        const unsigned u[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          dot += q[d + 2 * i] * __uint_as_float(u[i] << 16);
          dot += q[d + 2 * i + 1] * __uint_as_float(u[i] & 0xFFFF0000u);
        }
      } else {
        dot += q[d] * __uint_as_float(raw.x) + q[d + 1] * __uint_as_float(raw.y) + q[d + 2] * __uint_as_float(raw.z) + q[d + 3] * __uint_as_float(raw.w);
      }
    }
  } else {
    for (int d = 0; d < dk; ++d) dot += q[d] * to_f32(k[d]);
  }
  return dot;
}

template <typename T, bool FAST, bool VEC, int NCH>
__global__ __launch_bounds__(NT) void sink_rows_kernel(const T* __restrict__ q, const T* __restrict__ kn, const T* __restrict__ vn,
                                                      const T* __restrict__ kc, const T* __restrict__ vc, const int* __restrict__ seq,
                                                      const int* __restrict__ tok, T* __restrict__ out, const float* __restrict__ sink,
                                                      const T* __restrict__ gate, SinkGeo g, int rc, int splits, float* __restrict__ partial) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  const T** kptr = reinterpret_cast<const T**>(lds_raw);            // [KT] rows of the tile's keys
  const T** vptr = kptr + KT;                                        // [KT] and values
  float* ql = reinterpret_cast<float*>(vptr + KT);                   // [rc][dk]
  float* gl = ql + rc * g.dk;                                        // [rc][KT] scores, then weights
  float* ml = gl + rc * KT;                                          // [rc] running maximum
  float* ll = ml + rc;                                               // [rc] running denominator
  float* al = ll + rc;                                               // [rc] rescale of this tile
  float* sums = al + rc;                                             // [NW][rc * dv]
  const int64_t t = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int R = g.H / g.G;
  const int chunks = (R + rc - 1) / rc;
  const int kvh = blockIdx.y / chunks, r0 = (blockIdx.y % chunks) * rc;
  const int nr = min(rc, R - r0);                   // query heads of this workgroup: kvh * R + r0 + (0 .. nr-1)
  const int b = tok[2 * t], pos = tok[2 * t + 1];
  const int slot = seq[4 * b], pos0 = seq[4 * b + 1], row0 = seq[4 * b + 3];
  const int head0 = kvh * R + r0;
  for (int i = threadIdx.x; i < nr * g.dk; i += NT) ql[i] = to_f32(q[t * g.q_row + (head0 + i / g.dk) * g.q_head + i % g.dk]);
  if (threadIdx.x < nr) {
    const bool own_sink = sink && splits == 1;      // split key tiles: the sink joins in the reduce
    ml[threadIdx.x] = own_sink ? sink[head0 + threadIdx.x] : -INFINITY;
    ll[threadIdx.x] = own_sink ? 1.f : 0.f;
  }
  float acc[NCH][RC][2];
#pragma unroll
  for (int c = 0; c < NCH; ++c)
#pragma unroll
    for (int r = 0; r < RC; ++r) acc[c][r][0] = acc[c][r][1] = 0.f;
  const bool pair_loads = g.dv % 2 == 0 && VEC;
  // the visible keys as one run of indices: [0, na) are positions 0 .. na-1 (kept first tokens that left the window), the rest lo ..
  const int lo = first_seen(pos, g.window, g.chunk);
  const int na = min(g.keep, lo);
  const int total = na + (pos - lo + 1);
  for (int it = static_cast<int>(blockIdx.z) * KT; it < total; it += KT * splits) {
    __syncthreads();                                // the previous tile's weights and rows have been consumed
    if (threadIdx.x < KT) {
      const int iv = min(it + static_cast<int>(threadIdx.x), total - 1);
      const int j = iv < na ? iv : lo + (iv - na);
      if (j < pos0) {
        const int64_t row = j < g.keep ? j : g.keep + (j - g.keep) % g.ring;
        kptr[threadIdx.x] = kc + slot * g.kc_slot + row * g.kc_row + kvh * g.kc_head;
        vptr[threadIdx.x] = vc + slot * g.vc_slot + row * g.vc_row + kvh * g.vc_head;
      } else {
        const int64_t row = row0 + (j - pos0);
        kptr[threadIdx.x] = kn + row * g.k_row + kvh * g.k_head;
        vptr[threadIdx.x] = vn + row * g.v_row + kvh * g.v_head;
      }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nr * KT; i += NT) {
      const int r = i / KT, jj = i % KT;
      gl[i] = it + jj < total ? dot_row<T, VEC>(ql + r * g.dk, kptr[jj], g.dk) * (g.head_scale ? g.scale * g.head_scale[head0 + r] : g.scale) : -INFINITY;
    }
    __syncthreads();
    for (int r = wave; r < nr; r += NW) {           // a wave per head: the tile's maximum, the weights, their sum
      const float s = gl[r * KT + lane];
      float mx = s;
      mx = wave_max(mx);
      const float m_old = ml[r], m_new = fmaxf(m_old, mx);            // mx is finite: a tile holds at least one key
      const float p = exp_<FAST>(s - m_new);
      gl[r * KT + lane] = p;
      const float ps = wave_sum(p);
      if (lane == 0) {
        const float alpha = exp_<FAST>(m_old - m_new);                // exp(-inf) = 0 at the first tile without a sink
        ml[r] = m_new; ll[r] = ll[r] * alpha + ps; al[r] = alpha;
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RC; ++r)
      if (r < nr) {
        const float alpha = al[r];
#pragma unroll
        for (int c = 0; c < NCH; ++c) { acc[c][r][0] *= alpha; acc[c][r][1] *= alpha; }
      }
    const int nj = min(KT, total - it);
#pragma unroll 4
    for (int jj = wave; jj < nj; jj += NW) {
      const T* vr = vptr[jj];
#pragma unroll
      for (int c = 0; c < NCH; ++c) {
        const int d0 = c * DCH + 2 * lane;
        if (d0 < g.dv) {
          float v0, v1 = 0.f;
          if (pair_loads) {
            if constexpr (sizeof(T) == 2) {
              const unsigned u = *reinterpret_cast<const unsigned*>(vr + d0);
              v0 = __uint_as_float(u << 16); v1 = __uint_as_float(u & 0xFFFF0000u);
            } else {
              const float2 f = *reinterpret_cast<const float2*>(vr + d0);
              v0 = f.x; v1 = f.y;
            }
          } else {
            v0 = to_f32(vr[d0]);
            if (d0 + 1 < g.dv) v1 = to_f32(vr[d0 + 1]);
          }
#pragma unroll
          for (int r = 0; r < RC; ++r)
            if (r < nr) {
              const float p = gl[r * KT + jj];
              acc[c][r][0] += p * v0;
              acc[c][r][1] += p * v1;
            }
        }
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int d0 = c * DCH + 2 * lane;
    if (d0 < g.dv)
#pragma unroll
      for (int r = 0; r < RC; ++r)
        if (r < nr) {
          sums[(wave * rc + r) * g.dv + d0] = acc[c][r][0];
          if (d0 + 1 < g.dv) sums[(wave * rc + r) * g.dv + d0 + 1] = acc[c][r][1];
        }
  }
  __syncthreads();
  if (splits > 1) {
    const int pw = partial_width(g.dv);
    float* prow = partial + ((static_cast<int64_t>(blockIdx.z) * gridDim.x + t) * g.H + head0) * pw;
    for (int i = threadIdx.x; i < nr * g.dv; i += NT) {
      float s = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) s += sums[w * rc * g.dv + i];
      prow[(i / g.dv) * pw + i % g.dv] = s;
    }
    if (threadIdx.x < nr) {
      prow[threadIdx.x * pw + pw - 2] = ml[threadIdx.x];
      prow[threadIdx.x * pw + pw - 1] = ll[threadIdx.x];
    }
    return;
  }
  T* orow = out + t * g.out_row + head0 * g.dv;
  for (int i = threadIdx.x; i < nr * g.dv; i += NT) {
    const int r = i / g.dv;
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) s += sums[w * rc * g.dv + i];
    s /= ll[r];
    if (gate) s *= sigmoid_<FAST>(to_f32(gate[t * g.gate_row + (g.gate_channels ? head0 * g.dv + i : head0 + r)]));
    orow[i] = from_f32<T>(s);
  }
}

// The step's rows on their way into the slot tables; k null: none.
template <typename T> struct SlotRows {
  const T *k, *v;
  T *kc, *vc;
  int64_t k_stride, v_stride;
  int k_width, v_width, keep, ring, fours;
  const int *seq, *tok;
};
template <typename T> SlotRows<T> slot_rows(const gbxm_slot_rows& r, const int32_t* seq, const int32_t* tok, int keep, int ring) {
  const bool fours = (r.k_width | (r.v ? r.v_width : 0)) % 4 == 0 && r.k_stride % 4 == 0 && (!r.v || r.v_stride % 4 == 0) &&
                     all_aligned(4 * sizeof(T), static_cast<const char*>(r.k), static_cast<const char*>(r.v), static_cast<const char*>(r.kcache),
                                 static_cast<const char*>(r.v ? r.vcache : nullptr));
  return {static_cast<const T*>(r.k), static_cast<const T*>(r.v), static_cast<T*>(r.kcache), static_cast<T*>(r.vcache), r.k_stride, r.v_stride,
          r.k_width, r.v ? r.v_width : 0, keep, ring, fours, seq, tok};
}
// A workgroup copies row t, four channels a thread where rows, tables and their strides are in groups of four.
template <typename T, int V> __device__ __forceinline__ void copy_row(const SlotRows<T>& r, int64_t t, int64_t row) {
  struct alignas(V * sizeof(T)) Group { T v[V]; };
  for (int c = threadIdx.x * V; c < r.k_width + r.v_width; c += NT * V)
    *reinterpret_cast<Group*>(c < r.k_width ? r.kc + row * r.k_width + c : r.vc + row * r.v_width + (c - r.k_width)) =
        *reinterpret_cast<const Group*>(c < r.k_width ? r.k + t * r.k_stride + c : r.v + t * r.v_stride + (c - r.k_width));
}
template <typename T> __device__ __forceinline__ void append_row(const SlotRows<T>& r, int64_t t) {
  const int b = r.tok[2 * t], pos = r.tok[2 * t + 1];
  const int slot = r.seq[4 * b], pos0 = r.seq[4 * b + 1], n = r.seq[4 * b + 2];
  if (pos >= r.keep && pos + r.ring < pos0 + n) return;  // a later row of this step takes the same ring row
  const int64_t row = static_cast<int64_t>(slot) * (r.keep + r.ring) + (pos < r.keep + r.ring ? pos : r.keep + (pos - r.keep) % r.ring);
  if (r.fours) copy_row<T, 4>(r, t, row);
  else copy_row<T, 1>(r, t, row);
}

// Joins the key splits' (sum, maximum, denominator), adds the sink, applies the gate; one workgroup per (row, head, 128 channels).  Rows of `partial`
// are partial_width(dv) floats (the sums, padding to a multiple of four, maximum, denominator), so a thread reads four channels at once; eight
// groups of 32 threads take every eighth split, all of it (at most 64) in flight beside the splits' weights -- one trip to memory, where two
// halves of a workgroup for all channels made eight -- and meet in LDS in a fixed order.  Workgroups behind the last head append the step's rows: no query
// reads the tables any more, and a launch of its own costs a step more than the copy (a launch behind | here, us a token: 2 rows, three such layers 328.9 | 322.5).
template <typename T, bool FAST>
__global__ __launch_bounds__(256) void sink_reduce_kernel(const float* __restrict__ partial, T* __restrict__ out, const float* __restrict__ sink,
                                                         const T* __restrict__ gate, int64_t gate_row, int gate_channels, int64_t T_, int H, int dv,
                                                         int splits, int64_t out_row, const SlotRows<T> rows) {
  if (static_cast<int>(blockIdx.y) == H) {
    if (blockIdx.z == 0) append_row(rows, blockIdx.x);
    return;
  }
  __shared__ float wz[64];
  __shared__ float den;
  __shared__ float4 part[8][32];
  const int64_t t = blockIdx.x;
  const int head = blockIdx.y, pw = partial_width(dv), group = threadIdx.x >> 5, q = threadIdx.x & 31, d = blockIdx.z * 128 + 4 * q;
  const int64_t zs = T_ * H * pw;
  const float* p0 = partial + (t * H + head) * pw;
  float4 v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {                                          // (channels past dv inside the last four are padding)
    const int z = group + 8 * i;
    v[i] = z < splits && d < dv ? *reinterpret_cast<const float4*>(p0 + z * zs + d) : float4{0.f, 0.f, 0.f, 0.f};
  }
  if (threadIdx.x < 64) {
    const int z = threadIdx.x;
    const float m = z < splits ? p0[z * zs + pw - 2] : -INFINITY, lz = z < splits ? p0[z * zs + pw - 1] : 0.f;
    float top = wave_max(m);
    if (sink) top = fmaxf(top, sink[head]);
    const float w = z < splits ? exp_<FAST>(m - top) : 0.f;
    wz[z] = w;
    const float l = wave_sum(z < splits ? w * lz : 0.f);
    if (z == 0) den = l + (sink ? exp_<FAST>(sink[head] - top) : 0.f);
  }
  __syncthreads();
  float4 s = float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 8; ++i)
    if (group + 8 * i < splits) {
      const float w = wz[group + 8 * i];
      s.x += w * v[i].x; s.y += w * v[i].y; s.z += w * v[i].z; s.w += w * v[i].w;
    }
  part[group][q] = s;
  __syncthreads();
  if (group || d >= dv) return;
#pragma unroll
  for (int i = 1; i < 8; ++i) {
    const float4 u = part[i][q];
    s.x += u.x; s.y += u.y; s.z += u.z; s.w += u.w;
  }
  const float f = (gate && !gate_channels ? sigmoid_<FAST>(to_f32(gate[t * gate_row + head])) : 1.f) / den;
  const float r[4] = {s.x * f, s.y * f, s.z * f, s.w * f};
  for (int c = 0; c < 4 && d + c < dv; ++c)
    out[t * out_row + head * dv + d + c] = from_f32<T>(gate && gate_channels ? r[c] * sigmoid_<FAST>(to_f32(gate[t * gate_row + head * dv + d + c])) : r[c]);
}

// `rows`: appended in the same launch.
template <typename T, bool FAST>
int launch_reduce(const gbxm_sink_attn_args& a, int splits, int64_t out_row, const gbxm_slot_rows* rows, hipStream_t s) {
  const SlotRows<T> r = rows ? slot_rows<T>(*rows, a.seq, a.tok, a.keep, a.ring) : SlotRows<T>{};
  sink_reduce_kernel<T, FAST><<<dim3(a.T, a.H + (rows ? 1 : 0), (a.dv + 127) / 128), 256, 0, s>>>(
      static_cast<const float*>(a.partial), static_cast<T*>(a.out), a.sink, static_cast<const T*>(a.gate), a.gate_row, a.gate_channels, a.T, a.H, a.dv, splits, out_row, r);
  return after_launch("sink_attention (join of key splits)");
}

// Launches that join key splits take `rows` with them and clear it for the caller.
template <typename T, bool FAST>
int launch_rows(const gbxm_sink_attn_args& a, const SinkGeo& g, int rc, int chunks, size_t lds, const gbxm_slot_rows*& rows, hipStream_t s) {
  constexpr int PER = 16 / sizeof(T);
  auto al = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  bool vec = a.dk % PER == 0 && a.k_row % PER == 0 && a.k_head % PER == 0 && al(a.k_new) && a.v_row % 2 == 0 && a.v_head % 2 == 0 &&
             reinterpret_cast<uintptr_t>(a.v_new) % 8 == 0;
  if (a.kcache)
    vec = vec && a.kc_slot % PER == 0 && a.kc_row % PER == 0 && a.kc_head % PER == 0 && al(a.kcache) && a.vc_slot % 2 == 0 && a.vc_row % 2 == 0 &&
          a.vc_head % 2 == 0 && reinterpret_cast<uintptr_t>(a.vcache) % 8 == 0;
  int splits = 1;
  const int64_t groups = a.T * a.G * chunks;
  if (a.partial && a.partial_splits > 1 && groups < 256) {
    splits = static_cast<int>(std::min<int64_t>(std::min<int64_t>(512 / groups, 64), a.partial_splits));
    if (splits < 2) splits = 1;
  }
  const dim3 grid(a.T, a.G * chunks, splits);
  const T* q = static_cast<const T*>(a.q);
  const T* kn = static_cast<const T*>(a.k_new);
  const T* vn = static_cast<const T*>(a.v_new);
  const T* kc = static_cast<const T*>(a.kcache);
  const T* vc = static_cast<const T*>(a.vcache);
  const T* gate = static_cast<const T*>(a.gate);
  T* out = static_cast<T*>(a.out);
  float* part = static_cast<float*>(a.partial);
  auto go = [&](auto kernel) { kernel<<<grid, NT, lds, s>>>(q, kn, vn, kc, vc, a.seq, a.tok, out, a.sink, gate, g, rc, splits, part); };
  if (a.dv <= 4 * DCH) {
    if (vec) go(sink_rows_kernel<T, FAST, true, 4>);
    else go(sink_rows_kernel<T, FAST, false, 4>);
  } else {
    if (vec) go(sink_rows_kernel<T, FAST, true, NCH_MAX>);
    else go(sink_rows_kernel<T, FAST, false, NCH_MAX>);
  }
  if (splits > 1) {
    const int rc2 = after_launch("sink_attention (rows)");
    return rc2 != GBXM_OK ? rc2 : launch_reduce<T, FAST>(a, splits, g.out_row, std::exchange(rows, nullptr), s);
  }
  return after_launch("sink_attention (rows)");
}

// ------------------------------------------------------------------------------------------------ rotations and norms of heads
struct Segments {
  gbxm_head_segment s[GBXM_MAX_SEGMENTS];
};

// What a segment needs: nothing but rotations touches the rotated channels only, pair by pair; a plain norm of ONE head (a row part, of any
// length) is a workgroup's sum; everything else stages heads in LDS.
enum { SEG_STAGED = 0, SEG_PAIRS = 1, SEG_ROW_NORM = 2 };
__host__ __device__ __forceinline__ int segment_form(const gbxm_head_segment& g) {
  if (g.norm == 0) return SEG_PAIRS;
  return g.heads == 1 && g.rot_dims == 0 ? SEG_ROW_NORM : SEG_STAGED;
}

// PV neighbouring pairs of a head: (u, w) -> (u cos - w sin, w cos + u sin), channels p[i], p[half + i] or p[2i], p[2i + 1].
template <typename T, int PV>
__device__ __forceinline__ void turn_pairs(T* __restrict__ p, int half, bool interleaved, const float* __restrict__ cs, const float* __restrict__ sn) {
  float u[PV], w[PV];
  if (interleaved) {
    float v[2 * PV];
    if constexpr (PV == 1) {
      v[0] = to_f32(p[0]); v[1] = to_f32(p[1]);
    } else {
      Lanes<T, 4>::load(p, v);
      Lanes<T, 4>::load(p + 4, v + 4);
    }
#pragma unroll
    for (int i = 0; i < PV; ++i) { u[i] = v[2 * i]; w[i] = v[2 * i + 1]; }
  } else {
    Lanes<T, PV>::load(p, u);
    Lanes<T, PV>::load(p + half, w);
  }
  float a[PV], b[PV];
#pragma unroll
  for (int i = 0; i < PV; ++i) {
    a[i] = u[i] * cs[i] - w[i] * sn[i];
    b[i] = w[i] * cs[i] + u[i] * sn[i];
  }
  if (interleaved) {
    float v[2 * PV];
#pragma unroll
    for (int i = 0; i < PV; ++i) { v[2 * i] = a[i]; v[2 * i + 1] = b[i]; }
    if constexpr (PV == 1) {
      p[0] = from_f32<T>(v[0]); p[1] = from_f32<T>(v[1]);
    } else {
      Lanes<T, 4>::store(p, v);
      Lanes<T, 4>::store(p + 4, v + 4);
    }
  } else {
    Lanes<T, PV>::store(p, a);
    Lanes<T, PV>::store(p + half, b);
  }
}

// p[0 .. n) -> rms_norm(p) (* w), by the whole workgroup; V channels a thread keeps up to ZN groups of between statistic and result.
template <typename T, int V>
__device__ __forceinline__ void row_norm(T* __restrict__ p, int n, const float* __restrict__ w, float eps, float* red) {
  constexpr int ZN = 4;
  float z[ZN][V];
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < ZN; ++j) {
    const int c = (threadIdx.x + j * NT) * V;
    if (c < n) {
      Lanes<T, V>::load(p + c, z[j]);
#pragma unroll
      for (int i = 0; i < V; ++i) ss += z[j][i] * z[j][i];
    }
  }
  for (int c = (threadIdx.x + ZN * NT) * V; c < n; c += NT * V) {
    float v[V];
    Lanes<T, V>::load(p + c, v);
#pragma unroll
    for (int i = 0; i < V; ++i) ss += v[i] * v[i];
  }
  ss = block_sum<NW>(ss, red);
  const float r = 1.f / sqrtf(ss / n + eps);
  auto put = [&](int c, float* v) {
    if (w) {
      float g[V];
      Lanes<float, V>::load(w + c, g);
#pragma unroll
      for (int i = 0; i < V; ++i) v[i] *= g[i];
    }
#pragma unroll
    for (int i = 0; i < V; ++i) v[i] *= r;
    Lanes<T, V>::store(p + c, v);
  };
#pragma unroll
  for (int j = 0; j < ZN; ++j) {
    const int c = (threadIdx.x + j * NT) * V;
    if (c < n) put(c, z[j]);
  }
  for (int c = (threadIdx.x + ZN * NT) * V; c < n; c += NT * V) {
    float v[V];
    Lanes<T, V>::load(p + c, v);
    put(c, v);
  }
}

// One workgroup per (row, segment).  A staged segment: its waves take the heads four at a time.  A head is staged in LDS as fp32, every
// lane forms its rotated channels from there (its own and the partner of the pair), the statistic is a wave sum.  ``vec``: a bit per
// segment whose channels and row starts lie on the vector grid.
template <typename T>
__global__ __launch_bounds__(NT) void rotate_norm_kernel(T* __restrict__ rows, int64_t stride, const int* __restrict__ positions, int64_t pos_stride,
                                                        Segments segs, float eps, int max_dim, int max_half, unsigned vec) {
  extern __shared__ float head_lds[];               // cos [max_half], sin [max_half], then [NW][2][max_dim]
  __shared__ float red[NW];
  const gbxm_head_segment sg = segs.s[blockIdx.y];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int form = segment_form(sg);
  if (form == SEG_ROW_NORM) {
    T* p = rows + blockIdx.x * stride + sg.offset;
    const float* w = (sg.norm & 1) ? nullptr : sg.weight;
    if ((vec >> blockIdx.y) & 1) row_norm<T, 4>(p, sg.head_dim, w, eps, red);
    else row_norm<T, 1>(p, sg.head_dim, w, eps, red);
    return;
  }
  float* cs_t = head_lds;
  float* sn_t = cs_t + max_half;
  float* in = sn_t + max_half + wave * 2 * max_dim;
  float* turned = in + max_dim;
  const float pos = static_cast<float>(positions[blockIdx.x * pos_stride]);
  const int half = sg.rot_dims / 2;
  for (int i = threadIdx.x; i < half; i += NT) {    // the row's angles once, for all heads of the segment
    float sn, cs;
    sincosf(pos * sg.freq[i], &sn, &cs);
    cs_t[i] = cs * sg.mult;
    sn_t[i] = sn * sg.mult * sg.sign;
  }
  if (form == SEG_PAIRS) {
    __syncthreads();
    T* p0 = rows + blockIdx.x * stride + sg.offset + sg.rot_offset;
    if ((vec >> blockIdx.y) & 1) {
      const int per = half / 4;
      for (int i = threadIdx.x; i < sg.heads * per; i += NT) {
        const int c = (i % per) * 4;
        turn_pairs<T, 4>(p0 + static_cast<int64_t>(i / per) * sg.head_dim + (sg.interleaved ? 2 * c : c), half, sg.interleaved, cs_t + c, sn_t + c);
      }
    } else {
      for (int i = threadIdx.x; i < sg.heads * half; i += NT) {
        const int c = i % half;
        turn_pairs<T, 1>(p0 + static_cast<int64_t>(i / half) * sg.head_dim + (sg.interleaved ? 2 * c : c), half, sg.interleaved, cs_t + c, sn_t + c);
      }
    }
    return;
  }
  for (int h0 = 0; h0 < sg.heads; h0 += NW) {
    const int head = h0 + wave;
    const bool live = head < sg.heads;
    T* p = rows + blockIdx.x * stride + sg.offset + static_cast<int64_t>(live ? head : 0) * sg.head_dim;
    __syncthreads();
    if (live)
      for (int c = lane; c < sg.head_dim; c += 64) in[c] = to_f32(p[c]);
    __syncthreads();
    if (sg.norm >= 3) {                             // norm before the rotation: the staged head is replaced by its normed image
      if (live) {
        float s0 = 0.f;
        for (int c = lane; c < sg.head_dim; c += 64) s0 += in[c] * in[c];
        const float r0 = 1.f / sqrtf(wave_sum(s0) / sg.head_dim + eps);
        for (int c = lane; c < sg.head_dim; c += 64) in[c] = in[c] * r0 * (sg.norm == 4 ? sg.weight[c] : 1.f);
      }
      __syncthreads();
    }
    if (!live) continue;
    float ss = 0.f;
    for (int c = lane; c < sg.head_dim; c += 64) {
      float v = in[c];
      const int idx = c - sg.rot_offset;
      if (idx >= 0 && idx < sg.rot_dims) {
        int i, other;
        bool first;
        if (sg.interleaved) { i = idx >> 1; first = !(idx & 1); other = first ? c + 1 : c - 1; }
        else { first = idx < half; i = first ? idx : idx - half; other = first ? c + half : c - half; }
        const float sn = sn_t[i], cs = cs_t[i];
        // (u, w) -> (u cos - w sin, w cos + u sin)
        v = first ? v * cs - in[other] * sn : v * cs + in[other] * sn;
      }
      turned[c] = v;
      ss += v * v;
    }
    float r = 1.f;
    if (sg.norm == 1 || sg.norm == 2) r = 1.f / sqrtf(wave_sum(ss) / sg.head_dim + eps);
    for (int c = lane; c < sg.head_dim; c += 64) {
      float v = turned[c] * r;
      if (sg.norm == 2) v *= sg.weight[c];
      p[c] = from_f32<T>(v);
    }
  }
}

template <typename T>
__global__ __launch_bounds__(NT) void stream_add_kernel(float* __restrict__ x, const T* __restrict__ a, const T* __restrict__ b, int64_t n) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * NT + threadIdx.x;
  if (i >= n) return;
  float y = to_f32(a[i]);
  if (b) y += to_f32(b[i]);
  x[i] += y;
}

// x += a (+ b), then h = rms_norm(x) * w in the activation dtype: a parallel layer's stream update and the next layer's norm.
template <typename T>
__global__ __launch_bounds__(NT) void stream_add_norm_kernel(float* __restrict__ x, const T* __restrict__ a, const T* __restrict__ b,
                                                            const float* __restrict__ w, T* __restrict__ h, int width, float eps) {
  __shared__ float red[NW];
  const int64_t t = blockIdx.x;
  float* xr = x + t * width;
  float ss = 0.f;
  for (int c = threadIdx.x; c < width; c += NT) {
    float y = to_f32(a[t * width + c]);
    if (b) y += to_f32(b[t * width + c]);
    const float v = xr[c] + y;
    xr[c] = v;
    ss += v * v;
  }
  ss = block_sum<NW>(ss, red);
  const float r = 1.f / sqrtf(ss / width + eps);
  for (int c = threadIdx.x; c < width; c += NT) h[t * width + c] = from_f32<T>(xr[c] * r * w[c]);      // (each thread re-reads what it wrote)
}

// out[t][h][j] = sum_i in[t][h][i] w[h][i][j] for j < n_out (times a gate's sigmoid), then out[t][h][n_out + c] = in[t][h][n_in + c] for
// c < n_tail (copied or turned): a small matrix of its own per head, applied to few rows (single-row steps): one workgroup per (row, head),
// the head's input in LDS, threads across the outputs (coalesced reads of w), fp32 sums.
template <typename T, bool FAST>
struct HeadOut {
  const gbxm_head_project_args& a;
  int64_t row;
  const T* ip;
  T* op;
  const T* gp;                                     // this row and head's gates, or null
  __device__ __forceinline__ HeadOut(const gbxm_head_project_args& a_, int64_t row_) : a(a_), row(row_) {
    ip = static_cast<const T*>(a.in) + row * a.in_row + blockIdx.y * a.in_head;
    op = static_cast<T*>(a.out) + row * a.out_row + blockIdx.y * a.out_head;
    gp = a.gate ? static_cast<const T*>(a.gate) + row * a.gate_row + static_cast<int64_t>(blockIdx.y) * a.n_out : nullptr;
  }
  __device__ __forceinline__ void put(int j, float s) const { op[j] = from_f32<T>(gp ? s * sigmoid_<FAST>(to_f32(gp[j])) : s); }
  __device__ __forceinline__ void tail() const {
    if (!a.freq) {
      for (int c = threadIdx.x; c < a.n_tail; c += blockDim.x) op[a.n_out + c] = ip[a.n_in + c];
      return;
    }
    const int half = a.n_tail / 2;
    const float pos = static_cast<float>(a.positions[row * a.pos_stride]);
    for (int i = threadIdx.x; i < half; i += blockDim.x) {
      const int c0 = a.interleaved ? 2 * i : i, c1 = a.interleaved ? 2 * i + 1 : i + half;
      float sn, cs;
      sincosf(pos * a.freq[i], &sn, &cs);
      sn *= a.mult; cs *= a.mult;
      const float u = to_f32(ip[a.n_in + c0]), w = to_f32(ip[a.n_in + c1]);
      op[a.n_out + c0] = from_f32<T>(u * cs - w * sn);
      op[a.n_out + c1] = from_f32<T>(w * cs + u * sn);
    }
  }
};

template <typename T, bool FAST>
__global__ __launch_bounds__(NT) void head_project_kernel(const gbxm_head_project_args a) {
  extern __shared__ float xin[];                   // [n_in]
  const HeadOut<T, FAST> o(a, blockIdx.x);
  const T* ip = o.ip;
  const int n_in = a.n_in, n_out = a.n_out;
  const T* wp = static_cast<const T*>(a.w) + static_cast<int64_t>(blockIdx.y) * n_in * n_out;
  for (int i = threadIdx.x; i < n_in; i += NT) xin[i] = to_f32(ip[i]);
  __syncthreads();
  for (int j = threadIdx.x; j < n_out; j += NT) {
    float s4[4] = {0.f, 0.f, 0.f, 0.f};
    int i = 0;
    for (; i + 4 <= n_in; i += 4) {
#pragma unroll
      for (int u = 0; u < 4; ++u) s4[u] += xin[i + u] * to_f32(wp[static_cast<int64_t>(i + u) * n_out + j]);
    }
    for (; i < n_in; ++i) s4[i & 3] += xin[i] * to_f32(wp[static_cast<int64_t>(i) * n_out + j]);
    o.put(j, (s4[0] + s4[1]) + (s4[2] + s4[3]));
  }
  o.tail();
}

// The same with 16-byte loads of w, a workgroup per (row, head, JC runs of PER outputs): a thread owns a run and every IS-th input channel (IS = 256 / JC), eight of
// them in flight, the first ones asked for before the row is parked in LDS.  An output is 32 sums -- sum m over the channels m, m + 32, ... in turn -- which meet by
// halves, m and m + 16, then m and m + 8, and so on: in a thread's registers, across the waves in LDS, within a wave.  The same sums in the same order whatever JC,
// so a row does not depend on how many others the step has.  Channels past the last one are zeros on either side: no test in the loop.  Bound by the trip to memory
// while rows are few, then by the weights' way from L2.  Many rows go two a workgroup (ROWS), which halves that way.  A workgroup a (row, head), sums in its own order | that,
// and outputs cut into runs with sums in an order of the step's below 256 rows times heads | this, us, bf16, 16 heads: 128 -> 512 channels, 2 rows 5.0 | 3.5 | 3.0, 15 rows 5.2 | 5.5 |
// 4.0, 64 rows 8.5 | 8.5 | 8.4, 512 rows 45 | 46 | 42; 512 -> 128, 2 rows 5.0 | 4.1 | 3.4, 15 rows 5.2 | 5.8 | 4.1, 64 rows 8.5 | 8.4 | 6.8, 512 rows 45 | 44 | 30; 192 -> 1 024, 8 rows
// 12.1 | 18.3 | 9.9; fp32, 512 -> 128, 15 rows 7.1 | 10.8 | 5.5.  128 heads of 128 -> 512, 32 rows, are the one size found slower: 28 | 28 | 32.  Sums two at a time in few registers, 16 sums,
// 32 channels in flight a thread: slower at few rows or at many.
template <typename T, bool FAST, int JC, int ROWS>
__global__ __launch_bounds__(NT) void head_project_runs_kernel(const gbxm_head_project_args a, int own_tail) {
  constexpr int PER = 16 / sizeof(T), IS = NT / JC, SUMS = 32 / IS, PART = PER / NW;
  extern __shared__ float xin[];                   // [ROWS][n_in, in whole steps of 8 IS]
  __shared__ __attribute__((aligned(16))) float red[NW][NW][64][PART];
  const int64_t row0 = static_cast<int64_t>(blockIdx.x) * ROWS;
  const int n_in = a.n_in, n_out = a.n_out, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, j0 = blockIdx.z * JC * PER;
  if (j0 >= n_out) {                               // (a workgroup of its own copies or turns the tail)
    HeadOut<T, FAST>(a, row0).tail();
    return;
  }
  const int jc = tid & (JC - 1), first = tid / JC, bytes = n_out * static_cast<int>(sizeof(T)), steps = (n_in + 8 * IS - 1) / (8 * IS), padded = steps * 8 * IS;
  const T* w = static_cast<const T*>(a.w) + static_cast<int64_t>(blockIdx.y) * n_in * n_out;
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(w), 0, n_in * bytes, 0x00020000);
  int at = first * bytes + min(j0 + jc * PER, n_out - PER) * static_cast<int>(sizeof(T));
  u32x4 raw[8];
  auto load = [&]() {
#pragma unroll
    for (int k = 0; k < 8; ++k) raw[k] = __builtin_amdgcn_raw_buffer_load_b128(rw, at + k * IS * bytes, 0, 0);
    at += 8 * IS * bytes;
  };
  load();
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {                 // (a row behind the last one is the last one again; nobody writes it)
    const T* ip = HeadOut<T, FAST>(a, min(row0 + r, a.T - 1)).ip;
    for (int i = tid; i < padded; i += NT) xin[r * padded + i] = i < n_in ? to_f32(ip[i]) : 0.f;
  }
  __syncthreads();
  float acc[ROWS][SUMS][PER];
#pragma unroll
  for (int r = 0; r < ROWS; ++r)
#pragma unroll
    for (int c = 0; c < SUMS; ++c)
#pragma unroll
      for (int u = 0; u < PER; ++u) acc[r][c][u] = 0.f;
  const float* xp = xin + first;
  for (int t = 0; t < steps; ++t, xp += 8 * IS) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const float x = xp[r * padded + k * IS];
        float* to = acc[r][k % SUMS];
        if constexpr (sizeof(T) == 2) {
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            to[2 * u] += x * __uint_as_float(raw[k][u] << 16);
            to[2 * u + 1] += x * __uint_as_float(raw[k][u] & 0xFFFF0000u);
          }
        } else {
#pragma unroll
          for (int u = 0; u < 4; ++u) to[u] += x * __uint_as_float(raw[k][u]);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);             // (hoisted among the products, loads cost a wave a SIMD)
    if (t + 1 < steps) load();
  }
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    if (row0 + r >= a.T) break;
    const HeadOut<T, FAST> o(a, row0 + r);
#pragma unroll
    for (int c = SUMS / 2; c > 0; c /= 2)
#pragma unroll
      for (int k = 0; k < c; ++k)
#pragma unroll
        for (int u = 0; u < PER; ++u) acc[r][k][u] += acc[r][k + c][u];
    // wave w finishes the outputs w PART .. w PART + PART - 1 of every run
    if (r > 0) __syncthreads();
#pragma unroll
    for (int v = 0; v < NW; ++v)
#pragma unroll
      for (int u = 0; u < PART; ++u) red[v][wave][lane][u] = acc[r][0][v * PART + u];
    __syncthreads();
    float s[PART];
#pragma unroll
    for (int u = 0; u < PART; ++u) {
      s[u] = (red[wave][0][lane][u] + red[wave][2][lane][u]) + (red[wave][1][lane][u] + red[wave][3][lane][u]);
      if constexpr (JC <= 32) s[u] = lanes_apart_sum<32>(s[u]);
      if constexpr (JC <= 16) s[u] = lanes_apart_sum<16>(s[u]);
      if constexpr (JC <= 8) s[u] = lanes_apart_sum<8>(s[u]);
    }
    if (lane < JC && j0 + jc * PER < n_out) {
#pragma unroll
      for (int u = 0; u < PART; ++u) o.put(j0 + jc * PER + wave * PART + u, s[u]);
    }
    if (!own_tail && blockIdx.z == gridDim.z - 1) o.tail();
  }
}

// rows times heads from which a workgroup takes two rows.  One | two, us, bf16, 16 heads, 32 | 64 rows: 128 -> 512 5.4 | 9.2 against 5.5 | 8.4, 512 -> 128 5.2 | 7.6 against 5.6 | 6.8
constexpr int64_t PAIRS_FROM = 1024;

template <typename T, bool FAST>
int launch_head_project(const gbxm_head_project_args& a, hipStream_t s) {
  constexpr int PER = 16 / sizeof(T);
  // runs of outputs a workgroup takes: fewer while that leaves CUs without one and lines of 128 bytes whole
  const int64_t units = a.T * a.H;
  const auto cuts = [&](int runs) { return (a.n_out + runs * PER - 1) / (runs * PER); };
  const bool pairs = units >= PAIRS_FROM && a.n_in <= 4096;
  int runs = pairs ? 32 : 64;
  while (runs > 8 && (runs / 2 * PER >= a.n_out || units * cuts(runs) < 256)) runs /= 2;
  const int own_tail = a.n_tail > 0 && units < 256, step = 8 * NT / runs;
  const dim3 grid(pairs ? (a.T + 1) / 2 : a.T, a.H, cuts(runs) + own_tail);
  const size_t lds = (a.n_in + step - 1) / step * step * sizeof(float) * (pairs ? 2 : 1);
#define GBXM_RUNS(JC_)                                                                                       \
  do {                                                                                                       \
    if (pairs) head_project_runs_kernel<T, FAST, JC_, 2><<<grid, NT, lds, s>>>(a, own_tail);                 \
    else head_project_runs_kernel<T, FAST, JC_, 1><<<grid, NT, lds, s>>>(a, own_tail);                       \
  } while (0)
  if (runs == 64) head_project_runs_kernel<T, FAST, 64, 1><<<grid, NT, lds, s>>>(a, own_tail);
  else if (runs == 32) GBXM_RUNS(32);
  else if (runs == 16) GBXM_RUNS(16);
  else GBXM_RUNS(8);
#undef GBXM_RUNS
  return after_launch("head_project");
}

__device__ __forceinline__ float activation(float v, int kind) {
  if (kind == GBXM_ACT_RELU2) { const float r = fmaxf(v, 0.f); return r * r; }
  return 0.5f * v * (1.f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v)));
}

template <typename T>
__global__ __launch_bounds__(NT) void activate_kernel(T* __restrict__ z, int64_t n, int kind) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * NT + threadIdx.x;
  if (i >= n) return;
  z[i] = from_f32<T>(activation(to_f32(z[i]), kind));
}

// 16 bytes per thread (n a multiple of the vector, base 16-byte aligned)
template <typename T>
__global__ __launch_bounds__(NT) void activate_vec_kernel(T* __restrict__ z, int64_t n_vec, int kind) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * NT + threadIdx.x;
  if (i >= n_vec) return;
  uint4* p = reinterpret_cast<uint4*>(z) + i;
  uint4 raw = *p;
  unsigned u[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if constexpr (sizeof(T) == 2) {
      const float lo = activation(__uint_as_float(u[k] << 16), kind), hi = activation(__uint_as_float(u[k] & 0xFFFF0000u), kind);
      u[k] = static_cast<unsigned>(f32_to_bf16(lo)) | (static_cast<unsigned>(f32_to_bf16(hi)) << 16);
    } else {
      u[k] = __float_as_uint(activation(__uint_as_float(u[k]), kind));
    }
  }
  *p = uint4{u[0], u[1], u[2], u[3]};
}

// grid (rows)
template <typename T>
__global__ __launch_bounds__(NT) void slot_append_kernel(const SlotRows<T> r) { append_row(r, blockIdx.x); }

bool act_ok(int act) { return act == GBXM_BF16 || act == GBXM_F32; }

}  // namespace

int launch_sink_tiles(const gbxm_sink_attn_args& a, hipStream_t s);     // mixers_sink_mfma.hip; GBXM_ERR_UNSUPPORTED: not its shape
int launch_sink_group(const gbxm_sink_attn_args& a, const gbxm_slot_rows*& rows, hipStream_t s);     // the same for steps of single rows
bool sink_tiles_shape(int dk, int dv);

int launch_sink_reduce(const gbxm_sink_attn_args& a, int splits, const gbxm_slot_rows* rows, hipStream_t s) {
  return launch_reduce<bf16_t, true>(a, splits, a.out_row > 0 ? a.out_row : static_cast<int64_t>(a.H) * a.dv, rows, s);
}

}  // namespace gbxm

using namespace gbxm;

#define GBXM_DISPATCH(act, CALL)              \
  do {                                        \
    if ((act) == GBXM_BF16) { using T = bf16_t; CALL; } else { using T = float; CALL; } \
  } while (0)

extern "C" {

int gbxm_stream_add(float* x, const void* a, const void* b, int64_t n, int32_t act, void* stream) {
  if (!act_ok(act) || !x || !a || n < 0) return fail(GBXM_ERR_INVALID, "stream_add: bad argument");
  if (n == 0) return GBXM_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  GBXM_DISPATCH(act, (stream_add_kernel<T><<<dim3((n + NT - 1) / NT), NT, 0, s>>>(x, static_cast<const T*>(a), static_cast<const T*>(b), n)));
  return after_launch("stream_add");
}

int gbxm_stream_add_norm(float* x, const void* a, const void* b, const float* w, void* h, int64_t T_, int32_t width, float eps, int32_t act,
                         void* stream) {
  if (!act_ok(act) || !x || !a || !w || !h || T_ < 0 || width <= 0) return fail(GBXM_ERR_INVALID, "stream_add_norm: bad argument");
  if (T_ == 0) return GBXM_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  GBXM_DISPATCH(act, (stream_add_norm_kernel<T><<<dim3(T_), NT, 0, s>>>(x, static_cast<const T*>(a), static_cast<const T*>(b), w, static_cast<T*>(h),
                                                                          width, eps)));
  return after_launch("stream_add_norm");
}

int gbxm_head_project(const gbxm_head_project_args* a, void* stream) {
  if (!a || !act_ok(a->act) || !a->in || !a->w || !a->out || a->T < 0 || a->H < 1 || a->H > 65535 || a->n_in < 1 || a->n_out < 1 || a->n_tail < 0 ||
      (a->freq && (!a->positions || a->n_tail % 2)) || (a->gate && a->gate_row < static_cast<int64_t>(a->H) * a->n_out))
    return fail(GBXM_ERR_INVALID, "head_project: bad argument");
  if (a->n_in > 12 * 1024) return fail(GBXM_ERR_UNSUPPORTED, "head_project: %d input channels per head", a->n_in);
  if (a->T == 0) return GBXM_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int per = a->act == GBXM_BF16 ? 8 : 4;
  const bool near = static_cast<int64_t>(a->n_in + 256) * a->n_out < (1 << 29);      // (a head's matrix, and a step beyond it, by 32-bit byte offsets)
  if (a->n_out % per == 0 && near && reinterpret_cast<uintptr_t>(a->w) % 16 == 0)
    return a->act == GBXM_BF16 ? launch_head_project<bf16_t, true>(*a, s) : launch_head_project<float, false>(*a, s);
  const dim3 grid(a->T, a->H);
  if (a->act == GBXM_BF16) head_project_kernel<bf16_t, true><<<grid, NT, a->n_in * sizeof(float), s>>>(*a);
  else head_project_kernel<float, false><<<grid, NT, a->n_in * sizeof(float), s>>>(*a);
  return after_launch("head_project");
}

int gbxm_activate(void* z, int64_t n, int32_t kind, int32_t act, void* stream) {
  if (!act_ok(act) || !z || n < 0 || (kind != GBXM_ACT_RELU2 && kind != GBXM_ACT_GELU_TANH)) return fail(GBXM_ERR_INVALID, "activate: bad argument");
  if (n == 0) return GBXM_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int per = act == GBXM_BF16 ? 8 : 4;
  if (n % per == 0 && reinterpret_cast<uintptr_t>(z) % 16 == 0) {
    const int64_t nv = n / per;
    GBXM_DISPATCH(act, (activate_vec_kernel<T><<<dim3((nv + NT - 1) / NT), NT, 0, s>>>(static_cast<T*>(z), nv, kind)));
    return after_launch("activate");
  }
  GBXM_DISPATCH(act, (activate_kernel<T><<<dim3((n + NT - 1) / NT), NT, 0, s>>>(static_cast<T*>(z), n, kind)));
  return after_launch("activate");
}

int gbxm_rotate_norm_heads(void* rows, int64_t T_, int64_t row_stride, const int32_t* positions, int64_t pos_stride, const gbxm_head_segment* segs,
                           int32_t n_segs, float eps, int32_t act, void* stream) {
  if (!act_ok(act) || !rows || !positions || !segs || n_segs < 1 || n_segs > GBXM_MAX_SEGMENTS || T_ < 0)
    return fail(GBXM_ERR_INVALID, "rotate_norm_heads: bad argument");
  Segments sg{};
  int max_dim = 0, max_half = 0;
  unsigned vec = 0;
  for (int i = 0; i < n_segs; ++i) {
    const gbxm_head_segment& g = segs[i];
    if (g.offset < 0 || g.heads < 1 || g.head_dim < 1 || g.offset + static_cast<int64_t>(g.heads) * g.head_dim > row_stride || g.rot_dims < 0 ||
        g.rot_dims % 2 || g.rot_offset < 0 || g.rot_offset + g.rot_dims > g.head_dim || (g.rot_dims && !g.freq) || g.norm < 0 || g.norm > 4 ||
        ((g.norm == 2 || g.norm == 4) && !g.weight))
      return fail(GBXM_ERR_INVALID, "rotate_norm_heads: segment %d does not fit its rows", i);
    sg.s[i] = g;
    const int form = segment_form(g);
    if (form == SEG_STAGED) max_dim = std::max(max_dim, g.head_dim);
    max_half = std::max(max_half, g.rot_dims / 2);
    // groups of four channels (pairs: of four pairs) at 8-byte (bf16) or 16-byte (fp32) addresses
    const bool base = reinterpret_cast<uintptr_t>(rows) % (act == GBXM_BF16 ? 8 : 16) == 0 && row_stride % 4 == 0 && g.offset % 4 == 0;
    if (form == SEG_ROW_NORM && base && g.head_dim % 4 == 0 && (!g.weight || reinterpret_cast<uintptr_t>(g.weight) % 16 == 0)) vec |= 1u << i;
    if (form == SEG_PAIRS && base && g.rot_offset % 4 == 0 && g.head_dim % 4 == 0 && g.rot_dims % 8 == 0) vec |= 1u << i;
  }
  max_half = (max_half + 3) / 4 * 4;
  const size_t lds = (static_cast<size_t>(NW) * 2 * max_dim + 2 * max_half) * sizeof(float);
  if (lds > 60 * 1024) return fail(GBXM_ERR_UNSUPPORTED, "rotate_norm_heads: heads of %d channels", max_dim);
  if (T_ == 0) return GBXM_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  GBXM_DISPATCH(act, (rotate_norm_kernel<T><<<dim3(T_, n_segs), NT, lds, s>>>(static_cast<T*>(rows), row_stride, positions, pos_stride, sg, eps, max_dim, max_half,
                                                                                  vec)));
  return after_launch("rotate_norm_heads");
}

int gbxm_slot_append(const void* k, int64_t k_stride, int32_t k_width, const void* v, int64_t v_stride, int32_t v_width, void* kcache, void* vcache,
                     const int32_t* seq, const int32_t* tok, int64_t T_, int32_t keep, int32_t ring, int32_t act, void* stream) {
  if (!act_ok(act) || !k || !kcache || !seq || !tok || k_width <= 0 || k_stride < k_width || keep < 0 || ring < 1 || T_ < 0 ||
      (v && (!vcache || v_width <= 0 || v_stride < v_width)))
    return fail(GBXM_ERR_INVALID, "slot_append: bad argument");
  if (T_ == 0) return GBXM_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const gbxm_slot_rows rows{k, k_stride, k_width, v, v_stride, v_width, kcache, vcache};
  GBXM_DISPATCH(act, (slot_append_kernel<T><<<dim3(T_), NT, 0, s>>>(slot_rows<T>(rows, seq, tok, keep, ring))));
  return after_launch("slot_append");
}

int gbxm_sink_attention_tiled(int32_t dk, int32_t dv, int32_t act, int32_t decode_only) {
  return act == GBXM_BF16 && sink_tiles_shape(dk, dv);          // (steps of single rows: the grouped form of the same products)
}

static int sink_attention(const gbxm_sink_attn_args* a, const gbxm_slot_rows*& rows, void* stream) {
  if (!a || !a->q || !a->k_new || !a->v_new || !a->seq || !a->tok || !a->out) return fail(GBXM_ERR_INVALID, "sink_attention: null argument");
  if (!act_ok(a->act)) return fail(GBXM_ERR_INVALID, "sink_attention: dtype");
  if (a->H <= 0 || a->G <= 0 || a->H % a->G || a->dk <= 0 || a->dv <= 0 || a->keep < 0 || a->ring < 1 || a->T < 0 || a->B < 0 ||
      (a->kcache && !a->vcache))
    return fail(GBXM_ERR_INVALID, "sink_attention: bad geometry");
  if (a->window > 0 && a->ring < a->window) return fail(GBXM_ERR_INVALID, "sink_attention: a ring shorter than the window");
  if (a->chunk > 0 && (a->window > 0 || (a->kcache && a->ring < a->chunk)))
    return fail(GBXM_ERR_INVALID, "sink_attention: chunks exclude a window and need a ring of a chunk's length");
  if (a->chunk < 0 || (a->out_row > 0 && a->out_row < static_cast<int64_t>(a->H) * a->dv)) return fail(GBXM_ERR_INVALID, "sink_attention: chunk or output stride");
  if (a->T == 0) return GBXM_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (!a->decode_only && a->act == GBXM_BF16 && a->tiles && a->n_tiles > 0) {
    const int rc = launch_sink_tiles(*a, s);
    if (rc != GBXM_ERR_UNSUPPORTED) return rc;
  }
  if (a->decode_only && a->act == GBXM_BF16 && a->H <= 65535) {
    const int rc = launch_sink_group(*a, rows, s);
    if (rc != GBXM_ERR_UNSUPPORTED) return rc;
  }
  SinkGeo g{a->H, a->G, a->dk, a->dv, a->window, a->keep, a->ring, a->chunk, a->gate_channels, a->scale, a->head_scale,
            a->out_row > 0 ? a->out_row : static_cast<int64_t>(a->H) * a->dv, a->q_row, a->q_head, a->k_row, a->k_head, a->v_row, a->v_head,
            a->kc_slot, a->kc_row, a->kc_head, a->vc_slot, a->vc_row, a->vc_head, a->gate_row};
  const int R = a->H / a->G;
  if (a->dv > NCH_MAX * DCH) return fail(GBXM_ERR_UNSUPPORTED, "sink_attention: value size %d beyond the row kernel (%d)", a->dv, NCH_MAX * DCH);
  auto lds_of = [&](int rc_) {
    return static_cast<size_t>(2 * KT) * sizeof(void*) + static_cast<size_t>(rc_) * (a->dk + KT + 3 + NW * a->dv) * sizeof(float);
  };
  int rc = R < RC ? R : RC;
  while (rc > 1 && lds_of(rc) > 60 * 1024) --rc;
  if (lds_of(rc) > 60 * 1024) return fail(GBXM_ERR_UNSUPPORTED, "sink_attention: head sizes dk=%d dv=%d are beyond the row kernel", a->dk, a->dv);
  const int chunks = (R + rc - 1) / rc;
  if (a->T > 0x7fffffffLL || a->G * chunks > 65535 || a->H > 65535) return fail(GBXM_ERR_UNSUPPORTED, "sink_attention: grid");
  return a->act == GBXM_BF16 ? launch_rows<bf16_t, true>(*a, g, rc, chunks, lds_of(rc), rows, s) : launch_rows<float, false>(*a, g, rc, chunks, lds_of(rc), rows, s);
}

int gbxm_sink_attention(const gbxm_sink_attn_args* a, void* stream) {
  const gbxm_slot_rows* none = nullptr;
  return sink_attention(a, none, stream);
}

int gbxm_sink_attention_append(const gbxm_sink_attn_args* a, const gbxm_slot_rows* rows, void* stream) {
  if (!a || !rows || !rows->k || !rows->kcache || rows->k_width <= 0 || rows->k_stride < rows->k_width ||
      (rows->v && (!rows->vcache || rows->v_width <= 0 || rows->v_stride < rows->v_width)))
    return fail(GBXM_ERR_INVALID, "sink_attention_append: bad argument");
  const bool apart = a->H >= 65535;                             // (a grid has one place more)
  const gbxm_slot_rows* left = apart ? nullptr : rows;
  const int rc = sink_attention(a, left, stream);
  if (rc != GBXM_OK || !(left || apart)) return rc;
  return gbxm_slot_append(rows->k, rows->k_stride, rows->k_width, rows->v, rows->v_stride, rows->v_width, rows->kcache, rows->vcache, a->seq, a->tok, a->T, a->keep,
                          a->ring, a->act, stream);
}

}  // extern "C"
