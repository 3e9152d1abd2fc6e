// Matrix-core kernel of gated sliding-window attention for bf16 prompt portions (mechanism: mixers_attn.hip).
//
// One workgroup = one tile of up to 128 query rows of one (sequence, head), a wave owns 32 of them; one group of four waves, or two that take every
// other key tile.  Key / value tiles of 32 (two groups: 64) positions go global -> registers (one tile ahead) -> LDS once per group (ring rows for positions before the step, projection rows inside it; rows
// past the tile's last query are zero-filled so that a zero gate never meets a stale NaN).  Both products are computed swapped so
// that a lane owns ONE query and the gate arithmetic is lane-local:
//   S^T[key, q] = mfma(K rows, Q rows)      lane (q = lane % 32) holds 16 keys of the tile, the other 16 are in lane ^ 32
//   O^T[d, q]  += mfma(V^T rows, G^T)       the gate operand of k-step t is the lane's own g[8t .. 8t+7]; V^T comes out of LDS by
//                                            transposed reads in the same key order
// No softmax: gates of different keys are independent, O^T just accumulates -- no running maximum, no rescale, no final division.
// The fp32 part per score (four transcendentals, see `exponent`) costs more than the products: the kernel is bound by vector
// instructions, and by the tiles that start last -- late tiles of all heads come first.  Gates are rounded to bf16 for the value product.
// Measured against five transcendentals a score and one group for all: see `launch`.
#include <algorithm>
#include "mixers_mfma.h"

namespace gbxm {
namespace {

struct TileArgs {
  const bf16_t* qkv;
  const bf16_t* kc;
  const bf16_t* vc;
  const int* seq;
  const int* tiles;
  bf16_t* out;
  const float* dmul;
  const float* drate;
  const float* gbias;
  int64_t stride;
  int q_tile, H, G, window, nq, nk;
  float scale, softcap;
};

// Two groups of four waves take every other key tile of the same queries (their sums meet in LDS at the end): a tile late in a long prompt
// is a chain of key tiles that the rest of the launch would otherwise wait for.  `launch` chooses.
template <int DK, int DV, int GROUPS_, int KT_> struct WindowShape {
  static constexpr int GROUPS = GROUPS_, KT = KT_;          // KT: keys per tile
  static constexpr int KROW = DK * 2 + 16;                  // +16 B: conflict-free 16-byte fragment reads
  static constexpr int VROW = DV * 2 + 64;                  // pitch = 16 dwords mod 64: the 4 rows of a transposed block land on disjoint banks
  static constexpr int BYTES = KT * (KROW + VROW) + 1024;   // one group's key and value tile, and its 256 exponents by distance
  static constexpr int JOIN = GROUPS > 1 ? 4 * (DV / 32) * 16 * 64 * 4 : 0;
  static constexpr int LDS = GROUPS * BYTES > JOIN ? GROUPS * BYTES : JOIN;
  static constexpr int WAVES = DK + DV <= 320 ? 2 : 1;      // per SIMD: left to itself <192, 128> takes the registers of both
};

template <int DK, int DV, int GROUPS, int KT>
__global__ __launch_bounds__((256 * GROUPS), (WindowShape<DK, DV, GROUPS, KT>::WAVES)) void window_tile_kernel(const TileArgs a) {
  typedef WindowShape<DK, DV, GROUPS, KT> Shape;
  constexpr int KROW = Shape::KROW, VROW = Shape::VROW, STEP = GROUPS * KT;
  constexpr int KS = DK / 16, DT = DV / 32;
  extern __shared__ __attribute__((aligned(16))) unsigned char all_lds[];
  const int group = threadIdx.x >> 8, tid = threadIdx.x & 255, lane = tid & 63, wave = tid >> 6;
  unsigned char* lds = all_lds + group * Shape::BYTES;
  unsigned char* kl = lds;
  unsigned char* vl = lds + KT * KROW;
  float* dist_tab = reinterpret_cast<float*>(vl + KT * VROW);      // entry distance & 255

  const int r = lane & 31, hb = lane >> 5;
  const int tile = (gridDim.x - 1 - blockIdx.x) / a.H;      // (of all heads) late tiles, which see the most keys, start first
  const int b = a.tiles[2 * tile], tq = a.tiles[2 * tile + 1];
  const int head = blockIdx.x % a.H, kvh = head / (a.H / a.G);
  const int slot = a.seq[4 * b], pos0 = a.seq[4 * b + 1], n = a.seq[4 * b + 2], row0 = a.seq[4 * b + 3];
  const int W = a.window;
  const int qn = min(a.q_tile, n - tq);                     // queries of this tile
  const int qloc = wave * 32 + r;
  const bool qvalid = qloc < qn;
  const int qpos = pos0 + tq + qloc;
  const int nkv_k = a.G * DK, nkv_v = a.G * DV;

  u32x4 qf[KS];
  {
    const bf16_t* qp = a.qkv + (row0 + tq + min(qloc, qn - 1)) * a.stride + head * DK + hb * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const u32x4*>(qp + ks * 16);
  }
  f32x16 o[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i) o[i] = f32x16{0};

  const int jfirst = max(0, pos0 + tq - W + 1), jlast = pos0 + tq + qn - 1;
  const bool wave_live = wave * 32 < qn;
  const int wq0 = pos0 + tq + wave * 32, wq1 = min(wq0 + 31, jlast);   // positions of this wave's queries
  // gate = 1 / (1 + 2^z),  z = -log2e (s + gb) + dm log2(1 + dr dist),  s = cap tanh(x / cap) = cap - 2 cap / (1 + 2^(x 2 log2e / cap)): four
  // transcendentals a score.  What of z depends on the distance alone comes from a table that moves on with the key tile (the queries and keys
  // of a tile span 127 + KT distances, the ring holds 256); distances outside the window stand there as infinity, which
  // makes the gate zero without a test per score.
  constexpr float LOG2E = 1.4426950408889634f;
  const float dm = a.dmul[head], dr = a.drate[head], cap = fmaxf(a.softcap, 0.f);      // (zero or below: no cap)
  const float zc = -LOG2E * (a.gbias[head] + cap), z2 = 2.f * LOG2E * cap, xs = cap > 0.f ? a.scale * 2.f * LOG2E / cap : -LOG2E * a.scale;
  auto exponent = [&](int d) { return d >= 0 && d < W ? fmaf(dm, __log2f(1.f + dr * static_cast<float>(d)), zc) : INFINITY; };
  const unsigned char* vbase = vl + (4 * hb + ((lane >> 2) & 3)) * VROW + (16 * ((lane >> 4) & 1) + 4 * (lane & 3)) * 2;
  const unsigned char* kbase = kl + r * KROW + hb * 16;

  auto src = [&](const bf16_t* ring, int row_elems, int seg_off, int j) -> const bf16_t* {
    return j < pos0 ? ring + (static_cast<int64_t>(slot) * W + j % W) * row_elems : a.qkv + (row0 + (j - pos0)) * a.stride + seg_off;
  };

  // key / value tile: global -> registers one tile ahead, registers -> LDS at the top of its iteration
  constexpr int KP = (KT * (DK / 8) + 255) / 256, VP = (KT * (DV / 8) + 255) / 256;
  u32x4 kr[KP], vr[VP];
  auto fetch = [&](int jt) {
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      const int p = tid + 256 * i, row = p / (DK / 8), c = p % (DK / 8), j = jt + row;
      kr[i] = u32x4{0, 0, 0, 0};
      if (p < KT * (DK / 8) && j <= jlast) kr[i] = *reinterpret_cast<const u32x4*>(src(a.kc, nkv_k, a.nq, j) + kvh * DK + c * 8);
    }
#pragma unroll
    for (int i = 0; i < VP; ++i) {
      const int p = tid + 256 * i, row = p / (DV / 8), c = p % (DV / 8), j = jt + row;
      vr[i] = u32x4{0, 0, 0, 0};
      if (p < KT * (DV / 8) && j <= jlast) vr[i] = *reinterpret_cast<const u32x4*>(src(a.vc, nkv_v, a.nq + a.nk, j) + kvh * DV + c * 8);
    }
  };
  const int j1 = jfirst + group * KT, tiles = (jlast - jfirst + STEP) / STEP;      // (every group runs as many rounds: the barriers are common)
  if (j1 <= jlast) fetch(j1);
  const int d1 = pos0 + tq - j1;                              // distance of the tile's first query from the group's first key
  if (tid < 127 + KT) dist_tab[(d1 + 127 - tid) & 255] = exponent(d1 + 127 - tid);
  for (int round = 0; round < tiles; ++round) {
    const int jt = j1 + round * STEP;
    __syncthreads();                                          // the previous tile has been consumed
    if (tid < STEP) {                                         // the distances that the tile brings in
      const int d = pos0 + tq - jt - KT + 1 + tid;
      dist_tab[d & 255] = exponent(d);
    }
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      const int p = tid + 256 * i;
      if (p < KT * (DK / 8)) *reinterpret_cast<u32x4*>(kl + (p / (DK / 8)) * KROW + (p % (DK / 8)) * 16) = kr[i];
    }
#pragma unroll
    for (int i = 0; i < VP; ++i) {
      const int p = tid + 256 * i;
      if (p < KT * (DV / 8)) *reinterpret_cast<u32x4*>(vl + (p / (DV / 8)) * VROW + (p % (DV / 8)) * 16) = vr[i];
    }
    __syncthreads();
    if (jt + STEP <= jlast) fetch(jt + STEP);                 // the next tile travels while this one is computed
    if (!wave_live || jt > wq1 || jt + KT - 1 < wq0 - W + 1) continue;      // wave-uniform: no key of the tile is seen by this wave

    auto scores = [&](int h) {
      f32x16 st = f32x16{0};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) st = mfma_bf16(*reinterpret_cast<const u32x4*>(kbase + h * 32 * KROW + ks * 32), qf[ks], st);
      return st;
    };
    auto gates = [&](int h, const f32x16& st, u32x4 (&gf)[2]) {
      const int j0 = jt + 32 * h, dq = qpos - j0 - 4 * hb;
      float g[16], t[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        t[e] = dist_tab[(dq - 8 * (e >> 2) - (e & 3)) & 255];
        const float z = cap > 0.f ? fmaf(z2, __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(st[e] * xs)), t[e]) : fmaf(st[e], xs, t[e]);
        g[e] = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(z));
      }
      if (j0 + 31 > wq0 || wq1 - j0 >= W) {                     // (wave-uniform) keys outside: zero also where the score is no number
#pragma unroll
        for (int e = 0; e < 16; ++e) g[e] = t[e] == INFINITY ? 0.f : g[e];
      }
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
        gf[tt] = u32x4{pack2(g[8 * tt], g[8 * tt + 1]), pack2(g[8 * tt + 2], g[8 * tt + 3]), pack2(g[8 * tt + 4], g[8 * tt + 5]),
                       pack2(g[8 * tt + 6], g[8 * tt + 7])};
    };
    auto values = [&](int h, const u32x4 (&gf)[2]) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
          const u32x2 v0 = lds_read_tr(vbase + (32 * h + 16 * tt) * VROW + dt * 64);
          const u32x2 v1 = lds_read_tr(vbase + (32 * h + 16 * tt + 8) * VROW + dt * 64);
          o[dt] = mfma_bf16(u32x4{v0.x, v0.y, v1.x, v1.y}, gf[tt], o[dt]);
        }
    };
    auto half = [&](int h) {
      const int j0 = jt + 32 * h;
      if (j0 > wq1 || j0 + 31 < wq0 - W + 1) return;           // (wave-uniform)
      u32x4 gf[2];
      gates(h, scores(h), gf);
      values(h, gf);
    };
    if constexpr (KT == 64) {
      if (jt + 32 <= wq1 && jt + 31 >= wq0 - W + 1) {           // both halves are seen: one half's matrix products under the other's gates
        const f32x16 s0 = scores(0), s1 = scores(1);
        u32x4 g0[2], g1[2];
        gates(0, s0, g0);
        values(0, g0);
        gates(1, s1, g1);
        values(1, g1);
        continue;
      }
      half(0);
      half(1);
    } else {
      half(0);
    }
  }

  if constexpr (GROUPS > 1) {
    float* join = reinterpret_cast<float*>(all_lds) + wave * (DT * 16 * 64) + lane;
    __syncthreads();
    if (group == 1) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int e = 0; e < 16; ++e) join[(dt * 16 + e) * 64] = o[dt][e];
    }
    __syncthreads();
    if (group == 1) return;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[dt][e] += join[(dt * 16 + e) * 64];
  }
  if (qvalid) {
    bf16_t* op = a.out + (row0 + tq + qloc) * (static_cast<int64_t>(a.H) * DV) + head * DV;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const int d = dt * 32 + 8 * q4 + 4 * hb;
        *reinterpret_cast<u32x2*>(op + d) = u32x2{pack2(o[dt][4 * q4], o[dt][4 * q4 + 1]), pack2(o[dt][4 * q4 + 2], o[dt][4 * q4 + 3])};
      }
  }
}

template <int DK, int DV, int GROUPS, int KT>
int launch_shape(const TileArgs& t, int n_tiles, hipStream_t s) {
  constexpr int bytes = WindowShape<DK, DV, GROUPS, KT>::LDS;
  static OncePerDevice once;
  if (once.pending()) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(window_tile_kernel<DK, DV, GROUPS, KT>), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return hip_fail(e, "window_attention (tiles)");
    once.done();
  }
  window_tile_kernel<DK, DV, GROUPS, KT><<<static_cast<unsigned>(t.H) * n_tiles, 256 * GROUPS, bytes, s>>>(t);
  return after_launch("window_attention (tiles)");
}

// Two groups of waves a tile, 64 keys each, shorten the chain of a long tile; one group and 32 keys leave a CU room for two tiles.  Either form takes as
// long as its longest tile or as all of them on the tiles that fit at a time (256 | 512), in units of a key that one group multiplies, with what a tile
// costs beside its keys as 140 | 175 of them.  One | two, us (in brackets: one group, five transcendentals a score, before both):
//   32 heads of 128: 1 000 rows 65 | 40 (86), 1 300 82 | 49 (129), 2 200 137 | 109 (248), 4 000 256 | 295 (783), with a window of 64 41 | 59 (51); 2 047 + 1 100 + 333 +
//   1 rows 145 | 138 (339); 64 rows x 32 18 | 32 (21); 20 rows x 64 13 | 40 (19); 20 rows x 30 beside 2 000 126 | 101;
//   16 heads of 64: 4 000 rows 193 | 122 (351), with a window of 1 024 71 | 71 (112); 2 000 rows x 2 109 | 68 (182); 500 rows x 8 33 | 35 (53); 33 rows 5.7 | 6.1 (6.4).
template <int DK, int DV>
int launch(const TileArgs& t, int n_tiles, int64_t most, int64_t sum, hipStream_t s) {
  if constexpr (DK + DV <= 256) {                            // (larger heads: 64 keys or a second group would cost the second wave per SIMD)
    constexpr int64_t ONE = 140, TWO = 175;
    if (most <= 0 || sum <= 0) { most = t.window; sum = n_tiles * most; }
    const int64_t n = static_cast<int64_t>(t.H) * n_tiles, keys = sum * t.H;
    const int64_t one = std::max(most + ONE, (keys + n * ONE) / 512), two = std::max(most / 2 + TWO, (keys / 2 + n * TWO) / 256);
    if (two < one) return launch_shape<DK, DV, 2, 64>(t, n_tiles, s);
  }
  return launch_shape<DK, DV, 1, 32>(t, n_tiles, s);
}

}  // namespace

bool window_tiles_shape(int dk, int dv) {
  const int ok[][2] = {{64, 64}, {96, 64}, {128, 64}, {64, 128}, {128, 128}, {192, 128}, {256, 256}, {96, 96}, {64, 32}, {32, 32}, {32, 64}};
  for (const auto& p : ok)
    if (p[0] == dk && p[1] == dv) return true;
  return false;
}

int launch_window_tiles(const gbxm_window_attn_args& a, hipStream_t s) {
  if (!window_tiles_shape(a.dk, a.dv)) return GBXM_ERR_UNSUPPORTED;
  if (a.q_tile != 128 || static_cast<int64_t>(a.H) * a.n_tiles > 0x7fffffff || a.row_stride % 8 || (reinterpret_cast<uintptr_t>(a.qkv) | reinterpret_cast<uintptr_t>(a.kcache) |
                                                             reinterpret_cast<uintptr_t>(a.vcache) | reinterpret_cast<uintptr_t>(a.out)) % 16)
    return GBXM_ERR_UNSUPPORTED;
  TileArgs t{static_cast<const bf16_t*>(a.qkv), static_cast<const bf16_t*>(a.kcache), static_cast<const bf16_t*>(a.vcache), a.seq, a.tiles,
             static_cast<bf16_t*>(a.out), a.dist_mul, a.dist_rate, a.gate_bias, a.row_stride, a.q_tile, a.H, a.G, a.window, a.H * a.dk,
             a.G * a.dk, a.scale, a.softcap};
#define GBXM_TILE(DK_, DV_) if (a.dk == DK_ && a.dv == DV_) return launch<DK_, DV_>(t, a.n_tiles, a.most_keys, a.tile_keys, s)
  GBXM_TILE(64, 64); GBXM_TILE(96, 64); GBXM_TILE(128, 64); GBXM_TILE(64, 128); GBXM_TILE(128, 128); GBXM_TILE(192, 128); GBXM_TILE(256, 256);
  GBXM_TILE(96, 96); GBXM_TILE(64, 32); GBXM_TILE(32, 32); GBXM_TILE(32, 64);
#undef GBXM_TILE
  return GBXM_ERR_UNSUPPORTED;
}

}  // namespace gbxm
