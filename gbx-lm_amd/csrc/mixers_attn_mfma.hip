// Matrix-core kernel of gated sliding-window attention for bf16 prompt portions (mechanism: mixers_attn.hip).
//
// One workgroup = one tile of up to 128 query rows of one (sequence, head), a wave owns 32 of them; one group of four waves, or two that take every
// other key tile.  Key / value tiles of 64 (large heads and short sequences: 32) positions go global -> registers -> LDS once per group, in two buffers:
// one barrier a tile, two tiles ahead (ring rows for positions before the step, projection rows inside it; rows past the tile's last query are
// zero-filled so that a zero gate never meets a stale NaN).  Both products are computed swapped so that a lane owns ONE query and the gate arithmetic
// is lane-local:
//   S^T[key, q] = mfma(K rows, Q rows)      lane (q = lane % 32) holds 16 keys of the tile, the other 16 are in lane ^ 32
//   O^T[d, q]  += mfma(V^T rows, G^T)       the gate operand of k-step t is the lane's own g[8t .. 8t+7]; V^T comes out of LDS by
//                                            transposed reads in the same key order
// No softmax: gates of different keys are independent, O^T just accumulates -- no running maximum, no rescale, no final division.
// The fp32 part per score (four transcendentals, see `keep_exponent`) costs more than the products: the kernel is bound by vector
// instructions, and by the tiles that start last -- late tiles of all heads come first.  Gates are rounded to bf16 for the value product.
// Measured: see `launch`.
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
template <int DK, int DV, int GROUPS_, int KT_, int BUFS_> struct WindowShape {
  static constexpr int GROUPS = GROUPS_, KT = KT_, BUFS = BUFS_;   // KT: keys per tile; two buffers: a tile is read while the next is written
  static constexpr int KROW = DK * 2 + 16;                  // +16 B: conflict-free 16-byte fragment reads
  static constexpr int VROW = DV * 2 + 64;                  // pitch = 16 dwords mod 64: the 4 rows of a transposed block land on disjoint banks
  static constexpr int BUF = KT * (KROW + VROW);            // a key and value tile; two of them: one is read while the other is written
  static constexpr int RING = 512, WRAP = 32;               // exponents by distance, and the first of them again behind the last
  static constexpr int BYTES = BUFS * BUF + (RING + WRAP) * 4;   // of a group
  static constexpr int JOIN = GROUPS > 1 ? 4 * (DV / 32) * 16 * 64 * 4 : 0;
  static constexpr int LDS = GROUPS * BYTES > JOIN ? GROUPS * BYTES : JOIN;
  static constexpr int WAVES = BUFS == 1 ? (DK + DV <= 128 ? 4 : DK + DV <= 256 ? 3 : 2) : DK + DV <= 320 ? 2 : 1;      // per SIMD; one buffer (short sequences) lives on many waves
  static constexpr int SLOTS = BUFS == 1 ? 0 : DK <= 192 ? DK / 16 : 8;   // fragments read ahead: a key block's, as far as registers go
};

template <int DK, int DV, int GROUPS, int KT, int BUFS>
__global__ __launch_bounds__((256 * GROUPS), (WindowShape<DK, DV, GROUPS, KT, BUFS>::WAVES)) void window_tile_kernel(const TileArgs a) {
  typedef WindowShape<DK, DV, GROUPS, KT, BUFS> Shape;
  typedef RowPieces<DK, KT> KP;
  typedef RowPieces<DV, KT> VP;
  constexpr int KROW = Shape::KROW, VROW = Shape::VROW, STEP = GROUPS * KT, RING = Shape::RING, WRAP = Shape::WRAP;
  constexpr int KS = DK / 16, DT = DV / 32;
  extern __shared__ __attribute__((aligned(16))) unsigned char all_lds[];
  const int group = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8), tid = threadIdx.x & 255, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned char* kl = all_lds + group * Shape::BYTES;
  unsigned char* vl = kl + KT * KROW;
  float* dist_tab = reinterpret_cast<float*>(kl + BUFS * Shape::BUF);

  const int r = lane & 31, hb = lane >> 5;
  const int tile = (gridDim.x - 1 - blockIdx.x) / a.H;      // (of all heads) late tiles, which see the most keys, start first
  const int b = a.tiles[2 * tile], tq = a.tiles[2 * tile + 1];
  // the query heads of a key / value head stand G apart: where G goes with the eight XCDs they share one's cache
  const int place = blockIdx.x % a.H, kvh = place % a.G, head = kvh * (a.H / a.G) + place / a.G;
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
  // of a tile and those that the next one brings in span 127 + KT + STEP distances, the ring holds 512; its first entries stand again behind its
  // last, so that a lane reads its 28 neighbouring distances from one address); distances outside the window stand there as infinity, which
  // makes the gate zero without a test per score.
  constexpr float LOG2E = 1.4426950408889634f;
  const float dm = a.dmul[head], dr = a.drate[head], cap = fmaxf(a.softcap, 0.f);      // (zero or below: no cap)
  const float zc = -LOG2E * (a.gbias[head] + cap), z2 = 2.f * LOG2E * cap, xs = cap > 0.f ? a.scale * 2.f * LOG2E / cap : -LOG2E * a.scale;
  auto keep_exponent = [&](int d) {
    const float z = d >= 0 && d < W ? fmaf(dm, __log2f(1.f + dr * static_cast<float>(d)), zc) : INFINITY;
    const int at = d & (RING - 1);
    dist_tab[at] = z;
    if (at < WRAP) dist_tab[RING + at] = z;
  };
  const unsigned char* vbase = vl + (4 * hb + ((lane >> 2) & 3)) * VROW + (16 * ((lane >> 4) & 1) + 4 * (lane & 3)) * 2;
  const unsigned char* kbase = kl + r * KROW + hb * 16;

  const bf16_t *kc = a.kc + static_cast<int64_t>(slot) * W * nkv_k + kvh * DK, *vc = a.vc + static_cast<int64_t>(slot) * W * nkv_v + kvh * DV;
  const bf16_t *kn = a.qkv + a.nq + kvh * DK, *vn = a.qkv + a.nq + a.nk + kvh * DV;
  auto src = [&](const bf16_t* ring, int row_elems, const bf16_t* fresh, int j) -> const bf16_t* {
    return j < pos0 ? ring + static_cast<int64_t>(j % W) * row_elems : fresh + (row0 + (j - pos0)) * a.stride;
  };

  u32x4 kr[KP::N], vr[VP::N];
  const bool near = a.stride < (1 << 22) && nkv_k < (1 << 22) && nkv_v < (1 << 22);      // 32 bits of byte offset reach across a tile's rows
  // rows of a whole tile that follow each other in one buffer come by buffer loads from a scalar place (mixers_sink_mfma.hip); tiles that the last
  // query, the ring's seam or the step's first row cuts find every row by itself, rows past the last query are zeros
  auto fetch = [&](int jt) {
    const bool old = jt < pos0;
    bool whole = BUFS == 2 && near && jt + KT - 1 <= jlast && (!old || jt + KT <= pos0);
    int at = row0 + (jt - pos0);
    if (whole && old) {
      at = jt % W;
      whole = at + KT <= W;
    }
    if (whole) {
      const int ks = (old ? nkv_k : static_cast<int>(a.stride)) * 2, vs = (old ? nkv_v : static_cast<int>(a.stride)) * 2;
      const bf16_t* kp = (old ? kc : kn) + static_cast<int64_t>(at) * (ks / 2);
      const bf16_t* vp = (old ? vc : vn) + static_cast<int64_t>(at) * (vs / 2);
      const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(kp), 0, (KT - 1) * ks + DK * 2, 0x00020000);
      const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(vp), 0, (KT - 1) * vs + DV * 2, 0x00020000);
#pragma unroll
      for (int i = 0; i < KP::N; ++i)
        kr[i] = __builtin_amdgcn_raw_buffer_load_b128(krs, KP::used(tid, i) ? KP::row(tid, i) * ks + KP::piece(tid, i) * 16 : 0x7ffffff0, 0, 0);
#pragma unroll
      for (int i = 0; i < VP::N; ++i)
        vr[i] = __builtin_amdgcn_raw_buffer_load_b128(vrs, VP::used(tid, i) ? VP::row(tid, i) * vs + VP::piece(tid, i) * 16 : 0x7ffffff0, 0, 0);
      return;
    }
#pragma unroll
    for (int i = 0; i < KP::N; ++i) {
      const int j = jt + KP::row(tid, i);
      kr[i] = u32x4{0, 0, 0, 0};
      if (KP::used(tid, i) && j <= jlast) kr[i] = *reinterpret_cast<const u32x4*>(src(kc, nkv_k, kn, j) + KP::piece(tid, i) * 8);
    }
#pragma unroll
    for (int i = 0; i < VP::N; ++i) {
      const int j = jt + VP::row(tid, i);
      vr[i] = u32x4{0, 0, 0, 0};
      if (VP::used(tid, i) && j <= jlast) vr[i] = *reinterpret_cast<const u32x4*>(src(vc, nkv_v, vn, j) + VP::piece(tid, i) * 8);
    }
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int i = 0; i < KP::N; ++i)
      if (KP::used(tid, i)) *reinterpret_cast<u32x4*>(kl + buf * Shape::BUF + KP::row(tid, i) * KROW + KP::piece(tid, i) * 16) = kr[i];
#pragma unroll
    for (int i = 0; i < VP::N; ++i)
      if (VP::used(tid, i)) *reinterpret_cast<u32x4*>(vl + buf * Shape::BUF + VP::row(tid, i) * VROW + VP::piece(tid, i) * 16) = vr[i];
  };
  // Two buffers, one barrier a tile: behind it tile t and its distances are in LDS and tile t + 1 in registers; that one is parked in the other
  // buffer, whose readers have all passed the barrier, with the distances it brings in, and tile t + 2 is asked for.  One buffer: tile t + 1 is
  // asked for while tile t is read.
  const int j1 = jfirst + group * KT, tiles = (jlast - jfirst + STEP) / STEP;      // (every group runs as many rounds: the barriers are common)
  if (j1 <= jlast) fetch(j1);
  if constexpr (BUFS == 2) {
    if (j1 <= jlast) stage(0);
    if (j1 + STEP <= jlast) fetch(j1 + STEP);
  }
  if (tid < 127 + KT) keep_exponent(pos0 + tq - j1 + 127 - tid);       // distances of the tile's queries from the group's first keys
  for (int round = 0; round < tiles; ++round) {
    const int jt = j1 + round * STEP;
    __syncthreads();
    if constexpr (BUFS == 1) {
      if (jt <= jlast) stage(0);
      __syncthreads();
    } else if (jt + STEP <= jlast) {
      stage((round + 1) & 1);
    }
    if (tid < STEP) keep_exponent(pos0 + tq - jt - STEP - KT + 1 + tid);
    if (jt + BUFS * STEP <= jlast) fetch(jt + BUFS * STEP);
    if (!wave_live || jt > wq1 || jt + KT - 1 < wq0 - W + 1) continue;      // wave-uniform: no key of the tile is seen by this wave

    const unsigned char* kb = kbase + (BUFS == 2 ? round & 1 : 0) * Shape::BUF;
    const unsigned char* vb = vbase + (BUFS == 2 ? round & 1 : 0) * Shape::BUF;
    auto kfrag = [&](int h, int ks) { return *reinterpret_cast<const u32x4*>(kb + h * 32 * KROW + ks * 32); };
    auto vfrag = [&](int h, int i) {                            // i: block of 32 channels, half of the 32 keys
      const u32x2 v0 = lds_read_tr(vb + (32 * h + 16 * (i & 1)) * VROW + (i >> 1) * 64);
      const u32x2 v1 = lds_read_tr(vb + (32 * h + 16 * (i & 1) + 8) * VROW + (i >> 1) * 64);
      return u32x4{v0.x, v0.y, v1.x, v1.y};
    };
    auto gates = [&](int h, const f32x16& st, u32x4 (&gf)[2]) {
      const int j0 = jt + 32 * h;
      const float* tp = dist_tab + ((qpos - j0 - 4 * hb - 27) & (RING - 1));        // distances 27 down to 0 of the lane's keys from here
      const bool cut = j0 + 31 > wq0 || wq1 - j0 >= W;          // (wave-uniform) keys outside: zero also where the score is no number
      // scores' chains of transcendentals run side by side, as many as the registers take (the cap is asked for outside: a branch a score would run
      // them one after the other, 132 us instead of 97 for 2 047 + 1 100 + 333 + 1 rows)
      constexpr int C = BUFS == 2 ? 16 : 8;
#pragma unroll
      for (int c = 0; c < 16; c += C) {
        float g[C], t[C];
#pragma unroll
        for (int e = 0; e < C; ++e) t[e] = tp[27 - 8 * ((c + e) >> 2) - (e & 3)];
        if (cap > 0.f) {
#pragma unroll
          for (int e = 0; e < C; ++e) g[e] = fmaf(z2, __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(st[c + e] * xs)), t[e]);
        } else {
#pragma unroll
          for (int e = 0; e < C; ++e) g[e] = fmaf(st[c + e], xs, t[e]);
        }
#pragma unroll
        for (int e = 0; e < C; ++e) g[e] = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(g[e]));
        if (cut) {
#pragma unroll
          for (int e = 0; e < C; ++e) g[e] = t[e] == INFINITY ? 0.f : g[e];
        }
#pragma unroll
        for (int e = 0; e < C; e += 8) gf[(c + e) / 8] = u32x4{pack2(g[e], g[e + 1]), pack2(g[e + 2], g[e + 3]), pack2(g[e + 4], g[e + 5]), pack2(g[e + 6], g[e + 7])};
      }
    };
    auto half = [&](int h) {
      const int j0 = jt + 32 * h;
      if (j0 > wq1 || j0 + 31 < wq0 - W + 1) return;           // (wave-uniform)
      f32x16 st = f32x16{0};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) st = mfma_bf16(kfrag(h, ks), qf[ks], st);
      u32x4 gf[2];
      gates(h, st, gf);
#pragma unroll
      for (int i = 0; i < DT * 2; ++i) o[i >> 1] = mfma_bf16(vfrag(h, i), gf[i & 1], o[i >> 1]);
    };
    constexpr int NH = KT / 32, NK = KS * NH, NV = DT * 2 * NH, SLOTS = Shape::SLOTS, NF = SLOTS < NV ? SLOTS : NV;
    if constexpr (BUFS == 1) {
#pragma unroll
      for (int h = 0; h < NH; ++h) half(h);
      continue;
    }
    if (NH == 2 && !(jt + 32 <= wq1 && jt + 31 >= wq0 - W + 1)) {
      half(0);
      half(NH - 1);
      continue;
    }
    // all of the tile is seen: fragments are read in bulk ahead of the products that take them, a slot is filled again as its product leaves, and
    // one half's products run under the other's gates
    u32x4 fr[SLOTS ? SLOTS : 1], gf[NH][2];
    f32x16 st[NH];
#pragma unroll
    for (int h = 0; h < NH; ++h) st[h] = f32x16{0};
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) fr[i] = kfrag(i / KS, i % KS);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      st[i / KS] = mfma_bf16(fr[i % (SLOTS ? SLOTS : 1)], qf[i % KS], st[i / KS]);
      if (i + SLOTS < NK) fr[i % (SLOTS ? SLOTS : 1)] = kfrag((i + SLOTS) / KS, (i + SLOTS) % KS);
      if (i % KS == KS - 1) __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < NF; ++i) fr[i] = vfrag(i / (DT * 2), i % (DT * 2));
#pragma unroll
    for (int h = 0; h < NH; ++h) {
      gates(h, st[h], gf[h]);
#pragma unroll
      for (int i = h * DT * 2; i < (h + 1) * DT * 2; ++i) {
        o[i % (DT * 2) >> 1] = mfma_bf16(fr[i % (NF ? NF : 1)], gf[h][i & 1], o[i % (DT * 2) >> 1]);
        if (i + NF < NV) fr[i % (NF ? NF : 1)] = vfrag((i + NF) / (DT * 2), (i + NF) % (DT * 2));
      }
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

template <int DK, int DV, int GROUPS, int KT, int BUFS>
int launch_shape(const TileArgs& t, int n_tiles, hipStream_t s) {
  constexpr int bytes = WindowShape<DK, DV, GROUPS, KT, BUFS>::LDS;
  static OncePerDevice once;
  if (once.pending()) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(window_tile_kernel<DK, DV, GROUPS, KT, BUFS>), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return hip_fail(e, "window_attention (tiles)");
    once.done();
  }
  window_tile_kernel<DK, DV, GROUPS, KT, BUFS><<<static_cast<unsigned>(t.H) * n_tiles, 256 * GROUPS, bytes, s>>>(t);
  return after_launch("window_attention (tiles)");
}

// Two groups of waves a tile shorten the chain of a long tile; one leaves a CU room for two tiles.  Either form takes as long as its longest tile or
// as all of them on the tiles that fit at a time (256 | 512), in units of a key that one group multiplies, with what a tile costs beside its keys as
// 140 | 350 of them.  Sequences of a tile's keys and less take 32 keys, one buffer and as many waves as fit.  One | two, us (in brackets: one
// buffer, every row found by itself and a branch a score, the better of its forms):
//   32 heads of 128: 1 000 rows 36.5 | 31.4 (41), 1 300 47.9 | 38.2 (52), 2 200 85 | 85 (114), 4 000 216 | 223 (245), with a window of 64 32 | 47 (39);
//   2 047 + 1 100 + 333 + 1 rows 96 | 105 (134); 64 rows x 32 15.5 | 27.8 (18.7); 20 rows x 30 beside 2 000 82 | 87 (107);
//   16 heads of 64: 4 000 rows 108 | 91 (122), with a window of 1 024 47 | 52 (67); 500 rows x 8 23.8 | 28.0 (32).
// One buffer of 32 keys against two of 64: 20 rows x 64 12.5 | 17.3 (13.2), 64 heads' worth of 20 rows x 30 4.47 | 4.75, 64 rows x 32 16.1 | 15.5.
template <int DK, int DV>
int launch(const TileArgs& t, int n_tiles, int64_t most, int64_t sum, hipStream_t s) {
  if (most <= 0 || sum <= 0) { most = t.window; sum = n_tiles * most; }
  if (most <= 48) return launch_shape<DK, DV, 1, 32, 1>(t, n_tiles, s);
  if constexpr (DK + DV <= 256) {                            // (larger heads: 64 keys or a second group would cost the second wave per SIMD)
    constexpr int64_t ONE = 140, TWO = 350;
    const int64_t n = static_cast<int64_t>(t.H) * n_tiles, keys = sum * t.H;
    const int64_t one = std::max(most + ONE, (keys + n * ONE) / 512), two = std::max(most / 2 + TWO, (keys / 2 + n * TWO) / 256);
    if (two < one) return launch_shape<DK, DV, 2, 64, 2>(t, n_tiles, s);
    return launch_shape<DK, DV, 1, 64, 2>(t, n_tiles, s);
  } else {
    return launch_shape<DK, DV, 1, 32, 2>(t, n_tiles, s);
  }
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
