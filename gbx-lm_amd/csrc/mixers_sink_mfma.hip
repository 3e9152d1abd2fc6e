// Matrix-core kernel of softmax attention with a sink for bf16 prompt portions (mechanism and key order: mixers_sink.hip).
//
// One workgroup = a tile of up to 128 query rows of one (sequence, head); a wave owns 32 queries, and one or two groups of four waves share the
// tile's keys (SinkShape).  Key / value tiles of 64 (large heads and short sequences: 32) visible positions go global -> registers -> LDS once per
// group, in two buffers: one barrier a tile, two tiles ahead.
// Both products are computed swapped,
//   S^T[key, q] = mfma(K rows, Q rows),    O^T[d, q] += mfma(V^T rows, P^T),
// so that a lane owns ONE query: lane (q = lane % 32, half = lane / 32) holds 16 of the tile's 32 scores of its query, the other 16
// are in lane ^ 32 (and as many of each further 32 keys).  The running maximum is shared by the two lanes of a query (one cross-lane exchange per tile), each keeps its
// own part of the denominator (joined once at the end), and both rescale their accumulators (different channels of the same
// query) by the same factor.  The sink starts the running maximum and counts once in the denominator.  Weights, at most 1, are rounded to bf16
// for the value product; the denominator sums them in fp32.
//
// Bound by what a wave's own chain leaves idle (of a tile's time the matrix cores work a third, vector instructions a third: one exponential and
// four others a score) and, in short prompts, by how few tiles there are.  Before (one buffer, every row found by itself, tiles from both ends of
// a prompt in one workgroup) | now, us: 16 heads of <192, 128>, 8 192 rows 542 | 389, 2 000 + 777 rows 73 | 59, 7 500 rows 483 | 335; <128, 128>,
// 8 192 rows 404 | 301, 4 000 rows 116 | 91, 1 501 + 700 + 65 rows 43 | 33; <64, 64>, 2 000 + 777 rows 37 | 30; 8 heads of <256, 256>, 4 000 rows 425 | 248.
//
// Head sizes are run-time numbers (multiples of 8) inside a compiled capacity <DK, DV>: channels beyond them are staged as zeros.
#include <algorithm>
#include <utility>
#include "mixers_mfma.h"

namespace gbxm {

int launch_sink_reduce(const gbxm_sink_attn_args& a, int splits, const gbxm_slot_rows* rows, hipStream_t s);      // mixers_sink.hip

namespace {

struct SinkTileArgs {
  const bf16_t* q;
  const bf16_t* kn;
  const bf16_t* vn;
  const bf16_t* kc;
  const bf16_t* vc;
  const int* seq;
  const int* tiles;
  bf16_t* out;
  const float* sink;
  const bf16_t* gate;
  int64_t q_row, q_head, k_row, k_head, v_row, v_head, kc_slot, kc_row, kc_head, vc_slot, vc_row, vc_head, gate_row;
  int q_tile, H, G, dk, dv, window, keep, ring, chunk;
  float scale;
  const float* head_scale;
  int64_t out_row;
  int gate_channels;
};

// four neighbouring channels of a head's output, times f and (a gate per channel) their gates' sigmoids
__device__ __forceinline__ u32x2 out4(const SinkTileArgs& a, int64_t row, int head, int d, const f32x16& o, int q4, float f) {
  float v[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = o[4 * q4 + i] * f;
  if (a.gate_channels) {
    float g[4];
    Lanes<bf16_t, 4>::load(a.gate + row * a.gate_row + head * a.dv + d, g);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] *= sigmoid_<true>(g[i]);
  }
  return u32x2{pack2(v[0], v[1]), pack2(v[2], v[3])};
}

// With two GROUPS of four waves each takes every other key tile of the same queries, with a maximum and denominator of its own; the halves
// meet in LDS at the end.
template <int DK, int DV, int GROUPS_, int KT_, int BUFS_> struct SinkShape {
  static constexpr int GROUPS = GROUPS_, KT = KT_, BUFS = BUFS_;   // KT: keys per tile; two buffers: a tile is read while the next is written
  static constexpr int KROW = DK * 2 + 16;                   // +16 B: conflict-free 16-byte fragment reads
  static constexpr int VROW = DV * 2 + 64;                   // pitch = 16 dwords mod 64: the 4 rows of a transposed block land on disjoint banks
  static constexpr int BUF = KT * (KROW + VROW);             // one tile
  static constexpr int BYTES = BUFS * BUF;                   // of a group
  static constexpr int JOIN = GROUPS > 1 ? 4 * (DV / 32 * 16 + 2) * 64 * 4 : 0;
  static constexpr int LDS = GROUPS * BYTES > JOIN ? GROUPS * BYTES : JOIN;
  static constexpr bool MANY = GROUPS == 1 && BUFS == 1;     // short sequences live on many waves
  static constexpr int WAVES = DK + DV <= (MANY ? 128 : 64) ? 4 : DK + DV <= 256 && MANY ? 3 : DK + DV <= 320 ? 2 : 1;   // per SIMD
  // fragments read ahead: a key block's, as far as registers go
  static constexpr int SLOTS = BUFS == 1 ? 0 : DK <= 192 ? DK / 16 : 8;
};

template <int DK, int DV, int GROUPS, int KT, int BUFS>
__device__ __forceinline__ void sink_tile(const SinkTileArgs& a, const int tile, const int head, unsigned char* all_lds) {
  typedef SinkShape<DK, DV, GROUPS, KT, BUFS> Shape;
  typedef RowPieces<DK, KT> KP;
  typedef RowPieces<DV, KT> VP;
  constexpr int KROW = Shape::KROW, VROW = Shape::VROW, STEP = GROUPS * KT, NH = KT / 32;
  constexpr int KS = DK / 16, DT = DV / 32;
  const int group = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8), tid = threadIdx.x & 255, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned char* kl = all_lds + group * Shape::BYTES;
  unsigned char* vl = kl + KT * KROW;

  const int r = lane & 31, hb = lane >> 5;
  const int b = a.tiles[2 * tile], tq = a.tiles[2 * tile + 1];
  const int kvh = head / (a.H / a.G);
  const int slot = a.seq[4 * b], pos0 = a.seq[4 * b + 1], n = a.seq[4 * b + 2], row0 = a.seq[4 * b + 3];
  const int qn = min(a.q_tile, n - tq);                     // queries of this tile
  const int qloc = wave * 32 + r;
  const bool qvalid = qloc < qn;
  const int qpos = pos0 + tq + qloc;

  u32x4 qf[KS];
  {
    const bf16_t* qp = a.q + (row0 + tq + min(qloc, qn - 1)) * a.q_row + head * a.q_head;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int c = ks * 16 + hb * 8;
      qf[ks] = c < a.dk ? *reinterpret_cast<const u32x4*>(qp + c) : u32x4{0, 0, 0, 0};
    }
  }
  f32x16 o[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i) o[i] = f32x16{0};

  // the keys any query of the tile sees, as one run of indices: [0, na) are positions 0 .. na-1, the rest lo .. jlast
  const int qfirst = pos0 + tq, jlast = qfirst + qn - 1;
  const int lo = first_seen(qfirst, a.window, a.chunk);
  const int na = min(a.keep, lo);
  const int total = na + (jlast - lo + 1);
  auto pos_of = [&](int iv) { return iv < na ? iv : lo + (iv - na); };
  const bool wave_live = wave * 32 < qn;
  const int wq0 = qfirst + wave * 32, wq1 = min(wq0 + 31, jlast);      // positions of this wave's queries
  const int qlo = first_seen(qpos, a.window, a.chunk), wlo0 = first_seen(wq0, a.window, a.chunk), wlo1 = first_seen(wq1, a.window, a.chunk);

  constexpr float LOG2E = 1.4426950408889634f;
  const float scale2 = (a.head_scale ? a.scale * a.head_scale[head] : a.scale) * LOG2E;
  // what the weights are measured from: the largest score when it last moved, and 8 more, so that no weight exceeds 1 before the sums move again
  constexpr float ROOM = 8.f;
  float m = a.sink && group == 0 ? a.sink[head] * LOG2E + ROOM : -INFINITY;
  float l = (a.sink && group == 0 && hb == 0) ? 1.f / (1 << static_cast<int>(ROOM)) : 0.f;      // the sink counts once per query
  const unsigned char* vbase = vl + (4 * hb + ((lane >> 2) & 3)) * VROW + (16 * ((lane >> 4) & 1) + 4 * (lane & 3)) * 2;
  const unsigned char* kbase = kl + r * KROW + hb * 16;

  const bf16_t *kc = a.kc + slot * a.kc_slot + kvh * a.kc_head, *kn = a.kn + kvh * a.k_head;
  const bf16_t *vc = a.vc + slot * a.vc_slot + kvh * a.vc_head, *vn = a.vn + kvh * a.v_head;
  auto cached = [&](int j) { return j < a.keep ? j : a.keep + (j - a.keep) % a.ring; };
  auto krow = [&](int j) -> const bf16_t* {
    return j < pos0 ? kc + static_cast<int64_t>(cached(j)) * a.kc_row : kn + static_cast<int64_t>(row0 + (j - pos0)) * a.k_row;
  };
  auto vrow = [&](int j) -> const bf16_t* {
    return j < pos0 ? vc + static_cast<int64_t>(cached(j)) * a.vc_row : vn + static_cast<int64_t>(row0 + (j - pos0)) * a.v_row;
  };

  u32x4 kr[KP::N], vr[VP::N];
  // 32 bits of byte offset reach across a tile's rows
  const bool near = max(max(a.k_row, a.v_row), max(a.kc_row, a.vc_row)) < (1 << 22);
  // Rows of a whole tile that follow each other in one buffer -- nearly all tiles of long sequences -- come by buffer loads: the tile's place is
  // scalar, a lane adds a multiple of the stride, and channels beyond the head lie out of range and read as zeros.  Tiles that the end of the
  // keys, the kept rows, the ring's seam or the first new row cuts find every row by itself (of 16 vector instructions per matrix product the
  // search for rows was 10).
  auto fetch = [&](int it) {
    const int j0 = pos_of(it), j1 = j0 + KT;
    bool whole = BUFS == 2 && near && it + KT <= total && (it >= na || it + KT <= na);
    int at = row0 + (j0 - pos0);
    if (whole && j0 < pos0) {
      at = cached(j0);
      whole = j1 <= pos0 && (j1 <= a.keep || (j0 >= a.keep && at + KT <= a.keep + a.ring));
    }
    if (whole) {
      const bool old = j0 < pos0;
      const int ks = static_cast<int>(old ? a.kc_row : a.k_row) * 2, vs = static_cast<int>(old ? a.vc_row : a.v_row) * 2;
      const bf16_t* kp = (old ? kc : kn) + static_cast<int64_t>(at) * (ks / 2);
      const bf16_t* vp = (old ? vc : vn) + static_cast<int64_t>(at) * (vs / 2);
      const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(kp), 0, (KT - 1) * ks + a.dk * 2, 0x00020000);
      const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(vp), 0, (KT - 1) * vs + a.dv * 2, 0x00020000);
#pragma unroll
      for (int i = 0; i < KP::N; ++i) {
        const int c = KP::piece(tid, i), off = KP::row(tid, i) * ks + c * 16;
        kr[i] = __builtin_amdgcn_raw_buffer_load_b128(krs, KP::used(tid, i) && c * 8 < a.dk ? off : 0x7ffffff0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < VP::N; ++i) {
        const int c = VP::piece(tid, i), off = VP::row(tid, i) * vs + c * 16;
        vr[i] = __builtin_amdgcn_raw_buffer_load_b128(vrs, VP::used(tid, i) && c * 8 < a.dv ? off : 0x7ffffff0, 0, 0);
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < KP::N; ++i) {
      const int iv = it + KP::row(tid, i), c = KP::piece(tid, i);
      kr[i] = u32x4{0, 0, 0, 0};
      if (KP::used(tid, i) && iv < total && c * 8 < a.dk) kr[i] = *reinterpret_cast<const u32x4*>(krow(pos_of(iv)) + c * 8);
    }
#pragma unroll
    for (int i = 0; i < VP::N; ++i) {
      const int iv = it + VP::row(tid, i), c = VP::piece(tid, i);
      vr[i] = u32x4{0, 0, 0, 0};
      if (VP::used(tid, i) && iv < total && c * 8 < a.dv) vr[i] = *reinterpret_cast<const u32x4*>(vrow(pos_of(iv)) + c * 8);
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

  // Two buffers, one barrier a tile: behind it tile t is in buffer t % 2 and tile t + 1 in registers; it is parked in the other buffer, whose
  // readers have all passed the barrier, and tile t + 2 is asked for.  One buffer: tile t + 1 is asked for while tile t is read.
  const int i1 = group * KT, rounds = (total + STEP - 1) / STEP;        // (every group runs as many rounds: the barriers are common)
  if (i1 < total) fetch(i1);
  if constexpr (BUFS == 2) {
    if (i1 < total) stage(0);
    if (i1 + STEP < total) fetch(i1 + STEP);
  }
  for (int round = 0; round < rounds; ++round) {
    const int it = i1 + round * STEP;
    __syncthreads();
    if constexpr (BUFS == 2) {
      if (it + STEP < total) stage((round + 1) & 1);
      if (it + 2 * STEP < total) fetch(it + 2 * STEP);
    } else {
      if (it < total) stage(0);
      __syncthreads();
      if (it + STEP < total) fetch(it + STEP);
    }
    // wave-uniform: no key of the tile is seen by a query of this wave
    if (!wave_live || it >= total) continue;
    const int jmin = pos_of(it), jmax = pos_of(min(it + KT, total) - 1);
    if (jmin > wq1 || (jmax < wlo0 && jmin >= a.keep)) continue;

    // fragments are read in bulk ahead of the products that take them; a slot is filled again as its product leaves
    const unsigned char* kb = kbase + (BUFS == 2 ? round & 1 : 0) * Shape::BUF;
    const unsigned char* vb = vbase + (BUFS == 2 ? round & 1 : 0) * Shape::BUF;
    constexpr int NK = KS * NH, NV = DT * 2 * NH, SLOTS = Shape::SLOTS, NF = SLOTS < NV ? SLOTS : NV;
    auto kfrag = [&](int i) { return *reinterpret_cast<const u32x4*>(kb + i / KS * 32 * KROW + i % KS * 32); };
    auto vfrag = [&](int i) {
      const int dt = i / (2 * NH), j = i % (2 * NH);
      const u32x2 v0 = lds_read_tr(vb + 16 * j * VROW + dt * 64);
      const u32x2 v1 = lds_read_tr(vb + (16 * j + 8) * VROW + dt * 64);
      return u32x4{v0.x, v0.y, v1.x, v1.y};
    };
    u32x4 fr[SLOTS ? SLOTS : 1];
    f32x16 st[NH];
#pragma unroll
    for (int h = 0; h < NH; ++h) st[h] = f32x16{0};
    if constexpr (SLOTS) {
#pragma unroll
      for (int i = 0; i < SLOTS; ++i) fr[i] = kfrag(i);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < NK; ++i) {
        st[i / KS] = mfma_bf16(fr[i % SLOTS], qf[i % KS], st[i / KS]);
        if (i + SLOTS < NK) fr[i % SLOTS] = kfrag(i + SLOTS);
        if (i % KS == KS - 1) __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < NF; ++i) fr[i] = vfrag(i);           // the first fragments of V^T are read under the exponentials
      __builtin_amdgcn_sched_barrier(0);
    } else {
#pragma unroll
      for (int i = 0; i < NK; ++i) st[i / KS] = mfma_bf16(kfrag(i), qf[i % KS], st[i / KS]);
    }
    // scores in units of ln 2 (the exponentials below are base 2).  Inside the mask -- every key of the tile before every query of the
    // wave, inside every window -- nothing is tested per score, the scale meets the maximum once and the rest inside the exponent.
    const bool inside = it + KT <= total && jmax <= wq0 && (jmin >= wlo1 || jmax < a.keep);
    float mx;
    if (inside) {
      float e0 = st[0][0];
      if (scale2 >= 0.f) {
#pragma unroll
        for (int h = 0; h < NH; ++h)
#pragma unroll
          for (int e = 0; e < 16; ++e) e0 = fmaxf(e0, st[h][e]);
      } else {
#pragma unroll
        for (int h = 0; h < NH; ++h)
#pragma unroll
          for (int e = 0; e < 16; ++e) e0 = fminf(e0, st[h][e]);
      }
      mx = e0 * scale2;
    } else {
      mx = -INFINITY;
#pragma unroll
      for (int h = 0; h < NH; ++h)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int iv = it + 32 * h + 8 * (e >> 2) + 4 * hb + (e & 3);
          const int j = pos_of(iv);
          const bool seen = qvalid && iv < total && j <= qpos && (j >= qlo || j < a.keep);
          st[h][e] = seen ? st[h][e] * scale2 : -INFINITY;
          mx = fmaxf(mx, st[h][e]);
        }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));                   // the other half of the query's scores
    // the sums move to a new maximum only where a weight would exceed 1 (weights of 2^-8 keep as many bits, the factor falls out at the end; weights
    // above 1 would take sums of values near the end of the range past it).  The first scores always move it; with nothing seen yet and no sink every
    // weight below is 2^-inf = 0
    if (__any(mx > m)) {
      const float m_new = fmaxf(m, mx + ROOM);
      const float alpha = __builtin_amdgcn_exp2f(m - (m_new == -INFINITY ? 0.f : m_new));
      m = m_new;
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[dt][e] *= alpha;
    }
    const float m_ref = m == -INFINITY ? 0.f : m, f2 = inside ? scale2 : 1.f;
    float ps = 0.f;
    u32x4 pf[2 * NH];
#pragma unroll
    for (int h = 0; h < NH; ++h) {
#pragma unroll
      for (int e = 0; e < 16; ++e) { st[h][e] = __builtin_amdgcn_exp2f(fmaf(st[h][e], f2, -m_ref)); ps += st[h][e]; }
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
        pf[2 * h + tt] = u32x4{pack2(st[h][8 * tt], st[h][8 * tt + 1]), pack2(st[h][8 * tt + 2], st[h][8 * tt + 3]),
                               pack2(st[h][8 * tt + 4], st[h][8 * tt + 5]), pack2(st[h][8 * tt + 6], st[h][8 * tt + 7])};
    }
    l += ps;
    if constexpr (SLOTS) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      o[i / (2 * NH)] = mfma_bf16(SLOTS ? fr[i % (NF ? NF : 1)] : vfrag(i), pf[i % (2 * NH)], o[i / (2 * NH)]);
      if (SLOTS && i + NF < NV) fr[i % (NF ? NF : 1)] = vfrag(i + NF);
    }
  }

  if constexpr (GROUPS > 1) {
    float* join = reinterpret_cast<float*>(all_lds) + wave * ((DT * 16 + 2) * 64) + lane;
    __syncthreads();
    if (group == 1) {
      join[0] = m;
      join[64] = l;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int e = 0; e < 16; ++e) join[(2 + dt * 16 + e) * 64] = o[dt][e];
    }
    __syncthreads();
    if (group == 1) return;
    const float m1 = join[0], mj = fmaxf(m, m1), mr = mj == -INFINITY ? 0.f : mj;
    const float f0 = __builtin_amdgcn_exp2f(m - mr), f1 = __builtin_amdgcn_exp2f(m1 - mr);
    l = l * f0 + join[64] * f1;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[dt][e] = o[dt][e] * f0 + join[(2 + dt * 16 + e) * 64] * f1;
  }
  l += __shfl_xor(l, 32, 64);
  if (qvalid) {
    const int64_t row = row0 + tq + qloc;
    float f = 1.f / l;
    if (a.gate && !a.gate_channels) f *= sigmoid_<true>(to_f32(a.gate[row * a.gate_row + head]));
    bf16_t* op = a.out + row * a.out_row + head * a.dv;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const int d = dt * 32 + 8 * q4 + 4 * hb;
        if (d < a.dv)                                          // dv is a multiple of 8: the four channels are inside together
          *reinterpret_cast<u32x2*>(op + d) = out4(a, row, head, d, o[dt], q4, f);
      }
  }
}

// Steps of single rows (decoding): the query heads that share a key/value head are the 32 "query rows" of the same two products,
// all at one position, so a key tile staged once serves every head of the group.  One workgroup = one (row, kv head, 32 heads of
// its group, share of the key tiles); every wave forms all scores of a tile (the weights must be the same in all of them) and
// owns every fourth 32-channel block of the value product.  No mask besides the end of the key run.  With key splits a workgroup
// leaves (sum, maximum, denominator) per head for sink_reduce_kernel, else it finishes the row itself.
// ALIAS: the values are the first dv channels of the key rows (one staged tile serves both products).
// A launch is one trip to memory and one pass over code that is read cold (1.2 ns a byte): FULL drops the tests of heads smaller than <DK, DV> and of
// groups of more than 32 heads.
template <int DK, int DV, bool ALIAS, bool FULL>
__global__ __launch_bounds__(256) void sink_group_kernel(const SinkTileArgs a, const int* __restrict__ tok, int R, int splits, float* __restrict__ partial) {
  constexpr int KT = 32;
  constexpr int KROW = DK * 2 + 16;
  constexpr int VROW = ALIAS ? KROW : DV * 2 + 64;
  constexpr int KS = DK / 16, DT = DV / 32, DTW = (DT + 3) / 4;
  // long rows: the channels of the score product are shared out over the four waves (a quarter of the dependent matrix-core steps
  // and of the query fragments each); the four partial score tiles meet in LDS and every wave adds them in the same order, so all
  // waves hold identical scores.  The registers this frees hold the next key tile while the current one is computed.
  constexpr bool SPLITK = KS >= 16;
  constexpr int KSW = SPLITK ? (KS + 3) / 4 : KS;
  constexpr int TILE_BYTES = KT * KROW + (ALIAS ? 0 : KT * VROW);
  constexpr int SROW = 80;                                              // bytes of a lane's 16 partial scores (+16: conflict-free 16-byte accesses)
  __shared__ __attribute__((aligned(16))) unsigned char lds[TILE_BYTES + (SPLITK ? 4 * 64 * SROW : 0)];
  unsigned char* kl = lds;
  unsigned char* vl = ALIAS ? lds : lds + KT * KROW;
  unsigned char* sred = lds + TILE_BYTES;                               // [4 waves][64 lanes][16]

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 31, hb = lane >> 5;
  const int64_t t = blockIdx.x;
  const int chunks = FULL ? 1 : (R + 31) / 32;
  const int kvh = FULL ? blockIdx.y : blockIdx.y / chunks, hloc = FULL ? r : (blockIdx.y % chunks) * 32 + r;
  const bool hvalid = hloc < R;
  const int head = kvh * R + min(hloc, R - 1);
  const int b = tok[2 * t], pos = tok[2 * t + 1];
  const int slot = a.seq[4 * b], pos0 = a.seq[4 * b + 1], row0 = a.seq[4 * b + 3];

  const int ks0 = SPLITK ? wave * KSW : 0;                              // this wave's steps of the score product: ks0 .. ks0 + KSW - 1
  u32x4 qf[KSW];
  {
    const bf16_t* qp = a.q + t * a.q_row + head * a.q_head;
#pragma unroll
    for (int i = 0; i < KSW; ++i) {
      const int c = (ks0 + i) * 16 + hb * 8;
      qf[i] = (FULL && (!SPLITK || KS % 4 == 0)) || (ks0 + i < KS && c < a.dk) ? *reinterpret_cast<const u32x4*>(qp + c) : u32x4{0, 0, 0, 0};
    }
  }
  f32x16 o[DTW];
#pragma unroll
  for (int i = 0; i < DTW; ++i) o[i] = f32x16{0};

  const int lo = first_seen(pos, a.window, a.chunk);
  const int na = min(a.keep, lo);
  const int total = na + (pos - lo + 1);

  constexpr float LOG2E = 1.4426950408889634f;
  const float scale2 = (a.head_scale ? a.scale * a.head_scale[head] : a.scale) * LOG2E;
  const bool own_sink = a.sink && splits == 1;                          // split key tiles: the sink joins in the reduce
  float m = own_sink ? a.sink[head] * LOG2E : -INFINITY;
  float l = (own_sink && hb == 0) ? 1.f : 0.f;
  const unsigned char* vbase = vl + (4 * hb + ((lane >> 2) & 3)) * VROW + (16 * ((lane >> 4) & 1) + 4 * (lane & 3)) * 2;
  const unsigned char* kbase = kl + r * KROW + hb * 16;

  // A key (and value) tile: global -> registers -> LDS, one tile ahead.  A thread looks each of its rows up once and takes all its pieces of it from there.
  // The last key's row is read in place of those behind it; values behind it go to LDS as zeros, so that a weight of zero
  // meets no infinity (an infinite channel of a row that is key and value is no number in either case).
  typedef RowPieces<DK, KT> KP;
  typedef RowPieces<ALIAS ? 32 : DV, KT> VP;
  u32x4 kr[KP::N], vr[VP::N];
  const bool round = pos >= a.keep + a.ring;                            // the ring has come round
  auto row_of = [&](const bf16_t* old, int64_t old_row, const bf16_t* fresh, int64_t fresh_row, int iv) -> const bf16_t* {
    iv = min(iv, total - 1);
    const int j = iv < na ? iv : lo + (iv - na);
    return j < pos0 ? old + static_cast<int64_t>(round && j >= a.keep ? a.keep + (j - a.keep) % a.ring : j) * old_row
                    : fresh + static_cast<int64_t>(j - pos0) * fresh_row;
  };
  const bf16_t *kc = a.kc + slot * a.kc_slot + kvh * a.kc_head, *kn = a.kn + row0 * a.k_row + kvh * a.k_head;
  const bf16_t *vc = a.vc + slot * a.vc_slot + kvh * a.vc_head, *vn = a.vn + row0 * a.v_row + kvh * a.v_head;
  auto load = [&](auto pieces, u32x4* regs, const bf16_t* old, int64_t old_row, const bf16_t* fresh, int64_t fresh_row, int it, int width) {
    typedef decltype(pieces) P;
    const bf16_t* row = nullptr;
#pragma unroll
    for (int i = 0; i < P::N; ++i) {
      if (P::LINEAR || i % P::PER == 0) row = row_of(old, old_row, fresh, fresh_row, it + P::row(tid, i));
      const int c = P::piece(tid, i);
      regs[i] = P::used(tid, i) && (FULL || c * 8 < width) ? *reinterpret_cast<const u32x4*>(row + c * 8) : u32x4{0, 0, 0, 0};
    }
  };

  const int it0 = static_cast<int>(blockIdx.z) * KT, step = KT * splits;
  for (int it = it0;; it += step) {                           // (one loop body: a launch of one tile reads all of its code cold)
    if (it < total) {
      load(KP{}, kr, kc, a.kc_row, kn, a.k_row, it, a.dk);
      if constexpr (!ALIAS) load(VP{}, vr, vc, a.vc_row, vn, a.v_row, it, a.dv);
    }
    if (it != it0) {                                          // the tile before is multiplied while this one travels
      f32x16 st = f32x16{0};
#pragma unroll
      for (int i = 0; i < KSW; ++i)
        if (ks0 + i < KS) st = mfma_bf16(*reinterpret_cast<const u32x4*>(kbase + (ks0 + i) * 32), qf[i], st);      // wave-uniform test
      if constexpr (SPLITK) {
#pragma unroll
        for (int e = 0; e < 4; ++e) *reinterpret_cast<f32x4v*>(sred + (wave * 64 + lane) * SROW + e * 16) = f32x4v{st[4 * e], st[4 * e + 1], st[4 * e + 2], st[4 * e + 3]};
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          f32x4v p[4];
#pragma unroll
          for (int w = 0; w < 4; ++w) p[w] = *reinterpret_cast<const f32x4v*>(sred + (w * 64 + lane) * SROW + e * 16);
#pragma unroll
          for (int i = 0; i < 4; ++i) st[4 * e + i] = (p[0][i] + p[1][i]) + (p[2][i] + p[3][i]);
        }
      }
      const int first = it - step + 4 * hb;
      float s[16];
      float mx = -INFINITY;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        s[e] = first + 8 * (e >> 2) + (e & 3) < total ? st[e] * scale2 : -INFINITY;
        mx = fmaxf(mx, s[e]);
      }
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));                 // finite: a tile holds at least one key
      const float m_new = fmaxf(m, mx);
      const float alpha = __builtin_amdgcn_exp2f(m - m_new);
      m = m_new;
      float ps = 0.f;
#pragma unroll
      for (int e = 0; e < 16; ++e) { s[e] = __builtin_amdgcn_exp2f(s[e] - m_new); ps += s[e]; }
      l = l * alpha + ps;
      u32x4 gf[2];
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
        gf[tt] = u32x4{pack2(s[8 * tt], s[8 * tt + 1]), pack2(s[8 * tt + 2], s[8 * tt + 3]), pack2(s[8 * tt + 4], s[8 * tt + 5]),
                       pack2(s[8 * tt + 6], s[8 * tt + 7])};
#pragma unroll
      for (int i = 0; i < DTW; ++i) {
        const int dt = wave + 4 * i;                          // wave-uniform
        if (DT % 4 == 0 || dt < DT) {
          if (it != it0 + step)
#pragma unroll
            for (int e = 0; e < 16; ++e) o[i][e] *= alpha;
#pragma unroll
          for (int tt = 0; tt < 2; ++tt) {
            const u32x2 v0 = lds_read_tr(vbase + (16 * tt) * VROW + dt * 64);
            const u32x2 v1 = lds_read_tr(vbase + (16 * tt + 8) * VROW + dt * 64);
            o[i] = mfma_bf16(u32x4{v0.x, v0.y, v1.x, v1.y}, gf[tt], o[i]);
          }
        }
      }
    }
    if (it >= total) break;
    __syncthreads();                                          // the tile before (and its partial scores) has been consumed
#pragma unroll
    for (int i = 0; i < KP::N; ++i)
      if (KP::used(tid, i)) *reinterpret_cast<u32x4*>(kl + KP::row(tid, i) * KROW + KP::piece(tid, i) * 16) = kr[i];
    if constexpr (!ALIAS) {
#pragma unroll
      for (int i = 0; i < VP::N; ++i)
        if (VP::used(tid, i))
          *reinterpret_cast<u32x4*>(vl + VP::row(tid, i) * VROW + VP::piece(tid, i) * 16) = it + VP::row(tid, i) < total ? vr[i] : u32x4{0, 0, 0, 0};
    }
    __syncthreads();
  }

  l += __shfl_xor(l, 32, 64);
  if (!hvalid) return;
  if (splits > 1) {
    const int pw = partial_width(a.dv);
    float* prow = partial + ((static_cast<int64_t>(blockIdx.z) * gridDim.x + t) * a.H + head) * pw;
#pragma unroll
    for (int i = 0; i < DTW; ++i) {
      const int dt = wave + 4 * i;
      if (DT % 4 == 0 || dt < DT)
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          const int d = dt * 32 + 8 * q4 + 4 * hb;
          if (FULL || d < a.dv) *reinterpret_cast<float4*>(prow + d) = float4{o[i][4 * q4], o[i][4 * q4 + 1], o[i][4 * q4 + 2], o[i][4 * q4 + 3]};
        }
    }
    if (wave == 0 && hb == 0) { prow[pw - 2] = m / LOG2E; prow[pw - 1] = l; }
    return;
  }
  float f = 1.f / l;
  if (a.gate && !a.gate_channels) f *= sigmoid_<true>(to_f32(a.gate[t * a.gate_row + head]));
  bf16_t* op = a.out + t * a.out_row + head * a.dv;
#pragma unroll
  for (int i = 0; i < DTW; ++i) {
    const int dt = wave + 4 * i;
    if (dt < DT)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const int d = dt * 32 + 8 * q4 + 4 * hb;
        if (d < a.dv)
          *reinterpret_cast<u32x2*>(op + d) = out4(a, t, head, d, o[i], q4, f);
      }
  }
}

template <int DK, int DV, bool ALIAS>
int launch_group(const SinkTileArgs& t, const gbxm_sink_attn_args& a, const gbxm_slot_rows*& rows, hipStream_t s) {
  const int R = a.H / a.G, chunks = (R + 31) / 32;
  int splits = 1;
  const int64_t groups = a.T * a.G * chunks;
  if (a.partial && a.partial_splits > 1 && groups < 256) {
    splits = static_cast<int>(std::min<int64_t>(std::min<int64_t>(512 / groups, 64), a.partial_splits));
    if (splits < 2) splits = 1;
  }
  const dim3 grid(a.T, a.G * chunks, splits);
  if (a.dk == DK && a.dv == DV && R <= 32) sink_group_kernel<DK, DV, ALIAS, true><<<grid, 256, 0, s>>>(t, a.tok, R, splits, static_cast<float*>(a.partial));
  else sink_group_kernel<DK, DV, ALIAS, false><<<grid, 256, 0, s>>>(t, a.tok, R, splits, static_cast<float*>(a.partial));
  const int rc = after_launch("sink_attention (grouped rows)");
  if (rc != GBXM_OK || splits == 1) return rc;
  return launch_sink_reduce(a, splits, std::exchange(rows, nullptr), s);
}

// A workgroup = a query tile of a head, or (PAIRS, one group) two, one from each end of the list; tiles that see many keys, at the end of the step's list, go
// first.  Heads are the fast index, those of a key / value head G apart, so that an XCD's workgroups (every eighth) meet in few heads' keys.
template <int DK, int DV, int GROUPS, int KT, int BUFS, bool PAIRS>
__global__ __launch_bounds__((256 * GROUPS), (SinkShape<DK, DV, GROUPS, KT, BUFS>::WAVES)) void sink_tile_kernel(const SinkTileArgs a, const int n_tiles) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int place = blockIdx.x % a.H, head = place % a.G * (a.H / a.G) + place / a.G, at = blockIdx.x / a.H;
  sink_tile<DK, DV, GROUPS, KT, BUFS>(a, n_tiles - 1 - at, head, lds);
  if constexpr (PAIRS) {
    if (2 * at == n_tiles - 1) return;
    __syncthreads();                                         // (the first tile's last keys have been read)
    sink_tile<DK, DV, GROUPS, KT, BUFS>(a, at, head, lds);
  }
}

template <int DK, int DV, int GROUPS, int KT, int BUFS, bool PAIRS = false>
int launch_groups(const SinkTileArgs& t, int n_tiles, hipStream_t s) {
  static_assert(!PAIRS || GROUPS == 1, "a second group leaves before the second tile");
  constexpr int bytes = SinkShape<DK, DV, GROUPS, KT, BUFS>::LDS;
  static OncePerDevice once;
  if (once.pending()) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(sink_tile_kernel<DK, DV, GROUPS, KT, BUFS, PAIRS>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return hip_fail(e, "sink_attention (tiles)");
    once.done();
  }
  const unsigned grid = static_cast<unsigned>(t.H) * (PAIRS ? (n_tiles + 1) / 2 : n_tiles);
  sink_tile_kernel<DK, DV, GROUPS, KT, BUFS, PAIRS><<<grid, 256 * GROUPS, bytes, s>>>(t, n_tiles);
  return after_launch("sink_attention (tiles)");
}

// Which form, by tiles times heads n, the longest sequence's keys (0: unknown, long) and whether the others are about as long (even).  Measured in a
// replayed graph, us, 16 heads of <128, 128> unless named.
// Up to 64 keys: one group, 32 keys, one buffer, the form with most waves (start-up is all there is: 1 x 20 rows 6.4 | one group of two buffers 7.8 |
// two groups 8.5; 64 x 20 rows 9.9 | 15.6 | 29.7); up to 224 also where there is more than a tile a CU: 64 x 200 60 | 70 | 94, 8 .. 163 rows x 32
// 17.1 | 19.2 | 27.5, <64, 64> 32 heads, 64 x 128 32 | 35 | 60.
// Two groups halve the chain of key tiles behind the last query tile, at one workgroup a CU.  Two groups | one of two buffers: 4 x 256 rows 13.3 |
// 14.2, 2 x 500 17.8 | 21.0; small heads of few keys are done before a second buffer pays: two groups of one buffer | of two, <64, 64> 8 x 100 7.9 |
// 8.6, <32, 32> 16 x 200 8.5 | 9.5.  Beyond a tile a CU only long chains gain: 8 x 500 36.8 | 31.1, 4 x 1000 49.5 | 45.8, 2 x 1300 33.0 | 42.6, 2 x 2000 58 |
// 72, 4 000 rows 91 | 123, <192, 128> 2 000 + 777 rows 59 | 90; a chip whose two places a CU fill has less to wait for: 32 heads 2 x 1300 60 | 52, 3 000 rows
// 117 | 108, 3 700 157 | 147, <64, 64> 2 500 62 | 59, <192, 128> 2 500 114 | 117, 3 000 148 | 138, 16 heads 7 500 374 | 335; heads of 32 are long at their chain: 32
// heads 2 x 1300 28.7 | 31.3, 3 x 1100 30.3 | 35.5.
// Two tiles a workgroup where tiles of sequences of one length would fill the places twice: one tile | two, 32 heads, 32 x 128 rows 31.9 | 31.1 (32 keys, one
// buffer 34.7), 8 x 500 48.6 | 43.0, 4 x 1000 67.7 | 58.8, 3 x 1100 62 | 59, 16 heads, 16 x 500 56.7 | 45.3, 32 x 256 41.3 | 35.7, <192, 128> 16 x 500 68 | 55, <256, 256> 8 heads 16 x 500 87 |
// 65, <64, 64> 16 x 500 37.8 | 34.3; of many lengths the long ones first even out better: 60 .. 810 rows x 16 46.6 | 53.3, 100 .. 660 x 8, 32 heads 38.3 | 44.9; so do fewer or
// more tiles: 32 heads, 8 x 300 31 | 34, 4 x 700 46.7 | 47.6, 12 x 400 57.8 | 67.1.  Heads of 32: two groups of one buffer instead, 4 x 1000 40.7 | 32.8, 8 x 500 26.8 | 23.9, and pairs of
// one buffer at twice as many tiles, 16 x 500 44.4 | 39.1, 32 x 256 32.7 | 29.4.
constexpr int FEW_TILES = 960, LONG_TILES = 640;
template <int DK, int DV>
int launch(const SinkTileArgs& t, int n_tiles, int longest, bool even, hipStream_t s) {
  constexpr int KT = DK + DV > 256 ? 32 : 64;                // (larger heads: 64 would cost the second wave per SIMD)
  constexpr int PLACES = DK + DV <= 320 ? 512 : 256;
  constexpr bool SMALL = DK + DV <= 64;
  const int64_t n = static_cast<int64_t>(t.H) * n_tiles;
  const int keys = longest > 0 ? longest : 1 << 30;
  const auto twice = [&](int places) { return even && keys > 64 && keys <= 1100 && 8 * n > 13 * places && n <= 2 * places; };
  if constexpr (DK + DV > 128) {
    if (twice(PLACES)) return launch_groups<DK, DV, 1, KT, 2, true>(t, n_tiles, s);
  }
  if (keys <= 64 || (keys <= 224 && n > (SMALL ? FEW_TILES : 256))) return launch_groups<DK, DV, 1, 32, 1>(t, n_tiles, s);
  if constexpr (DK + DV < 256) {
    if ((keys <= (SMALL ? 256 : 128) && n <= FEW_TILES) || (SMALL && twice(PLACES))) return launch_groups<DK, DV, 2, KT, 1>(t, n_tiles, s);
  }
  if constexpr (SMALL) {
    if (twice(2 * PLACES)) return launch_groups<DK, DV, 1, KT, 1, true>(t, n_tiles, s);
  } else if constexpr (DK + DV <= 128) {
    if (twice(PLACES)) return launch_groups<DK, DV, 1, KT, 2, true>(t, n_tiles, s);
  }
  if constexpr (DK + DV <= 320) {
    if (n <= 256 || (n <= (SMALL ? FEW_TILES : LONG_TILES) && keys > 1024)) return launch_groups<DK, DV, 2, KT, 2>(t, n_tiles, s);
  }
  return launch_groups<DK, DV, 1, KT, 2>(t, n_tiles, s);
}

constexpr int CAPS[][2] = {{32, 32}, {64, 64}, {64, 128}, {96, 96}, {128, 128}, {192, 128}, {256, 256}};

}  // namespace

bool sink_tiles_shape(int dk, int dv) {
  if (dk % 8 || dv % 8) return false;
  for (const auto& c : CAPS)
    if (dk <= c[0] && dv <= c[1]) return true;
  return false;
}

static bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

static bool tile_operands(const gbxm_sink_attn_args& a) {
  if ((a.q_row | a.q_head | a.k_row | a.k_head | a.v_row | a.v_head) % 8 || !aligned16(a.q) || !aligned16(a.k_new) || !aligned16(a.v_new) ||
      !aligned16(a.out) || a.out_row % 8)
    return false;
  if (a.gate && a.gate_channels && (a.gate_row % 4 || reinterpret_cast<uintptr_t>(a.gate) % 8)) return false;
  if (a.kcache && ((a.kc_slot | a.kc_row | a.kc_head | a.vc_slot | a.vc_row | a.vc_head) % 8 || !aligned16(a.kcache) || !aligned16(a.vcache))) return false;
  return true;
}

static SinkTileArgs tile_args(const gbxm_sink_attn_args& a) {
  return SinkTileArgs{static_cast<const bf16_t*>(a.q), static_cast<const bf16_t*>(a.k_new), static_cast<const bf16_t*>(a.v_new),
                      static_cast<const bf16_t*>(a.kcache), static_cast<const bf16_t*>(a.vcache), a.seq, a.tiles, static_cast<bf16_t*>(a.out), a.sink,
                      static_cast<const bf16_t*>(a.gate), a.q_row, a.q_head, a.k_row, a.k_head, a.v_row, a.v_head, a.kc_slot, a.kc_row, a.kc_head,
                      a.vc_slot, a.vc_row, a.vc_head, a.gate_row, a.q_tile, a.H, a.G, a.dk, a.dv, a.window, a.keep, a.ring, a.chunk, a.scale, a.head_scale,
                      a.out_row > 0 ? a.out_row : static_cast<int64_t>(a.H) * a.dv, a.gate && a.gate_channels};
}

int launch_sink_tiles(const gbxm_sink_attn_args& a, hipStream_t s) {
  if (!sink_tiles_shape(a.dk, a.dv) || a.q_tile != 128 || static_cast<int64_t>(a.H) * a.n_tiles > 0x7fffffff || !tile_operands(a)) return GBXM_ERR_UNSUPPORTED;
  const SinkTileArgs t = tile_args(a);
  const bool even = a.longest > 0 && 8 * a.T >= 7 * static_cast<int64_t>(a.B) * a.longest;
#define GBXM_TILE(DK_, DV_) if (a.dk <= DK_ && a.dv <= DV_) return launch<DK_, DV_>(t, a.n_tiles, a.longest, even, s)
  GBXM_TILE(32, 32); GBXM_TILE(64, 64); GBXM_TILE(64, 128); GBXM_TILE(96, 96); GBXM_TILE(128, 128); GBXM_TILE(192, 128); GBXM_TILE(256, 256);
#undef GBXM_TILE
  return GBXM_ERR_UNSUPPORTED;
}

// values that are the leading channels of the key rows (same buffers, same strides): one staged tile serves both products
static bool values_alias_keys(const gbxm_sink_attn_args& a) {
  return a.G == 1 && a.dv <= a.dk && a.v_new == a.k_new && (a.T == 1 || a.v_row == a.k_row) &&     // (one row: its stride is never used)
         (!a.kcache || (a.vcache == a.kcache && a.vc_slot == a.kc_slot && a.vc_row == a.kc_row));
}

bool sink_group_shape(int dk, int dv, bool alias) {
  if (dk % 8 || dv % 8) return false;
  if (alias) return dk <= 576 && dv <= 512;
  return sink_tiles_shape(dk, dv);
}

int launch_sink_group(const gbxm_sink_attn_args& a, const gbxm_slot_rows*& rows, hipStream_t s) {
  const bool alias = values_alias_keys(a);
  const int chunks = (a.H / a.G + 31) / 32;
  if (!sink_group_shape(a.dk, a.dv, alias) || a.G * chunks > 65535 || !tile_operands(a)) return GBXM_ERR_UNSUPPORTED;
  const SinkTileArgs t = tile_args(a);
  if (alias) {
#define GBXM_GROUP(DK_, DV_) if (a.dk <= DK_ && a.dv <= DV_) return launch_group<DK_, DV_, true>(t, a, rows, s)
    // (latent rows without rotated channels have capacities of their own, which they fill: 62 launches of 256 / 256 as 320 / 256 308 us | 296)
    GBXM_GROUP(96, 96); GBXM_GROUP(160, 128); GBXM_GROUP(256, 256); GBXM_GROUP(320, 256); GBXM_GROUP(512, 512); GBXM_GROUP(576, 512);
#undef GBXM_GROUP
    return GBXM_ERR_UNSUPPORTED;
  }
#define GBXM_GROUP(DK_, DV_) if (a.dk <= DK_ && a.dv <= DV_) return launch_group<DK_, DV_, false>(t, a, rows, s)
  GBXM_GROUP(32, 32); GBXM_GROUP(64, 64); GBXM_GROUP(64, 128); GBXM_GROUP(96, 96); GBXM_GROUP(128, 128); GBXM_GROUP(192, 128); GBXM_GROUP(256, 256);
#undef GBXM_GROUP
  return GBXM_ERR_UNSUPPORTED;
}

}  // namespace gbxm
