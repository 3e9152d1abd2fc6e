// The decayed matrix states token by token (mixers_state.hip): a device function, which the chunks' launch (mixers_state_mfma.hip) runs too for the
// sequences that do not go by chunks.
#pragma once
#include "mixers_mfma.h"

namespace gbxm {

// A step's rows, states and shape.
struct StateArgs {
  const float* r;
  int64_t r_stride;
  float *state, *out;
  const int* seq;
  int B, H, G, dk, dv;
};

// Sequences of STATE_CHUNKS_FROM rows and more go by chunks of STATE_CHUNK rows (mixers_state_mfma.hip) -- a rule of the sequence alone, so that its sums do not
// depend on what else is in the step -- their heads whose numbers pass the check of their
// chunks (`flags` [H][places], 0: passed).  Sequence b's first place is row0 / STATE_CHUNK + b, which leaves room for its part of a chunk.
constexpr int STATE_CHUNK = 16;
struct StateChunks { const int* flags; int places; };
__device__ __forceinline__ int first_chunk(int row0, int b) { return row0 / STATE_CHUNK + b; }
// (a workgroup asks with all its threads)
__device__ __forceinline__ bool state_by_chunks(const StateChunks& made, int b, int h, int n, int row0) {
  if (n < STATE_CHUNKS_FROM) return false;
  const int* flags = made.flags + static_cast<int64_t>(h) * made.places + first_chunk(row0, b);
  int bad = 0;
  for (int i = threadIdx.x; i < (n + STATE_CHUNK - 1) / STATE_CHUNK; i += blockDim.x) bad |= flags[i];
  return !__syncthreads_or(bad);
}

// tokens of a chunk in LDS; one-wave workgroups serve steps of few rows
constexpr int scan_tokens(int R, int NW) { return NW == 1 ? (R <= 4 ? 4 : 2) : R <= 4 ? 32 : R <= 8 ? 16 : 8; }
template <int R, int NW, int CH> struct ScanShape {
  static constexpr int ROW = 3 * 16 * R + 4 * NW, FLOATS = 2 * CH * ROW + 2 * CH;
};

// NW waves per workgroup = 4 NW columns of one (sequence, head).  The operands of CH tokens (q | k | decay padded to 16 R channels, the
// workgroup's value columns; the betas beside them) are staged in LDS, shared by the waves, two buffers: the next chunk is fetched into registers
// before the current one is computed and parked in the other buffer afterwards, one barrier per chunk.  Lane ks of a 16-lane row owns the key
// channels 4 ks .. 4 ks + 3, and those 64, 128, ... further on (R a multiple of 4; heads of up to 16, 32 or 96 channels: 1, 2 or 2 neighbours): LDS reads,
// and the state's loads and stores, are 16-byte accesses that are contiguous over the row.  Bound by issue slots (a long prompt leaves one or two waves a SIMD, each token costs a wave 4 R multiply-adds and what
// feeds them), so operands are read four at a time: V = 4 floats per staging access where sizes, strides and addresses allow, else 1.
// (4-byte accesses and operands read where they are used -> now, us: rows of 1501 + 700 + 65 tokens, 8 heads of 128 x 256 393 -> 253, delta rule over 32
// of 128 x 128 507 -> 351; 32 prompts of 8 to 163 tokens 273 -> 144; one token of 32 sequences, 67 MB of state 30.1 -> 15.1.)
// Heads of few channels have forms of their own, which stage and multiply no more than there is (16 heads, 32 prompts of 40 tokens, every lane four
// channels | this: 16 x 64 25.3 | 15.6, 32 x 128 45.3 | 29.5, 16 x 50 element by element 44.4 | 17.7); 48 channels are the four-channel form's (R = 3 at
// one channel a lane 51.6, 28.4 here), 66 to 96 only where sizes are not in groups of four (94 x 64 59.4 | 43.1; 96 x 96 in groups of four 50).
template <int R, bool DELTA, int NW, int V, int CH = scan_tokens(R, NW)>
__device__ __forceinline__ void scan_columns(const StateArgs& a, int b, int h, int col0, float* lds) {
  typedef ScanShape<R, NW, CH> Shape;
  constexpr int C = R % 4 == 0 ? 4 : R % 2 == 0 ? 2 : 1;                 // neighbouring channels of a lane
  constexpr int DKP = 16 * R, NCOL = 4 * NW, ROW = Shape::ROW, NTH = 64 * NW, Q = R / C;
  constexpr int SLOTS = CH * ROW / V, PF = (SLOTS + NTH - 1) / NTH;
  float* betas = lds + 2 * CH * ROW;
  const int64_t r_stride = a.r_stride;
  const int H = a.H, G = a.G, dk = a.dk, dv = a.dv;
  const int slot = a.seq[4 * b], pos0 = a.seq[4 * b + 1], n = a.seq[4 * b + 2], row0 = a.seq[4 * b + 3];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, ks = lane & 15;
  const int lcol = wave * 4 + (lane >> 4), col = col0 + lcol;
  const bool col_ok = col < dv;
  const int colc = col_ok ? col : dv - 1;
  const int nq = G * dk, nv = H * dv;
  const int g = h / (H / G);
  float* sp = a.state + ((static_cast<int64_t>(slot) * H + h) * dv + colc) * dk;     // (channels past the last one hold zeros)
  // every load below is issued unconditionally from an address inside the buffers (what it must not deliver is replaced afterwards):
  // loads under a branch wait for one another, and a chunk's fetch then costs the sum of their latencies
  float S[R];
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    const int c = C * ks + 16 * C * i;
    if constexpr (V == 4 && C == 4) {
      Lanes<float, 4>::load(sp + min(c, dk - 4), S + 4 * i);
    } else {
#pragma unroll
      for (int j = 0; j < C; ++j) S[C * i + j] = sp[min(c + j, dk - 1)];
    }
#pragma unroll
    for (int j = 0; j < C; ++j) S[C * i + j] = (pos0 > 0 && c + j < dk) ? S[C * i + j] : 0.f;
  }
  const float* base = a.r + static_cast<int64_t>(row0) * r_stride;
  const int oq = g * dk, ok = nq + g * dk, ov = 2 * nq + h * dv, og = 2 * nq + nv + h * dk, ob = 2 * nq + nv + H * dk + h;
  float pf[PF][V], pb = 0.f;
  int offs[PF], tts[PF];                    // where slot i of this thread's share of a chunk comes from: token of the chunk, offset in its row
  unsigned loaded = 0, decays = 0;          // bit i: pf[i] is an operand (else the slot's neutral value: 1 for a decay, 0 elsewhere)
  static_assert(PF <= 32, "a bit per slot");
#pragma unroll
  for (int i = 0; i < PF; ++i) {
    const int idx = min(static_cast<int>(threadIdx.x) + i * NTH, SLOTS - 1);
    const int tt = idx / (ROW / V), j = (idx - tt * (ROW / V)) * V;
    const int seg = j < DKP ? 0 : (j < 2 * DKP ? 1 : (j < 3 * DKP ? 2 : 3));
    const int jj = j - seg * DKP;                                     // segment 3: the value columns
    const int first = seg == 0 ? oq : (seg == 1 ? ok : (seg == 2 ? og : ov + col0));
    const bool valid = jj < (seg < 3 ? dk : min(dv - col0, NCOL));
    offs[i] = valid ? first + jj : oq;
    tts[i] = tt;
    loaded |= static_cast<unsigned>(valid) << i;
    decays |= static_cast<unsigned>(seg == 2) << i;
  }
  auto fetch = [&](int t0) {
    const float* cb = base + static_cast<int64_t>(t0) * r_stride;
    const int last = min(CH, n - t0) - 1;   // the sequence's last chunk: rows past its end are read as its last row (and never used)
#pragma unroll
    for (int i = 0; i < PF; ++i) Lanes<float, V>::load(cb + static_cast<int64_t>(min(tts[i], last)) * r_stride + offs[i], pf[i]);
    if (DELTA) pb = cb[static_cast<int64_t>(min(static_cast<int>(threadIdx.x), last)) * r_stride + ob];
  };
  auto park = [&](int which) {
#pragma unroll
    for (int i = 0; i < PF; ++i) {
      const int idx = threadIdx.x + i * NTH;
      const float neutral = (decays >> i) & 1u ? 1.f : 0.f;
#pragma unroll
      for (int j = 0; j < V; ++j) pf[i][j] = ((loaded >> i) & 1u) ? pf[i][j] : neutral;
      if (idx < SLOTS) Lanes<float, V>::store(lds + which * CH * ROW + idx * V, pf[i]);
    }
    if (DELTA && static_cast<int>(threadIdx.x) < CH) betas[which * CH + threadIdx.x] = pb;
  };
  fetch(0);
  park(0);
  __syncthreads();
  float* op = a.out + static_cast<int64_t>(row0) * nv + h * dv + colc;
  int which = 0;
  for (int t0 = 0; t0 < n; t0 += CH, which ^= 1) {
    const bool more = t0 + CH < n;
    if (more) fetch(t0 + CH);
    const float* cur = lds + which * CH * ROW;
    const int cn = min(CH, n - t0);
    struct Token { float q[R], k[R], d[R], v, beta; };
    auto read = [&](int tt, Token& x) {
      const float* at = cur + tt * ROW + C * ks;
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        Lanes<float, C>::load(at + 16 * C * i, x.q + C * i);
        Lanes<float, C>::load(at + DKP + 16 * C * i, x.k + C * i);
        Lanes<float, C>::load(at + 2 * DKP + 16 * C * i, x.d + C * i);
      }
      x.v = cur[tt * ROW + 3 * DKP + lcol];
      if (DELTA) x.beta = betas[which * CH + tt];
    };
    auto step = [&](int tt, const Token& x) {
#pragma unroll
      for (int i = 0; i < R; ++i) S[i] *= x.d[i];
      float u = x.v;
      if constexpr (DELTA) {
        float dot[2] = {0.f, 0.f};
#pragma unroll
        for (int i = 0; i < R; ++i) dot[i & 1] += x.k[i] * S[i];
        u = x.beta * (u - row16_sum(dot[0] + dot[1]));
      }
      float o[2] = {0.f, 0.f};
#pragma unroll
      for (int i = 0; i < R; ++i) { S[i] += x.k[i] * u; o[i & 1] += x.q[i] * S[i]; }
      const float sum = row16_sum(o[0] + o[1]);
      if (ks == 0 && col_ok) op[static_cast<int64_t>(t0 + tt) * nv] = sum;
    };
    Token x;
    if constexpr (NW > 1) {                  // a token's operands are read while the one before it is computed
      Token y;
      read(0, x);
      int tt = 0;
      for (; tt + 1 < cn; tt += 2) {
        read(tt + 1, y);
        step(tt, x);
        read(min(tt + 2, cn - 1), x);
        step(tt + 1, y);
      }
      if (tt < cn) step(tt, x);
    } else {                                 // few tokens, many sequences: the registers serve occupancy
      for (int tt = 0; tt < cn; ++tt) {
        read(tt, x);
        step(tt, x);
      }
    }
    if (more) park(which ^ 1);
    __syncthreads();
  }
  if (col_ok) {
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const int c = C * ks + 16 * C * i;
      if constexpr (V == 4 && C == 4) {
        if (c < dk) Lanes<float, 4>::store(sp + c, S + 4 * i);
      } else {
#pragma unroll
        for (int j = 0; j < C; ++j)
          if (c + j < dk) sp[c + j] = S[C * i + j];
      }
    }
  }
}

}  // namespace gbxm
