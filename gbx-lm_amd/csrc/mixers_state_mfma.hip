// The decayed matrix states of mixers_state.hip for prompt portions: 16 tokens at a time on the matrix cores, in fp32 (products of decays in fp64).
//
// With P_i = d_1 .. d_i the decays of a chunk up to token i (per key channel) and S the state before it,
//   A[i][j] = sum_c k_i k_j d_{j+1} .. d_i  (j < i),   B[i][j] = sum_c q_i k_j d_{j+1} .. d_i  (j <= i),   M = (1 + diag(beta) A)^-1 diag(beta)
//   U = M (V - (K P) S)      (without the delta rule U = V)
//   O = (Q P) S + B U,       S <- P_16 S + sum_j (k_j d_{j+1} .. d_16) u_j
// -- every factor is a product of decays forward in time, so none of them grows, whatever the decays.
//
//   state_pairs_kernel   A, B and M of every (chunk, head): they do not depend on the state, so all chunks run at once.
//   state_chunk_kernel   the chain over the chunks.  A workgroup holds 16 columns of a head's state: four waves multiply, a quarter of the key channels each, the
//                        state in accumulators of v_mfma_f32_16x16x4_f32; their layout (channel 4 (lane / 16) + i, column lane % 16) is also that of a right
//                        operand whose contraction index runs 4 (lane / 16) + i at step i, so the state, U and V never change place.  The waves' parts of the
//                        two products with S meet in LDS.  Four more waves carry: they fetch the rows two chunks ahead, multiply the decays in and write O.
//
// Token by token a wave of four columns spends 8 instructions a channel and waits for two sums over lanes a token (590 cycles a token and more).  A chunk here is
// 2 600 cycles, of which the matrix cores are busy 930: it is a chain of waits (LDS, two barriers, dependent products), not bound by a unit.  Tried: carrying and
// multiplying in the same four waves (3 080 cycles), loads four chunks ahead (no change), pairs of channels a lane (8 % slower).  Shorter sequences of the step go token by
// token in the same launch (TOGETHER), in chunks of few tokens, which keep the kernel's registers at two workgroups a CU (16 tokens: 8 registers spilled).
// Measured, all kernels of a call, token by token | chunks, us: 1 501 + 700 + 65 rows, delta rule, 32 heads of 128 x 128 325 | 182, 8 of 128 x 256 without it 243 | 99;
// 130 + 100 + 64 + 17 + 8 rows, delta rule, 32 heads 52 | 54, 16 heads 40 | 39; 32 sequences of 8 .. 163 rows 305 | 300 and 176 | 178, 8 heads of 128 x 256 without it 141 | 134;
// one sequence of 128 | 200 rows, 32 heads 34 | 23 and 50 | 32.  The first kernel's 6 us are lost where a sequence that just goes by chunks meets one that just does not: 127 + 128
// rows, 16 heads 34 | 42.  Error against 64 bits, relative, 1e-8, over rows that models prepare:
// delta rule 19.4 | 16.2, without it 42.8 | 38.0 (decays 0.92 .. 0.9998 a token and channel), 8.1 | 7.7 (one decay a head).
#include <type_traits>
#include "mixers_mfma.h"
#include "mixers_state_scan.h"

namespace gbxm {
namespace {

constexpr int CT = STATE_CHUNK;
constexpr int PAIR = 2 * CT * CT;            // numbers per (chunk, head): M, B
// 2^40: what the first kernel lets pass; it only looks at its own operands, and a chain whose sums leave the range all the same is seen at its end
constexpr float STATE_MOST = 1099511627776.f;

__device__ __forceinline__ f32x4v mfma_f32(float a, float b, const f32x4v& c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// Rows of fp32 numbers from `p` on, `bytes` long: what lies beyond reads as zero and is not written
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_of(const float* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0, bytes, 0x00020000);
}
__device__ __forceinline__ float load1(__amdgpu_buffer_rsrc_t r, int at) { return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, at, 0, 0)); }
__device__ __forceinline__ f32x4v load4(__amdgpu_buffer_rsrc_t r, int at) { return __builtin_bit_cast(f32x4v, __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, 0)); }
__device__ __forceinline__ void store1(__amdgpu_buffer_rsrc_t r, int at, float x) { __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, x), r, at, 0, 0); }
__device__ __forceinline__ constexpr unsigned bits(float x) { return __builtin_bit_cast(unsigned, x) & 0x7FFFFFFFu; }
constexpr int PAST = 0x7FFFFFF0;             // an offset beyond every buffer

// grid (chunk places, heads): wave w takes the tokens j = 4 w .. 4 w + 3, a 16-lane row each; lane ks of it the channels 4 ks .. 4 ks + 3 and those 64 further on.
template <int TPW, bool DELTA>
__global__ __launch_bounds__(256) void state_pairs_kernel(const float* __restrict__ r, int64_t r_stride, float* __restrict__ pairs, int* __restrict__ flags,
                                                         const int* __restrict__ seq, int B_, int H, int G, int dk, int dv) {
  constexpr int CP = 64 * TPW;
  __shared__ __attribute__((aligned(16))) float qs[CT][CP], ks_[CT][CP], ds[CT][CP];
  __shared__ __attribute__((aligned(16))) float am[CT][CT], bm[CT][CT];
  __shared__ float betas[CT];
  const int place = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  int lo = 0, hi = B_ - 1;                                              // the last sequence whose first place is not behind this one
  while (lo < hi) {
    const int mid = (lo + hi + 1) / 2;
    if (first_chunk(seq[4 * mid + 3], mid) <= place) lo = mid; else hi = mid - 1;
  }
  const int n = seq[4 * lo + 2], row0 = seq[4 * lo + 3], t0 = (place - first_chunk(row0, lo)) * CT;
  if (n < STATE_CHUNKS_FROM || t0 >= n || t0 < 0) return;
  const int g = h / (H / G), nq = G * dk, nv = H * dv;
  const float* base = r + static_cast<int64_t>(row0 + t0) * r_stride;
  const int cn = min(CT, n - t0), rs = static_cast<int>(r_stride) * 4;
  // (rows past the end lie past the buffer's end and read as zeros; a decay of zero there meets keys and queries of zero)
  const __amdgpu_buffer_rsrc_t rq = rows_of(base + g * dk, cn * rs), rk = rows_of(base + nq + g * dk, cn * rs), rd = rows_of(base + 2 * nq + nv + h * dk, cn * rs);
  unsigned most = 0, decays = 0;            // largest magnitudes, as bits: infinities and NaN above all numbers
#pragma unroll
  for (int m = 0; m < CT * TPW * 16 / 256; ++m) {
    const int i = tid + 256 * m, t = i / (CP / 4), c = i % (CP / 4) * 4, at = c < dk ? t * rs + c * 4 : PAST;
    const f32x4v q = load4(rq, at), k = load4(rk, at), d = load4(rd, at);
    *reinterpret_cast<f32x4v*>(&qs[t][c]) = q;
    *reinterpret_cast<f32x4v*>(&ks_[t][c]) = k;
    *reinterpret_cast<f32x4v*>(&ds[t][c]) = d;
#pragma unroll
    for (int e = 0; e < 4; ++e) { most = max(most, max(bits(q[e]), bits(k[e]))); decays = max(decays, bits(d[e])); }
  }
  for (int t = tid >> 6; t < cn; t += 4)
    for (int c = tid & 63; c < dv; c += 64) most = max(most, bits(base[static_cast<int64_t>(t) * r_stride + 2 * nq + h * dv + c]));
  if (DELTA && tid < CT) {
    const float b = base[static_cast<int64_t>(min(tid, cn - 1)) * r_stride + 2 * nq + nv + H * dk + h];
    betas[tid] = tid < cn ? b : 0.f;
    most = max(most, bits(b));
  }
  bool bad = most > bits(STATE_MOST) || decays > bits(1.f);
  am[tid >> 4][tid & 15] = bm[tid >> 4][tid & 15] = 0.f;
  __syncthreads();
  const int lane = tid & 63, ks = lane & 15, first = 4 * (tid >> 6), j = first + (lane >> 4);
  float w[4 * TPW];
#pragma unroll
  for (int t = 0; t < TPW; ++t) Lanes<float, 4>::load(&ks_[j][4 * ks + 64 * t], w + 4 * t);
  auto row = [&](int i, auto own) {                                     // own: the rows among this wave's tokens
    float a = 0.f, b = 0.f;
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      float d[4], k[4], q[4];
      Lanes<float, 4>::load(&ds[i][4 * ks + 64 * t], d);
      Lanes<float, 4>::load(&qs[i][4 * ks + 64 * t], q);
      if (DELTA) Lanes<float, 4>::load(&ks_[i][4 * ks + 64 * t], k);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if constexpr (decltype(own)::value) d[c] = i > j ? d[c] : 1.f;
        w[4 * t + c] *= d[c];
        b += q[c] * w[4 * t + c];
        if (DELTA) a += k[c] * w[4 * t + c];
      }
    }
    b = row16_sum(b);
    if (DELTA) a = row16_sum(a);
    if (ks == 0 && i >= j) bm[i][j] = b;
    if (DELTA && ks == 0 && i > j) am[i][j] = a;
  };
#pragma unroll
  for (int i = 0; i < 4; ++i) row(first + i, std::true_type{});
#pragma unroll 2
  for (int i = first + 4; i < CT; ++i) row(i, std::false_type{});
  __syncthreads();
  float* to = pairs + (static_cast<int64_t>(place) * H + h) * PAIR;
  if (DELTA && tid < CT) {                                              // lane c: column c of M, from the first row down
    float x[CT];
#pragma unroll
    for (int i = 0; i < CT; ++i) {
      float s = i == tid ? 1.f : 0.f;
#pragma unroll
      for (int m = 0; m < i; ++m) s -= am[i][m] * x[m];
      x[i] = betas[i] * s;
      bad |= !(fabsf(x[i]) <= STATE_MOST);
      to[i * CT + tid] = x[i];
    }
  }
  to[CT * CT + tid] = bm[tid >> 4][tid & 15];
  const int any = __syncthreads_or(bad);
  if (tid == 0) flags[static_cast<int64_t>(h) * gridDim.x + place] = any;
}

// A chunk's operands in LDS: Q P and K P by token, K D by channel, P_16
template <int TPW, bool DELTA> struct ChunkLds {
  static constexpr int CP = 64 * TPW, LD = CP + 4, LT = CT + 4;
  static constexpr int Q = 0, K = Q + CT * LD, KT = K + (DELTA ? CT * LD : 0), P = KT + CP * LT, SIZE = P + CP;
  static constexpr int OUT = 2 * SIZE, RED = OUT + 2 * 4 * 256, END = RED + (DELTA ? 4 * 256 : 0);   // the waves' parts of O (twice) and of (K P) S
  static constexpr int TOKENS = TPW == 1 ? 16 : 8;                      // of a chunk of the sequences that go token by token: few, so that registers and LDS stay the chunks'
  static constexpr int SCAN = ScanShape<4 * TPW, 4, TOKENS>::FLOATS, BYTES = (END > SCAN ? END : SCAN) * 4;
};

// Loads that fly across a barrier: only LDS has to be settled
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int TPW, bool DELTA>
__global__ __launch_bounds__(512, (TPW <= 2 ? 4 : 2)) void state_chunk_kernel(const StateArgs a, const float* __restrict__ pairs, const StateChunks made, int together) {
  typedef ChunkLds<TPW, DELTA> L;
  constexpr int CP = L::CP, LD = L::LD, LT = L::LT, CI = (CP + 127) / 128;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int64_t r_stride = a.r_stride;
  const int H = a.H, G = a.G, dk = a.dk, dv = a.dv;
  const int* seq = a.seq;
  // the column blocks of one (sequence, head) read the same operands: neighbours on one XCD
  const int cols = (dv + 15) / 16, unit = blockIdx.x >> 3, which = unit / cols * 8 + (blockIdx.x & 7);
  if (which >= a.B * H) return;
  const int b = which / H, h = which % H;
  const int slot = seq[4 * b], pos0 = seq[4 * b + 1], n = seq[4 * b + 2], row0 = seq[4 * b + 3];
  const int tid = threadIdx.x, lane = tid & 63, part = __builtin_amdgcn_readfirstlane(tid >> 6), wave = part & 3, fr = lane & 15, g4 = 4 * (lane >> 4);
  const int place0 = first_chunk(row0, b), chunks = (n + CT - 1) / CT;
  if (!state_by_chunks(made, b, h, n, row0)) {                          // token by token: half of the waves
    if (together && tid < 256) scan_columns<4 * TPW, DELTA, 4, 4, L::TOKENS>(a, b, h, unit % cols * 16, lds);
    return;
  }
  const int col = unit % cols * 16 + fr, colc = min(col, dv - 1);
  const int g = h / (H / G), nq = G * dk, nv = H * dv;
  const float* base = a.r + static_cast<int64_t>(row0) * r_stride;
  // a wave takes 32 channels (of every 128), its halves eight tokens each; what the other half's decays multiply to comes across the wave
  const int late = lane >> 5, ch = 32 * wave + (lane & 31), rs = static_cast<int>(r_stride) * 4;
  const float *bq = base + g * dk, *bk = bq + nq, *bd = base + 2 * nq + nv + h * dk, *bv = base + 2 * nq + h * dv;
  struct Raw { float q[CI][CT / 2], k[CI][CT / 2], d[CI][CT / 2]; } even, odd;   // two chunks fly: a trip to memory is longer than a chunk's work
  int at[CI][CT / 2];
#pragma unroll
  for (int m = 0; m < CI; ++m)
#pragma unroll
    for (int t = 0; t < CT / 2; ++t) at[m][t] = ch + 128 * m < dk ? (t + late * (CT / 2)) * rs + (ch + 128 * m) * 4 : PAST;
  auto tokens = [&](int c) { return __builtin_amdgcn_readfirstlane(max(min(CT, n - c * CT), 0)); };
  auto fetch = [&](int c, Raw& f) {                                     // (tokens past the end and channels past the last read as zeros)
    const int64_t skip = static_cast<int64_t>(c) * CT * r_stride;
    const int bytes = tokens(c) * rs;
    const __amdgpu_buffer_rsrc_t rq = rows_of(bq + skip, bytes), rk = rows_of(bk + skip, bytes), rd = rows_of(bd + skip, bytes);
#pragma unroll
    for (int m = 0; m < CI; ++m) {
      if (CP - 128 * m < 128 && 32 * wave + 128 * m >= CP) break;
#pragma unroll
      for (int t = 0; t < CT / 2; ++t) {
        f.d[m][t] = load1(rd, at[m][t]);
        f.q[m][t] = load1(rq, at[m][t]);
        f.k[m][t] = load1(rk, at[m][t]);
      }
    }
  };
  auto park = [&](int c, Raw& f, float* to) {
    const int cn = n - c * CT - late * (CT / 2);
    if (n - c * CT < CT) {                                              // a token past the end decays nothing
#pragma unroll
      for (int m = 0; m < CI; ++m)
#pragma unroll
        for (int t = 0; t < CT / 2; ++t) f.d[m][t] = t < cn ? f.d[m][t] : 1.f;
    }
#pragma unroll
    for (int m = 0; m < CI; ++m) {
      const int cc = ch + 128 * m;
      if (CP - 128 * m < 128 && 32 * wave + 128 * m >= CP) break;
      // Products in 64 bits (as fast here): a head whose decays are all one number would round them all to one side, chunk after chunk
      double d[CT / 2], p[CT / 2], s[CT / 2];
      float k[CT / 2];
#pragma unroll
      for (int t = 0; t < CT / 2; ++t) d[t] = f.d[m][t];
      p[0] = d[0];
#pragma unroll
      for (int t = 1; t < CT / 2; ++t) p[t] = p[t - 1] * d[t];
      s[CT / 2 - 1] = 1.;
#pragma unroll
      for (int t = CT / 2 - 2; t >= 0; --t) s[t] = s[t + 1] * d[t + 1];
      const double whole = p[CT / 2 - 1], other = __shfl_xor(whole, 32, 64), before = late ? other : 1., behind = late ? 1. : other;
      float* rows = to + late * (CT / 2) * LD + cc;
#pragma unroll
      for (int t = 0; t < CT / 2; ++t) {
        const float x = static_cast<float>(p[t] * before);
        rows[L::Q + t * LD] = f.q[m][t] * x;
        if constexpr (DELTA) rows[L::K + t * LD] = f.k[m][t] * x;
        k[t] = f.k[m][t] * static_cast<float>(s[t] * behind);
      }
      float* kt = to + L::KT + cc * LT + late * (CT / 2);
      *reinterpret_cast<f32x4v*>(kt) = f32x4v{k[0], k[1], k[2], k[3]};
      *reinterpret_cast<f32x4v*>(kt + 4) = f32x4v{k[4], k[5], k[6], k[7]};
      to[L::P + cc] = static_cast<float>(whole * other);                                    // (both halves write the same bits)
    }
  };
  float* sp = a.state + ((static_cast<int64_t>(slot) * H + h) * dv + colc) * dk;
  f32x4v S[TPW];
  bool wild = false;                                                    // an infinity or NaN came up ...
  __shared__ int any_wild;                                              // ... in some thread
  if (tid == 0) any_wild = 0;
  if (part >= 4) {                                                      // four waves carry: operands in, read-outs out
    // O of a chunk is summed and written during the next one, a number per thread
    const int ocol = unit % cols * 16 + (tid >> 2 & 15), ato = ocol < dv ? ((4 * wave + (tid & 3)) * nv + ocol) * 4 : PAST;
    auto put = [&](int c) {
      const float* o = lds + L::OUT + (c & 1) * (4 * 256) + (tid & 255);
      const float x = (o[0] + o[256]) + (o[512] + o[768]);
      wild |= !(fabsf(x) < INFINITY);
      store1(rows_of(a.out + static_cast<int64_t>(row0 + c * CT) * nv + h * dv, tokens(c) * nv * 4), ato, x);
    };
    auto carry = [&](int c, Raw& f) {                                   // `f` holds chunk c + 1, whose buffer nobody reads since the last barrier
      if (c > 0) put(c - 1);
      if constexpr (DELTA) lds_barrier();
      park(c + 1, f, lds + ((c + 1) & 1) * L::SIZE);
      fetch(c + 3, f);
      lds_barrier();
    };
    fetch(0, even);
    fetch(1, odd);
    park(0, even, lds);
    fetch(2, even);
    lds_barrier();
    for (int c = 0; c < chunks; c += 2) {                               // (a chunk behind the last one has no tokens: it changes and writes nothing)
      carry(c, odd);
      carry(c + 1, even);
    }
    put((chunks - 1) | 1);
  } else {                                                              // and four multiply
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      const int c = 16 * (wave * TPW + t) + g4;
      const f32x4v v = *reinterpret_cast<const f32x4v*>(sp + min(c, dk - 4));
      S[t] = pos0 > 0 && c < dk ? v : f32x4v{0};
    }
    // M and B of a chunk by lanes as left operands (row lane % 16, contraction index 4 (lane / 16) + i), V as the accumulators lie
    struct Small { f32x4v m, v; float b; } now, then;
    const float* pairs0 = pairs + (static_cast<int64_t>(place0) * H + h) * PAIR;
    const int atm = (fr * CT + g4) * 4;
    int atv[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      atv[i] = (g4 + i) * rs + colc * 4;
    }
    auto fetch_small = [&](int c, Small& s) {
      const __amdgpu_buffer_rsrc_t rp = rows_of(pairs0 + static_cast<int64_t>(c) * H * PAIR, PAIR * 4);
      if constexpr (DELTA) s.m = load4(rp, atm);
      s.b = load1(rp, atm + CT * CT * 4 + wave * 4);                      // B U is shared out by steps of the contraction
      const __amdgpu_buffer_rsrc_t rv = rows_of(bv + static_cast<int64_t>(c) * CT * r_stride, min(CT, n - c * CT) * rs);
#pragma unroll
      for (int i = 0; i < 4; ++i) s.v[i] = load1(rv, atv[i]);
    };
    auto chunk = [&](int c, const Small& now, Small& next) {              // (products are interleaved so that neighbours do not wait for one another)
      const float* cur = lds + (c & 1) * L::SIZE;
      f32x4v u = now.v, y = now.v, o[TPW], z[TPW], q[TPW], k[TPW], p[TPW];
      f32x4v* red = reinterpret_cast<f32x4v*>(lds + L::RED);
      fetch_small(min(c + 1, chunks - 1), next);
      const int rows = fr * LD + 16 * wave * TPW + g4;
#pragma unroll
      for (int t = 0; t < TPW; ++t) {
        if constexpr (DELTA) k[t] = *reinterpret_cast<const f32x4v*>(cur + L::K + rows + 16 * t);
        q[t] = *reinterpret_cast<const f32x4v*>(cur + L::Q + rows + 16 * t);
        o[t] = z[t] = f32x4v{0};
      }
      if constexpr (DELTA) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int t = 0; t < TPW; ++t) z[t] = mfma_f32(k[t][i], S[t][i], z[t]);
#pragma unroll
        for (int t = 1; t < TPW; ++t) z[0] += z[t];
        red[wave * 64 + lane] = z[0];
        lds_barrier();
        y -= (red[lane] + red[64 + lane]) + (red[128 + lane] + red[192 + lane]);
        u = f32x4v{0};
      }
#pragma unroll
      for (int t = 0; t < TPW; ++t) {
        k[t] = *reinterpret_cast<const f32x4v*>(cur + L::KT + (16 * (wave * TPW + t) + fr) * LT + g4);
        p[t] = *reinterpret_cast<const f32x4v*>(cur + L::P + 16 * (wave * TPW + t) + g4);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int t = 0; t < TPW; ++t) o[t] = mfma_f32(q[t][i], S[t][i], o[t]);
        if constexpr (DELTA) u = mfma_f32(now.m[i], y[i], u);
      }
#pragma unroll
      for (int t = 0; t < TPW; ++t) S[t] *= p[t];
      o[0] = mfma_f32(now.b, wave == 0 ? u[0] : wave == 1 ? u[1] : wave == 2 ? u[2] : u[3], o[0]);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < TPW; ++t) S[t] = mfma_f32(k[t][i], u[i], S[t]);
#pragma unroll
      for (int t = 1; t < TPW; ++t) o[0] += o[t];
      *reinterpret_cast<f32x4v*>(lds + L::OUT + (c & 1) * (4 * 256) + wave * 256 + lane * 4) = o[0];
      lds_barrier();
    };
    fetch_small(0, now);
    lds_barrier();
    for (int c = 0; c < chunks; c += 2) {
      chunk(c, now, then);
      chunk(c + 1, then, now);
    }
#pragma unroll
    for (int t = 0; t < TPW; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) wild |= !(fabsf(S[t][i]) < INFINITY);
  }
  // What an infinity of the carried state, or sums that left the range, make of a chunk's other tokens (zeros of the factors between them times
  // infinity) is not what they make token by token: such columns start again, from the state as it was.
  if (wild) any_wild = 1;
  lds_barrier();
  if (any_wild) {
    __threadfence();                                                    // this wave's results are behind those that come
    __syncthreads();
    if (tid < 256) scan_columns<4 * TPW, DELTA, 4, 4, L::TOKENS>(a, b, h, unit % cols * 16, lds);
    return;
  }
  if (part >= 4 || col >= dv) return;
#pragma unroll
  for (int t = 0; t < TPW; ++t) {
    const int c = 16 * (wave * TPW + t) + g4;
    if (c < dk) *reinterpret_cast<f32x4v*>(sp + c) = S[t];
  }
}

int64_t chunk_places(int64_t T, int64_t B) { return T / CT + B; }
size_t flag_bytes(int64_t places, int H) { return (static_cast<size_t>(places) * H * sizeof(int) + 15) & ~static_cast<size_t>(15); }
int64_t chunk_units(const StateArgs& a) { return (static_cast<int64_t>(a.B) * a.H + 7) / 8 * 8 * ((a.dv + 15) / 16); }
// Column blocks of a step up to which the chunks' launch also takes what goes token by token: the two need not wait for one another, but such a workgroup works
// with half of its waves, two a CU.  Above, the chip is full many times over either way, and the token kernel's own launch has three workgroups a CU.  One launch |
// two, us: delta rule, heads of 128 x 128, 16 heads 130 + 100 + 64 + 17 + 8 rows 39 | 57, 16 sequences (2 048 blocks) 99 | 99, 24 136 | 132, 32 heads, 16 sequences 171 | 161,
// 32 328 | 299; without it, 32 sequences (4 096 blocks) of 16 heads 135 | 143, of 8 heads of 128 x 256 134 | 135.
constexpr int64_t TOGETHER_DELTA = 2048, TOGETHER = 4096;

template <int TPW, bool DELTA>
int launch(const StateArgs& a, const StateChunks& made, int* flags, float* pairs, bool together, hipStream_t s) {
  constexpr int BYTES = ChunkLds<TPW, DELTA>::BYTES;
  static OncePerDevice once;
  if (once.pending()) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(state_chunk_kernel<TPW, DELTA>), hipFuncAttributeMaxDynamicSharedMemorySize, BYTES);
    if (e != hipSuccess) return hip_fail(e, "state_scan");
    once.done();
  }
  state_pairs_kernel<TPW, DELTA><<<dim3(made.places, a.H), 256, 0, s>>>(a.r, a.r_stride, pairs, flags, a.seq, a.B, a.H, a.G, a.dk, a.dv);
  state_chunk_kernel<TPW, DELTA><<<static_cast<unsigned>(chunk_units(a)), 512, BYTES, s>>>(a, pairs, made, together);
  return after_launch("state_scan (chunks)");
}

}  // namespace

size_t state_chunks_workspace(int64_t T, int64_t B, int H, int dk, int dv) {
  const int64_t places = chunk_places(T, B);
  if (dk % 4 || dk < 64 || dk > 256 || dv < 16 || dv % 4 || H > 65535 || B < 1 || places > (1 << 24) || B * H * ((dv + 15) / 16) > (1 << 26)) return 0;
  return flag_bytes(places, H) + static_cast<size_t>(places) * H * PAIR * sizeof(float);
}

int launch_state_chunks(const StateArgs& a, int64_t T, bool delta, void* ws, hipStream_t s, StateChunks* left) {
  int* flags = static_cast<int*>(ws);
  const StateChunks made{flags, static_cast<int>(chunk_places(T, a.B))};
  float* pairs = reinterpret_cast<float*>(static_cast<unsigned char*>(ws) + flag_bytes(made.places, a.H));
  const bool together = chunk_units(a) <= (delta ? TOGETHER_DELTA : TOGETHER);
  *left = together ? StateChunks{nullptr, 0} : made;
#define GBXM_CHUNKS(N) (delta ? launch<N, true>(a, made, flags, pairs, together, s) : launch<N, false>(a, made, flags, pairs, together, s))
  switch ((a.dk + 63) / 64) {
    case 1: return GBXM_CHUNKS(1);
    case 2: return GBXM_CHUNKS(2);
    case 3: return GBXM_CHUNKS(3);
    default: return GBXM_CHUNKS(4);
  }
#undef GBXM_CHUNKS
}

}  // namespace gbxm
