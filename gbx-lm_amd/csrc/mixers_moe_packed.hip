// Routed experts over GBA-packed weights for steps with many (row, choice) pairs: y[pair] = x[pair / x_div] . (s q + z)_e^T, e = idx[pair], fields of
// 2, 3 or 4 bits in groups of 32, 64 or 128 -- or two such matrices and silu(gate) * up of their results (the three roundings of the
// separate operations).  Prompts and batched decoding of quantised models with routed experts.
//
// The pairs are bucketed by expert on the device (expert_buckets); a workgroup takes one tile of up to 64 pairs of one expert and 256 weight rows
// (gated: 128 rows of each matrix), a wave 64 of them.  Weights are never expanded: a field ORed under the exponent of 128.0 (bf16) or
// 1024.0 (fp16) IS the number C + q, a shift and an and-or make two operands of a product, and the affine map meets the fp32 sums of a group:
//   acc[m, n] += s[n, g] t[m, n] + (z[n, g] - C s[n, g]) xsum[m, g],   t = sum_k x (C + q),   xsum = sum_k x.
// No weight is rounded to the activation type, so the error is that of the fp32 sums and of the one rounding of the result.  Infinite activations, for
// which this form has infinity minus infinity, are seen in the sums, and their outputs taken again weight by weight (expanded_dot).
// The contraction runs in chunks of 128.  Inside a chunk the order of k is free as long as both operands agree: step t of lane quarter f
// multiplies octet o(t, f) of the row -- the one that lets a lane read its packed words of a group in one piece -- and the activations are
// stored in that order, in the pair order in which fields leave a word ((j, j + 8) of 16 fields of 2 bits, (j, j + 4) of 8 of 4 bits).
// What bounds it: with tens of pairs per expert the packed weights are read once (227 MB at 128 experts of 3 x 2048 x 768 in 3 bits, 46 us) and
// the vector instructions that build operands cost about what the products do (four tiles of 16 rows share an activation fragment, so LDS
// stays at half its rate); the tile is 64 pairs high because 16 products per built operand leave registers for one chunk of weights in flight.
// Measured (us; before: pairs grouped on the host, an expert at a time, some ten launches each):
//   3 600 pairs, 128 experts, 3 bits, group 128: 2 x 768 x 2048 gated  78 (2.0 TB/s of packed weights), 2048 x 768  43
//   32 experts of 768 x 2048, 280 | 1 800 | 8 000 pairs: 3 bits 32 | 49 | 79, 4 bits 37 | 53 | 90 -- before 2 454 | 2 455 | 2 777
// and the relative error against 64 bits at 1 800 pairs 1.66e-3 (bf16) and 2.1e-4 (fp16), before 2.16e-3 and 2.7e-4.
#include "mixers_mfma.h"
#include "packed_fields.h"

namespace gbxm {
namespace {

using gbx::Packed;

constexpr int PT = 64;                 // pairs per tile at most
constexpr int PLDS = 4 * PT * 144;     // LDS bytes: two chunks of activations (2 x 64 x 256) and xsum, then four output tiles of 64 rows x 144

struct PackedArgs {
  const unsigned short* x;
  const uint32_t* w[2];                // [E][N][K * BITS / 32]; [1]: the up matrix
  const unsigned short* s[2];
  const unsigned short* z[2];
  const unsigned short* bias;          // [E][N] or null
  const int *offsets, *sorted;
  const int4* tile_tab;
  unsigned short* y;                   // [pairs][N]
  int N, K, E, x_div, cols;
};

template <bool BF16> __device__ __forceinline__ float pair_sum(unsigned v, float acc) {
  return acc + gbx::act_lo<BF16>(v) + gbx::act_hi<BF16>(v);
}

// One tile of up to 16 NR pairs x 256 weight rows.
template <int BITS, int GRP, bool BF16, bool GATED, int NR>
__device__ __forceinline__ void packed_tile(const PackedArgs& a, unsigned char* lds, int e, int lo, int hi, int col) {
  typedef Packed<BITS, GRP, BF16> P;
  constexpr int NF = P::NF, SPG = P::SPG;
  constexpr int XI = NR < 2 ? 1 : NR / 2;                               // activation pieces (16 values) per thread and chunk
  constexpr int XBUF = NR * 16 * 256;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), fr = lane & 15, f = lane >> 4;
  const int N = a.N, K = a.K, n = K >> 7;
  const int64_t words = static_cast<int64_t>(K >> 5) * BITS, groups = K / GRP;
  float* xsum = reinterpret_cast<float*>(lds + 2 * XBUF);               // [2][NF][16 NR]
  // activations: thread t moves pieces t + 256 i; piece p is 16 values at column piece p % 8 of row p / 8
  const bool mover = NR > 1 || tid < 128;
  const unsigned short* xp[XI];
#pragma unroll
  for (int i = 0; i < XI; ++i) {
    const int row = (tid >> 3) + 32 * i;
    xp[i] = a.x + static_cast<int64_t>(a.sorted[min(lo + min(row, 16 * NR - 1), hi - 1)] / a.x_div) * K + (tid & 7) * 16;
  }
  u32x4 xs[XI][2];
  auto load_x = [&](int c) {
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      xs[i][0] = *reinterpret_cast<const u32x4*>(xp[i] + c * 128);
      xs[i][1] = *reinterpret_cast<const u32x4*>(xp[i] + c * 128 + 8);
    }
  };
  auto store_x = [&](int buf) {
    if (!mover) return;
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const int row = (tid >> 3) + 32 * i, pc = tid & 7;
      const u32x4 l = xs[i][0], h = xs[i][1];
      u32x4 u0 = l, u1 = h;
      if constexpr (BITS == 2) {                                        // units of a word: dword j = values (4 b + j, 4 b + j + 8)
        u0.x = __builtin_amdgcn_perm(h.x, l.x, 0x05040100u); u0.y = __builtin_amdgcn_perm(h.x, l.x, 0x07060302u);
        u0.z = __builtin_amdgcn_perm(h.y, l.y, 0x05040100u); u0.w = __builtin_amdgcn_perm(h.y, l.y, 0x07060302u);
        u1.x = __builtin_amdgcn_perm(h.z, l.z, 0x05040100u); u1.y = __builtin_amdgcn_perm(h.z, l.z, 0x07060302u);
        u1.z = __builtin_amdgcn_perm(h.w, l.w, 0x05040100u); u1.w = __builtin_amdgcn_perm(h.w, l.w, 0x07060302u);
      } else if constexpr (BITS == 4) {                                 // dword j = values (j, j + 4) of a word's eight
        u0.x = __builtin_amdgcn_perm(l.z, l.x, 0x05040100u); u0.y = __builtin_amdgcn_perm(l.z, l.x, 0x07060302u);
        u0.z = __builtin_amdgcn_perm(l.w, l.y, 0x05040100u); u0.w = __builtin_amdgcn_perm(l.w, l.y, 0x07060302u);
        u1.x = __builtin_amdgcn_perm(h.z, h.x, 0x05040100u); u1.y = __builtin_amdgcn_perm(h.z, h.x, 0x07060302u);
        u1.z = __builtin_amdgcn_perm(h.w, h.y, 0x05040100u); u1.w = __builtin_amdgcn_perm(h.w, h.y, 0x07060302u);
      }
      const int o = 2 * pc, p0 = 4 * P::step_of(o) + P::quarter_of(o), p1 = 4 * P::step_of(o + 1) + P::quarter_of(o + 1);
      unsigned char* dst = lds + buf * XBUF + row * 256;
      *reinterpret_cast<u32x4*>(dst + ((p0 ^ row) & 15) * 16) = u0;
      *reinterpret_cast<u32x4*>(dst + ((p1 ^ row) & 15) * 16) = u1;
      float sm = 0.f;
#pragma unroll
      for (int q = 0; q < 4; ++q) sm = pair_sum<BF16>(h[q], pair_sum<BF16>(l[q], sm));
      sm += __shfl_xor(sm, 1, 64);                                      // 32 values
      if constexpr (GRP >= 64) sm += __shfl_xor(sm, 2, 64);
      if constexpr (GRP == 128) sm += __shfl_xor(sm, 4, 64);
      if (pc % (GRP / 16) == 0) xsum[(buf * NF + pc / (GRP / 16)) * 16 * NR + row] = sm;
    }
  };
  // weights: row tile j of the wave; gated: tiles 0, 1 are gate rows and 2, 3 the up rows of the same channels
  const int c0 = GATED ? col * 128 + wave * 32 : col * 256 + wave * 64;
  // (byte offsets inside the expert's matrices, which stay under 4 GB: one register a row and array instead of two)
  unsigned wo[4], go[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const unsigned row = min(c0 + (GATED ? j & 1 : j) * 16 + fr, N - 1);
    wo[j] = row * static_cast<unsigned>(words * 4);
    go[j] = row * static_cast<unsigned>(groups * 2);
  }
  const int64_t ew = static_cast<int64_t>(e) * N * words, eg = static_cast<int64_t>(e) * N * groups;
  auto load_w = [&](P& q, int c) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int m = GATED ? j >> 1 : 0;
      auto at = [](const void* base, unsigned off) { return static_cast<const unsigned char*>(base) + off; };
      q.load(j, reinterpret_cast<const uint32_t*>(at(a.w[m] + ew + c * P::WPC, wo[j])), f);
      q.load_affine(j, reinterpret_cast<const unsigned short*>(at(a.s[m] + eg + c * NF, go[j])), reinterpret_cast<const unsigned short*>(at(a.z[m] + eg + c * NF, go[j])));
    }
  };
  f32x4v acc[4][NR];
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < NR; ++i) acc[j][i] = f32x4v{0};
  auto compute = [&](const P& q, int buf) {
    const unsigned char* xb = lds + buf * XBUF;
    const float* xm = xsum + buf * NF * 16 * NR;
#pragma unroll
    for (int g = 0; g < NF; ++g) {
      u32x4 op[4][SPG];
      float s[4], zc[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int t = 0; t < SPG; ++t) op[j][t] = q.operand(j, g * SPG + t, f);
        s[j] = gbx::act_to_f32<BF16>(q.sc[j][g]);
        zc[j] = gbx::act_to_f32<BF16>(q.ze[j][g]) - P::C * s[j];
      }
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        u32x4 xf[SPG];
#pragma unroll
        for (int t = 0; t < SPG; ++t) xf[t] = *reinterpret_cast<const u32x4*>(xb + (i * 16 + fr) * 256 + (((4 * (g * SPG + t) + f) ^ fr) & 15) * 16);
        const f32x4v xv = *reinterpret_cast<const f32x4v*>(xm + g * 16 * NR + i * 16 + 4 * f);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          f32x4v d = f32x4v{0};
#pragma unroll
          for (int t = 0; t < SPG; ++t) d = gbx::mfma16<BF16>(xf[t], op[j][t], d);
#pragma unroll
          for (int v = 0; v < 4; ++v) acc[j][i][v] = fmaf(s[j], d[v], fmaf(zc[j], xv[v], acc[j][i][v]));
        }
      }
    }
  };
  P q0, q1;
  load_x(0);
  load_w(q0, 0);
  store_x(0);
  if (n > 1) load_x(1);
  __syncthreads();
  for (int c = 0; c < n; c += 2) {                                      // (requests past the end repeat the last chunk)
    if (c + 1 < n) store_x(1);
    load_x(min(c + 2, n - 1));
    load_w(q1, min(c + 1, n - 1));
    compute(q0, 0);
    __syncthreads();
    if (c + 1 < n) {                                                    // (workgroup-uniform)
      if (c + 2 < n) store_x(0);
      load_x(min(c + 3, n - 1));
      load_w(q0, min(c + 2, n - 1));
      compute(q1, 1);
      __syncthreads();
    }
  }
  // a lane holds pairs 4 f + v of channel fr: through LDS of the wave's own, then rows of 64 (gated: 32) channels in 16-byte pieces
  constexpr int OC = GATED ? 32 : 64, OROW = 144;
  unsigned char* ot = lds + wave * (PT * OROW);
  // the roundings of the separate operations
  auto result = [&](float c, float up, float b) {
    unsigned short r = gbx::f32_to_act<BF16>(c);
    if constexpr (GATED) {
      const float g = gbx::act_to_f32<BF16>(r), u = gbx::act_to_f32<BF16>(gbx::f32_to_act<BF16>(up));
      r = gbx::f32_to_act<BF16>(gbx::act_to_f32<BF16>(gbx::f32_to_act<BF16>(g / (1.f + __expf(-g)))) * u);
    } else if (a.bias) {
      r = gbx::f32_to_act<BF16>(gbx::act_to_f32<BF16>(r) + b);
    }
    return r;
  };
  float odd = 0.f;                                                      // (0 times what is no finite number is no number)
#pragma unroll
  for (int j = 0; j < (GATED ? 2 : 4); ++j) {
    const float b = !GATED && a.bias ? gbx::act_to_f32<BF16>(a.bias[static_cast<int64_t>(e) * N + min(c0 + j * 16 + fr, N - 1)]) : 0.f;
#pragma unroll
    for (int i = 0; i < NR; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float c = acc[j][i][v], u = GATED ? acc[j + 2][i][v] : 0.f;
        odd = fmaf(c, 0.f, fmaf(u, 0.f, odd));
        *reinterpret_cast<unsigned short*>(ot + (i * 16 + 4 * f + v) * OROW + (j * 16 + fr) * 2) = result(c, u, b);
      }
  }
  auto visible = [] { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); __builtin_amdgcn_wave_barrier(); };
  visible();
  if (__any(odd != 0.f)) {                                              // infinite activations: those outputs again, weight by weight
#pragma unroll 1
    for (int p = lane; p < 16 * NR * OC; p += 64) {
      const int row = p / OC, ch = c0 + p % OC;
      unsigned short* at = reinterpret_cast<unsigned short*>(ot + row * OROW + p % OC * 2);
      constexpr unsigned short MOST = BF16 ? 0x7F80 : 0x7C00;
      if (lo + row >= hi || ch >= N || (*at & MOST) != MOST) continue;
      const unsigned short* x = a.x + static_cast<int64_t>(a.sorted[lo + row] / a.x_div) * K;
      float c[2] = {0.f, 0.f};
      for (int m = 0; m < (GATED ? 2 : 1); ++m)
        c[m] = gbx::expanded_dot<BITS, GRP, BF16>(x, a.w[m] + ew + ch * words, a.s[m] + eg + ch * groups, a.z[m] + eg + ch * groups, K);
      *at = result(c[0], c[1], !GATED && a.bias ? gbx::act_to_f32<BF16>(a.bias[static_cast<int64_t>(e) * N + ch]) : 0.f);
    }
    visible();
  }
  constexpr int PPR = OC / 8;                                           // 16-byte pieces per row
  const bool whole = c0 + OC <= N && N % 8 == 0;
#pragma unroll
  for (int k = 0; k < 16 * NR * PPR / 64; ++k) {
    const int p = k * 64 + lane, row = p / PPR, pc = p % PPR;
    if (lo + row >= hi) continue;
    unsigned short* dst = a.y + static_cast<int64_t>(a.sorted[lo + row]) * N + c0 + pc * 8;
    const u32x4 v = *reinterpret_cast<const u32x4*>(ot + row * OROW + pc * 16);
    if (whole) {
      *reinterpret_cast<u32x4*>(dst) = v;
    } else {
#pragma unroll
      for (int q = 0; q < 8; ++q)
        if (c0 + pc * 8 + q < N) dst[q] = static_cast<unsigned short>(v[q >> 1] >> (16 * (q & 1)));
    }
  }
}

template <int BITS, int GRP, bool BF16, bool GATED>
__global__ __launch_bounds__(256, 2) void packed_experts_kernel(const PackedArgs a) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[PLDS];
  const int u = xcd_unit(a.offsets[a.E + 2] * a.cols);
  if (u < 0) return;                                                    // (workgroup-uniform, as everything that picks the tile)
  const int bt = u / a.cols, col = u % a.cols;
  const int4 tab = a.tile_tab[bt];
  const int e = tab.x, lo = tab.y, hi = tab.z;
  if (e >= a.E) {                                                       // indices that name no expert: rows that nobody can take for results
    const int cn = min((GATED ? 128 : 256), a.N - col * (GATED ? 128 : 256));
    for (int i = threadIdx.x; i < (hi - lo) * cn; i += 256) a.y[static_cast<int64_t>(a.sorted[lo + i / cn]) * a.N + col * (GATED ? 128 : 256) + i % cn] = 0x7FFF;
    return;
  }
  if (hi - lo <= 16) packed_tile<BITS, GRP, BF16, GATED, 1>(a, lds, e, lo, hi, col);
  else if (hi - lo <= 32) packed_tile<BITS, GRP, BF16, GATED, 2>(a, lds, e, lo, hi, col);
  else packed_tile<BITS, GRP, BF16, GATED, 4>(a, lds, e, lo, hi, col);
}

template <int BITS, int GRP>
void launch(const PackedArgs& a, bool bf16, bool gated, unsigned grid, hipStream_t s) {
  if (bf16 && gated) packed_experts_kernel<BITS, GRP, true, true><<<grid, 256, 0, s>>>(a);
  else if (bf16) packed_experts_kernel<BITS, GRP, true, false><<<grid, 256, 0, s>>>(a);
  else if (gated) packed_experts_kernel<BITS, GRP, false, true><<<grid, 256, 0, s>>>(a);
  else packed_experts_kernel<BITS, GRP, false, false><<<grid, 256, 0, s>>>(a);
}
template <int BITS>
void launch(const PackedArgs& a, int group, bool bf16, bool gated, unsigned grid, hipStream_t s) {
  if (group == 32) launch<BITS, 32>(a, bf16, gated, grid, s);
  else if (group == 64) launch<BITS, 64>(a, bf16, gated, grid, s);
  else launch<BITS, 128>(a, bf16, gated, grid, s);
}

bool served(int64_t pairs, int64_t K, int E) { return pairs > 0 && pairs <= 0x3fffffff && K % 128 == 0 && E <= 4096; }
bool fits(int64_t N, int64_t K, int bits, int group) { return N * (K / 32 * bits * 4) <= 0xFFFFFFFFll && N * (K / group * 2) <= 0xFFFFFFFFll; }

}  // namespace
}  // namespace gbxm

using namespace gbxm;

extern "C" size_t gbxm_packed_experts_workspace(int64_t pairs, int32_t K, int32_t E) {
  return K > 0 && E > 0 && served(pairs, K, E) ? expert_buckets_bytes(pairs, PT, E) : 0;
}

extern "C" int gbxm_packed_experts(const gbxm_packed_experts_args* a, void* stream) {
  if (!a || a->pairs < 0 || a->x_div < 1 || a->E < 1 || a->N < 1 || a->K < 1 || a->bits < 2 || a->bits > 4 ||
      (a->group != 32 && a->group != 64 && a->group != 128) || a->K % a->group)
    return fail(GBXM_ERR_INVALID, "packed_experts: bad argument");
  if (a->pairs == 0) return GBXM_OK;
  const bool gated = a->up_qweight != nullptr;
  if (!a->x || !a->qweight || !a->scales || !a->zeros || !a->idx || !a->y || (gated && (!a->up_scales || !a->up_zeros || a->bias)))
    return fail(GBXM_ERR_INVALID, "packed_experts: null pointer");
  if (!served(a->pairs, a->K, a->E)) return fail(GBXM_ERR_UNSUPPORTED, "packed_experts: contractions in multiples of 128, at most 4096 experts");
  if (!fits(a->N, a->K, a->bits, a->group)) return fail(GBXM_ERR_UNSUPPORTED, "packed_experts: an expert's matrix of 4 GB or more");
  if (!a->ws || a->ws_bytes < gbxm_packed_experts_workspace(a->pairs, a->K, a->E)) return fail(GBXM_ERR_INVALID, "packed_experts: workspace too small");
  const uintptr_t wide = reinterpret_cast<uintptr_t>(a->x) | reinterpret_cast<uintptr_t>(a->qweight) | reinterpret_cast<uintptr_t>(a->up_qweight) |
                         reinterpret_cast<uintptr_t>(a->y) | reinterpret_cast<uintptr_t>(a->ws);
  const uintptr_t eight = reinterpret_cast<uintptr_t>(a->scales) | reinterpret_cast<uintptr_t>(a->zeros) | reinterpret_cast<uintptr_t>(a->up_scales) |
                          reinterpret_cast<uintptr_t>(a->up_zeros);
  if (wide % 16 || eight % 8) return fail(GBXM_ERR_UNSUPPORTED, "packed_experts: rows and packed words on 16, scales and zeros on 8 bytes");
  hipStream_t s = static_cast<hipStream_t>(stream);
  ExpertBuckets k;
  const int rc = expert_buckets(a->idx, static_cast<int>(a->pairs), PT, a->E, a->ws, &k, s);
  if (rc != GBXM_OK) return rc;
  const unsigned short *sc = static_cast<const unsigned short*>(a->scales), *ze = static_cast<const unsigned short*>(a->zeros);
  const int cols = gated ? (a->N + 127) / 128 : (a->N + 255) / 256;
  const int64_t units = static_cast<int64_t>(k.tiles) * cols;
  if (units > 0x7fffffff - 8) return fail(GBXM_ERR_UNSUPPORTED, "packed_experts: grid");
  const PackedArgs p{static_cast<const unsigned short*>(a->x), {a->qweight, a->up_qweight}, {sc, static_cast<const unsigned short*>(a->up_scales)},
                     {ze, static_cast<const unsigned short*>(a->up_zeros)}, static_cast<const unsigned short*>(a->bias), k.offsets, k.sorted, k.tile_tab,
                     static_cast<unsigned short*>(a->y), a->N, a->K, a->E, a->x_div, cols};
  const unsigned grid = static_cast<unsigned>((units + 7) / 8 * 8);
  if (a->bits == 2) launch<2>(p, a->group, !a->f16, gated, grid, s);
  else if (a->bits == 3) launch<3>(p, a->group, !a->f16, gated, grid, s);
  else launch<4>(p, a->group, !a->f16, gated, grid, s);
  return after_launch("packed_experts");
}
