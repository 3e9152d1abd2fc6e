// Quantised products of 2 to 32 rows: the rows stay in registers, the packed weights stream past them.  More rows are groups of up to 32, which share the chip out between
// them (grid.y; the weights come from memory for the first and from the L2 for the others): gbx_qlinear_groups, mfma_rows.hip.
//   y[m, n] = sum_g s[n, g] (sum_k x (C + q)) + (z[n, g] - C s[n, g]) sum_k x
// A workgroup owns the whole contraction (up to 4096) for up to 8 (16 rows of x: 16) tiles of 16 outputs.  Each of its eight waves owns CW
// neighbouring chunks of 128 of it: it brings its part of the rows into registers once (LDS-DMA in row order, then fragments), and walks the tiles with
// weights requested up to three tiles ahead.  Waves share nothing until the end, where their sums meet in LDS: one barrier per workgroup.
//   * fields go to the matrix cores as the numbers C + q (packed_fields.h); sum_k x per group comes from a product with ones at the start;
//   * lane quarter f loads scale and zero of chunk f of the wave: the scales reach the other quarters by one exchange a chunk, and the zeros' part
//     sum_g (z - C s)[n, g] (sum x)[m, g] is one fp32 16 x 16 x 4 product per group place of a tile, lane quarter f being its k.
//   * neighbouring lanes fetch neighbouring bytes of one weight row, and the words then change lanes: with a lane per row, as the matrix cores want them, every lane
//     is a request of its own and a load takes 64 cycles of the CU's address path instead of some 25 (32 rows of 28672 x 4096, 2 bits 22.7 -> 20.2 us);
//   * what is cold is the code: a launch starts with some 190 cycles per 64 bytes of straight-line code on its way to the first request, so requests go out
//     first, tile addresses are scalar, and the repair of odd sums is out of the way.
// An output whose sum is not finite is taken again, weight by weight (expanded_dot).
// Bound by its start -- arguments, code, then the rows: 256 KB of them a CU (32 x 4096) take 3 us -- and by the field and scale arithmetic of a tile.  Measured (us, weights
// cold; before: mfma_rows.hip, and mfma_batch.hip where groups are of 128 and K a multiple of 1024): 27 rows of 8192 x 3072, 3 bits, group 64
// 14.3 -> 10.0; 32 rows of 14336 x 4096, 4 bits, group 32 49 -> 18.5; 32 of 16384 x 2048, 3 bits, group 32 34 -> 14.3; group 128: 16 of 11008 x 4096, 3 bits 18.9 -> 10.8;
// 2 of 4096 x 4096, 4 bits 9.2 -> 6.7; 17, 2 bits 10.0 -> 7.6; q, k and v of 4096 x 4096, 32 rows 11.6 -> 9.1.
#pragma once
#include <algorithm>
#include <type_traits>
#include "kernels.h"
#include "mfma_slab.h"
#include "packed_fields.h"

namespace gbx {
namespace slab {

constexpr int SLAB_WAVES = 8;
constexpr int SLAB_BYTES = 16384;          // a wave's LDS: its rows on their way to the registers, then its sums
constexpr int SLAB_LDS = SLAB_WAVES * SLAB_BYTES;

struct SlabArgs {
  const unsigned short* x;
  const uint32_t* qw[3];
  const unsigned short *sc[3], *ze[3], *bias[3];
  unsigned short* y[3];
  int N[3], block0[3];                     // rows of a matrix, first workgroup of it
  int M, K, tpb;                           // tpb: tiles of a workgroup
  int rows;                                // of a group of x's rows (at most 32), grid.y of them
};

// s_waitcnt: at most n vector memory accesses outstanding
__device__ __forceinline__ constexpr int slab_vmcnt(int n) { return (n & 0xF) | ((n >> 4) << 14) | (0x7 << 4) | (0xF << 8); }

template <typename T> __device__ __forceinline__ T pick(int g, T a, T b, T c) { return g == 0 ? a : g == 1 ? b : c; }

template <int N, int I = 0, typename F> __device__ __forceinline__ void each(F&& fn) {
  if constexpr (I < N) { fn(std::integral_constant<int, I>{}); each<N, I + 1>(fn); }
}

// Reads from `end` bytes on give zero and make no access.  gfx950 takes the scalar offset into that check, and one that is past the end by itself reads nothing (lanes
// of 64 bytes over 4096, scalar offsets 0, 1024, 4032, 4096 and 65 536: 64, 48, 1, 0 and 0 of them read; over 0 bytes none, from registers and to LDS alike).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t slab_buffer(const void* p, int64_t first, int64_t end) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(static_cast<const char*>(p)) + first, 0, static_cast<int>(end - first < 0x7FFFFFFF ? end - first : 0x7FFFFFFF), 0x00020000);
}

template <int BITS, int GRP, bool BF16, int MT, int CW>
__device__ __forceinline__ void qgemm_slab(const SlabArgs& a) {
  typedef Packed<BITS, GRP, BF16, CW> P;
  constexpr int NF = P::NF, SPG = P::SPG;
  // tiles of weights in registers: what the rows leave of them, the first of them under way while the rows come
  constexpr int RING = CW * MT * 16 + 60 + 4 * (CW * P::RAW + 2 * NF) <= 250 ? 4 : CW * MT * 16 + 60 + 3 * (CW * P::RAW + 2 * NF) <= 250 ? 3 : 2;
  constexpr int SLOTS = SLAB_BYTES / (MT * 4096), FIRST = SLOTS < CW ? SLOTS : CW;      // chunks of rows in flight
  extern __shared__ __attribute__((aligned(16))) unsigned char slab_lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), fr = lane & 15, f = lane >> 4;
  unsigned char* mine = slab_lds + wave * SLAB_BYTES;
  const int K = a.K, words = (K >> 5) * BITS, groups = K / GRP, chunks = K >> 7;
  const int c0 = wave * CW, own = chunks - c0;                         // the wave's first chunk, and how many there are from it on
  // (every argument is asked for at once: one trip to memory instead of one per use)
  asm volatile("" ::"s"(a.qw[0]), "s"(a.qw[1]), "s"(a.qw[2]), "s"(a.sc[0]), "s"(a.sc[1]), "s"(a.sc[2]), "s"(a.ze[0]), "s"(a.ze[1]), "s"(a.ze[2]), "s"(a.x), "s"(a.N[0]), "s"(a.N[1]), "s"(a.N[2]),
               "s"(a.block0[1]), "s"(a.block0[2]), "s"(a.M), "s"(a.K), "s"(a.tpb), "s"(a.rows));
  const int m_first = blockIdx.y * a.rows, M = min(a.rows, a.M - m_first);
  const unsigned short* xg = a.x + static_cast<int64_t>(m_first) * K;
  const int seg = (blockIdx.x >= a.block0[1]) + (blockIdx.x >= a.block0[2]);
  const int N = pick(seg, a.N[0], a.N[1], a.N[2]), tile0 = (blockIdx.x - pick(seg, a.block0[0], a.block0[1], a.block0[2])) * a.tpb, nt = min(a.tpb, ((N + 15) >> 4) - tile0);

  if (own > 0) {
    // buffers: a tile's place is scalar, a lane's place in it does not change, rows past the end read as zeros
    const int lr = lane >> 2, lf = lane & 3;                            // neighbouring lanes fetch neighbouring pieces of one row
    const int vw = lr * words * 4 + P::lane_byte(lf), va = (lr * groups + lf * NF) * 2;
    const int64_t wfirst = static_cast<int64_t>(tile0) * 64 * words, wend = static_cast<int64_t>(N) * words * 4;
    const int64_t afirst = static_cast<int64_t>(tile0) * 32 * groups, aend = static_cast<int64_t>(N) * groups * 2;
    const uint32_t* qw = pick(seg, a.qw[0], a.qw[1], a.qw[2]);
    const unsigned short *sc = pick(seg, a.sc[0], a.sc[1], a.sc[2]), *ze = pick(seg, a.ze[0], a.ze[1], a.ze[2]);
    auto load = [&](int i, P& w) {
      const bool none = i >= nt;                                       // past the last tile: empty buffers, which cost no memory access
      const __amdgpu_buffer_rsrc_t rw = slab_buffer(qw, wfirst, none ? wfirst : wend);
      const __amdgpu_buffer_rsrc_t rs = slab_buffer(sc, afirst, none ? afirst : aend), rz = slab_buffer(ze, afirst, none ? afirst : aend);
#pragma unroll
      for (int j = 0; j < CW; ++j) w.load_buffer(j, rw, vw, i * 64 * words + (c0 + j) * (P::WPC * 4));
      w.load_affine_buffer(0, rs, rz, va, i * 32 * groups + c0 * NF * 2);
      asm volatile("" ::: "memory");                                   // (here, and not where the words are used)
    };
    // the rows: 16-byte piece p of row r of a chunk lies in slot p ^ (r % 16) of the row's 256 bytes, so that the 16 rows of a fragment read meet
    // different banks; four rows a request, in pieces of 256 bytes
    packed_x4 x[CW][MT][4];
    float xs[NF][MT];                                                  // lane (m, f): the sum of row m over a group of chunk f
    const __amdgpu_buffer_rsrc_t rx = slab_buffer(xg, 0, static_cast<int64_t>(M) * K * 2);
    int from[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) from[i] = f * K * 2 + ((fr ^ f ^ (4 * i)) << 4);
    auto stage = [&](int j, int i) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (__attribute__((address_space(3))) void*)(mine + (j % SLOTS) * (MT * 4096) + i * 1024), 16, from[i & 3],
                                               (c0 + j) * 256 + i * 8 * K, 0, 0);
    };
#pragma unroll
    for (int j = 0; j < FIRST; ++j)
#pragma unroll
      for (int i = 0; i < MT * 4; ++i) stage(j, i);
    P ring[RING];
#pragma unroll
    for (int i = 0; i < RING; ++i) load(i, ring[i]);
    each<CW>([&](auto jc) {
      // requests behind the chunk's: of its round, and of the weights at least one a chunk
      constexpr int j = decltype(jc)::value, later = j < FIRST ? (FIRST - 1 - j) * MT * 4 + RING * CW : (CW - 1 - j) * MT * 4;
      __builtin_amdgcn_s_waitcnt(slab_vmcnt(later));
      asm volatile("" ::: "memory");
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          auto piece = [&](int o) { return mine + (j % SLOTS) * (MT * 4096) + (16 * i + fr) * 256 + ((o ^ fr) << 4); };
          if constexpr (BITS == 2 && GRP == 32) {          // half of a word's 16: values 4 (f % 2) .. + 3 and the 4 that lie 8 further on
            const int o = 4 * t + 2 * (f >> 1);
            const packed_x2 lo = *reinterpret_cast<const packed_x2*>(piece(o) + 8 * (f & 1)), hi = *reinterpret_cast<const packed_x2*>(piece(o + 1) + 8 * (f & 1));
            x[j][i][t] = packed_x4{lo.x, lo.y, hi.x, hi.y};
          } else {
            x[j][i][t] = *reinterpret_cast<const packed_x4*>(piece(GRP == 128 ? 4 * f + t : GRP == 64 ? (t >> 1) * 8 + 2 * f + (t & 1) : 4 * t + f));
          }
        }
      if (j + 1 == FIRST && FIRST < CW) {                              // the next round takes the same places
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int q = FIRST; q < CW; ++q)
#pragma unroll
          for (int i = 0; i < MT * 4; ++i) stage(q, i);
      }
    });
    static_assert(CW <= 2 * SLOTS, "two rounds");
    unsigned mask = P::MASK, magic = P::MAGIC;
    asm("" : "+s"(mask));
    asm("" : "+v"(magic));
    constexpr unsigned ONE = BF16 ? 0x3F803F80u : 0x3C003C00u;
    const packed_x4 ones{ONE, ONE, ONE, ONE};
#pragma unroll
    for (int j = 0; j < CW; ++j)
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        packed_order<BITS, GRP>(x[j][i]);
#pragma unroll
        for (int g = 0; g < NF; ++g) {
          f32x4v d{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int t = 0; t < SPG; ++t) d = mfma16<BF16>(ones, x[j][i][g * SPG + t], d);
          xs[g][i] = j == 0 || f == j ? d[0] : xs[g][i];
        }
      }

    const bool live = lf < own && lf < CW;                             // chunk lf counts (the words of one that does not meet scales of zero)
    auto from_lane = [](int v, int at) { return __builtin_amdgcn_ds_bpermute(at * 4, v); };
    const int here = fr * 4 + f;                                       // the lane that fetched this lane's operands
    unsigned char* put = mine + lane * 16;
    auto compute = [&](P& w) {
      f32x4v acc[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[m] = f32x4v{0.f, 0.f, 0.f, 0.f};
      float sc[NF];
#pragma unroll
      for (int g = 0; g < NF; ++g) {
        sc[g] = live ? act_to_f32<BF16>(w.sc[0][g]) : 0.f;
        const float zc = __int_as_float(from_lane(__float_as_int(live ? act_to_f32<BF16>(w.ze[0][g]) - P::C * sc[g] : 0.f), here));
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(xs[g][m], zc, acc[m], 0, 0, 0);
      }
#pragma unroll
      for (int j = 0; j < CW; ++j) {
#pragma unroll
        for (int q = 0; q < P::RAW; ++q) w.raw[j][q] = from_lane(w.raw[j][q], here);
#pragma unroll
        for (int g = 0; g < NF; ++g) {
          const float s = __int_as_float(from_lane(__float_as_int(sc[g]), fr * 4 + j));
          packed_x4 op[SPG];
#pragma unroll
          for (int t = 0; t < SPG; ++t) op[t] = w.operand(j, g * SPG + t, f, mask, magic);
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            f32x4v d{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int t = 0; t < SPG; ++t) d = mfma16<BF16>(x[j][m][g * SPG + t], op[t], d);
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[m][v] = fmaf(s, d[v], acc[m][v]);
          }
        }
      }
#pragma unroll
      for (int m = 0; m < MT; ++m) *reinterpret_cast<f32x4v*>(put + m * 1024) = acc[m];
      put += MT * 1024;
    };
    // (past the last tile it is asked for again: without a branch around the loads, every wait is for the words that are needed next)
#pragma unroll 1
    for (int i = 0; i < nt;) {
#pragma unroll
      for (int u = 0; u < RING; ++u) {
        compute(ring[u]);
        if (++i >= nt) break;
        load(i + RING - 1, ring[u]);
      }
    }
  } else {
#pragma unroll 1
    for (int p = lane; p < nt * MT * 64; p += 64) *reinterpret_cast<f32x4v*>(mine + p * 16) = f32x4v{0.f, 0.f, 0.f, 0.f};
  }
  __syncthreads();

  // lane l of a tile's place holds rows 16 i + 4 (l / 16) + v of output l % 16
  auto sum = [&](int at) {
    f32x4v v = *reinterpret_cast<const f32x4v*>(slab_lds + at * 16);
#pragma unroll
    for (int w = 1; w < SLAB_WAVES; ++w) v += *reinterpret_cast<const f32x4v*>(slab_lds + w * SLAB_BYTES + at * 16);
    return v;
  };
  const int places = nt * MT * 64, n0 = tile0 * 16;
  const unsigned short* bias = a.bias[seg];
  unsigned short* y = a.y[seg] + static_cast<int64_t>(m_first) * N;
  auto write = [&](int n, int m, float r) {
    const size_t at = static_cast<size_t>(m) * N + n;
    unsigned short o = f32_to_act<BF16>(r);
    if (bias) o = f32_to_act<BF16>(act_to_f32<BF16>(o) + act_to_f32<BF16>(bias[n]));       // (a second rounding)
    y[at] = o;
  };
  bool finite = true;
#pragma unroll 1
  for (int p = tid; p < places; p += 64 * SLAB_WAVES) {
    const int m0 = (p >> 6) % MT * 16 + 4 * f, n = n0 + p / (MT * 64) * 16 + fr;
    const f32x4v s = sum(p);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      finite &= __builtin_isfinite(s[v]);
      if (n < N && m0 + v < M) write(n, m0 + v, s[v]);
    }
  }
  if (finite) return;
  // (the places that this thread has written: nobody else's results change)
#pragma unroll 1
  for (int q = 0; tid + (q >> 2) * 64 * SLAB_WAVES < places; ++q) {
    const int p = tid + (q >> 2) * 64 * SLAB_WAVES, v = q & 3, m = (p >> 6) % MT * 16 + 4 * f + v;
    const int64_t n = n0 + p / (MT * 64) * 16 + fr;
    if (n >= N || m >= M) continue;
    float r = 0.f;
    for (int w = 0; w < SLAB_WAVES; ++w) r += *reinterpret_cast<const float*>(slab_lds + w * SLAB_BYTES + p * 16 + v * 4);
    if (!__builtin_isfinite(r))
      write(n, m, expanded_dot<BITS, GRP, BF16>(xg + static_cast<int64_t>(m) * K, a.qw[seg] + n * words, a.sc[seg] + n * groups, a.ze[seg] + n * groups, K));
  }
}

template <int BITS, int GRP, bool BF16, int MT, int CW>
__global__ __launch_bounds__(64 * SLAB_WAVES) void qgemm_slab_kernel(const SlabArgs a) {
  qgemm_slab<BITS, GRP, BF16, MT, CW>(a);
}

template <int BITS, int GRP, bool BF16, int MT, int CW>
hipError_t launch_slab_shape(const MfmaArgs& a, hipStream_t s) {
  static DeviceOnce done;
  if (done.pending()) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&qgemm_slab_kernel<BITS, GRP, BF16, MT, CW>), hipFuncAttributeMaxDynamicSharedMemorySize, SLAB_LDS);
    if (e != hipSuccess) return e;
    done.done();
  }
  SlabArgs t{a.x, {a.qweight, a.qweight_x[0], a.qweight_x[1]}, {a.scales, a.scales_x[0], a.scales_x[1]}, {a.zeros, a.zeros_x[0], a.zeros_x[1]},
             {a.bias, a.bias_x[0], a.bias_x[1]}, {a.y, a.y_x[0], a.y_x[1]}, {a.N, 0, 0}, {0, 0x7FFFFFFF, 0x7FFFFFFF}, a.M, a.K, 0, 0};
  constexpr int most = SLAB_BYTES / (MT * 1024);
  // a workgroup fills a CU: as many tiles a workgroup as spread them evenly over as few rounds of 256 as their sums' place in LDS allows
  int tiles = 0;
  for (int g = 0; g < std::max(a.nseg, 1); ++g) {
    if (a.nseg > 1) t.N[g] = a.n_seg[g];
    tiles += (t.N[g] + 15) / 16;
  }
  const int groups = (a.M + 31) / 32, wgs = std::max(256 / groups, 1);         // (groups of rows share the chip)
  t.rows = (a.M + groups - 1) / groups;
  const int rounds = (tiles + wgs * most - 1) / (wgs * most);
  t.tpb = (tiles + wgs * rounds - 1) / (wgs * rounds);
  int blocks = 0;
  for (int g = 0; g < std::max(a.nseg, 1); ++g) {
    t.block0[g] = blocks;
    blocks += ((t.N[g] + 15) / 16 + t.tpb - 1) / t.tpb;
  }
  qgemm_slab_kernel<BITS, GRP, BF16, MT, CW><<<dim3(blocks, groups), 64 * SLAB_WAVES, SLAB_LDS, s>>>(t);
  return hipGetLastError();
}

template <int BITS, int GRP, int MT, int CW>
hipError_t launch_slab_type(const MfmaArgs& a, bool bf16, hipStream_t s) {
  return bf16 ? launch_slab_shape<BITS, GRP, true, MT, CW>(a, s) : launch_slab_shape<BITS, GRP, false, MT, CW>(a, s);
}

template <int BITS, int GRP, int MT>
hipError_t launch_slab_chunks(const MfmaArgs& a, bool bf16, hipStream_t s) {
  switch ((a.K / 128 + SLAB_WAVES - 1) / SLAB_WAVES) {
    case 1: return launch_slab_type<BITS, GRP, MT, 1>(a, bf16, s);
    case 2: return launch_slab_type<BITS, GRP, MT, 2>(a, bf16, s);
    case 3: return launch_slab_type<BITS, GRP, MT, 3>(a, bf16, s);
    case 4: return launch_slab_type<BITS, GRP, MT, 4>(a, bf16, s);
    default: return hipErrorInvalidValue;
  }
}

template <int BITS, int GRP>
hipError_t launch_slab_rows(const MfmaArgs& a, bool bf16, hipStream_t s) {
  const int groups = (a.M + 31) / 32;
  return (a.M + groups - 1) / groups <= 16 ? launch_slab_chunks<BITS, GRP, 1>(a, bf16, s) : launch_slab_chunks<BITS, GRP, 2>(a, bf16, s);
}

}  // namespace slab

template <int BITS>
hipError_t launch_slab_bits(const MfmaArgs& a, bool bf16, hipStream_t s) {
  return a.log2g == 7 ? slab::launch_slab_rows<BITS, 128>(a, bf16, s)
         : a.log2g == 6 ? slab::launch_slab_rows<BITS, 64>(a, bf16, s)
                        : slab::launch_slab_rows<BITS, 32>(a, bf16, s);
}

}  // namespace gbx
