// Quantised products of 2 to 32 rows over contractions whose rows do not fit the registers (beyond 4096; shorter ones: mfma_slab_impl.h, except for few rows off the
// grid of 1024), outside the batch kernel.
//   y[m, n] = sum_g s[n, g] (sum_k x (C + q)) + (z[n, g] - C s[n, g]) sum_k x
// A workgroup takes 16 NT outputs, its waves share out the chunks of 128 of K; packed words, scales and the rows' image go straight to the registers of
// the lane that feeds them to the matrix cores (packed_fields.h), one chunk ahead of the one being multiplied; sum_k x comes from the matrix cores too
// (a product with ones, shared by the wave's outputs), and the waves' sums meet in LDS.  No weight is expanded or rounded to the activation type; only an
// output whose sum is not finite is taken again, weight by weight (expanded_dot): infinite activations give what their products with the weights give.
// Bound by the latency of a wave's two or three chunks and by the rows' way through the first cache (27 rows: five bytes of rows for each byte of
// weights).  Measured against the dequantising kernel that took these (us, weights cold): 4 bits, group 32: 8 rows of 4096 x 11008 38.5 -> 20.4.
#include "gbx_env.h"
#include "mfma_slab.h"
#include "packed_fields.h"

namespace gbx {
namespace {

constexpr int RW = 8;                      // waves

template <int BITS, int GRP, bool BF16, int MT, int NT>
__global__ __launch_bounds__(64 * RW) void qgemm_rows_kernel(MfmaArgs args) {
  typedef Packed<BITS, GRP, BF16, NT> P;
  constexpr int NF = P::NF, SPG = P::SPG;
  __shared__ float part[RW][MT * NT * 256];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, fr = lane & 15, f = lane >> 4;
  // the matrix: one, or one of up to three that share the rows, tiled one after another
  const uint32_t* qw = args.qweight;
  const unsigned short *sc = args.scales, *ze = args.zeros, *bias = args.bias;
  unsigned short* y = args.y;
  int N = args.nseg > 1 ? args.n_seg[0] : args.N, tile = blockIdx.x;
  for (int g = 1; g < args.nseg && tile >= (N + 16 * NT - 1) / (16 * NT); ++g) {
    tile -= (N + 16 * NT - 1) / (16 * NT);
    qw = args.qweight_x[g - 1]; sc = args.scales_x[g - 1]; ze = args.zeros_x[g - 1]; bias = args.bias_x[g - 1]; y = args.y_x[g - 1];
    N = args.n_seg[g];
  }
  const unsigned short* x = args.x;
  const int M = args.M, K = args.K;
  const int n0 = tile * (16 * NT), chunks = K >> 7, words = (K >> 5) * BITS, groups = K / GRP;
  const unsigned short* xp[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) xp[i] = x + static_cast<int64_t>(min(16 * i + fr, M - 1)) * K;
  struct Chunk { P w; packed_x4 x[MT][4]; };
  auto load = [&](int c, Chunk& k) {
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int64_t n = min(n0 + 16 * j + fr, N - 1);
      k.w.load(j, qw + n * words + c * P::WPC, f);
      k.w.load_affine(j, sc + n * groups + c * NF, ze + n * groups + c * NF);
    }
    // the octet of step t: 4 f + t of 16 (groups of 128), 2 f + t % 2 of the group's eight (64), f of its four (32)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const unsigned short* p = xp[i] + c * 128;
        if constexpr (BITS == 2 && GRP == 32) {            // half of the word's 16: values 4 (f % 2) .. + 3 and the 4 that lie 8 further on
          const packed_x2 lo = *reinterpret_cast<const packed_x2*>(p + 32 * t + 16 * (f >> 1) + 4 * (f & 1));
          const packed_x2 hi = *reinterpret_cast<const packed_x2*>(p + 32 * t + 16 * (f >> 1) + 4 * (f & 1) + 8);
          k.x[i][t] = packed_x4{lo.x, lo.y, hi.x, hi.y};
        } else {
          const int o = GRP == 128 ? 4 * f + t : GRP == 64 ? (t >> 1) * 8 + 2 * f + (t & 1) : 4 * t + f;
          k.x[i][t] = *reinterpret_cast<const packed_x4*>(p + 8 * o);
        }
      }
  };
  auto arrange = [&](Chunk& k) {
#pragma unroll
    for (int i = 0; i < MT; ++i) packed_order<BITS, GRP>(k.x[i]);
  };
  constexpr unsigned ONE = BF16 ? 0x3F803F80u : 0x3C003C00u;
  const packed_x4 ones{ONE, ONE, ONE, ONE};
  f32x4v acc[NT][MT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[j][i] = f32x4v{0.f, 0.f, 0.f, 0.f};
  auto compute = [&](Chunk& k) {
    arrange(k);
#pragma unroll
    for (int g = 0; g < NF; ++g) {
      f32x4v xs[MT];
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        xs[i] = f32x4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < SPG; ++t) xs[i] = mfma16<BF16>(k.x[i][g * SPG + t], ones, xs[i]);
      }
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const float s = act_to_f32<BF16>(k.w.sc[j][g]), zc = act_to_f32<BF16>(k.w.ze[j][g]) - P::C * s;
        packed_x4 op[SPG];
#pragma unroll
        for (int t = 0; t < SPG; ++t) op[t] = k.w.operand(j, g * SPG + t, f);
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          f32x4v d{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int t = 0; t < SPG; ++t) d = mfma16<BF16>(k.x[i][g * SPG + t], op[t], d);
#pragma unroll
          for (int v = 0; v < 4; ++v) acc[j][i][v] = fmaf(s, d[v], fmaf(zc, xs[i][v], acc[j][i][v]));
        }
      }
    }
  };
  if (wave < chunks) {
    Chunk a, b;
    load(wave, a);
    for (int c = wave; c < chunks; c += 2 * RW) {
      if (c + RW < chunks) load(c + RW, b);
      compute(a);
      if (c + RW < chunks) {
        if (c + 2 * RW < chunks) load(c + 2 * RW, a);
        compute(b);
      }
    }
  }
  // a lane holds rows 4 f + v of output fr
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) part[wave][(i * 16 + 4 * f + v) * (16 * NT) + 16 * j + fr] = acc[j][i][v];
  __syncthreads();
  auto put = [&](int n, int m, float v) {
    unsigned short r = f32_to_act<BF16>(v);                                // (a bias is a second rounding)
    if (bias) r = f32_to_act<BF16>(act_to_f32<BF16>(r) + act_to_f32<BF16>(bias[n]));
    y[static_cast<int64_t>(m) * N + n] = r;
  };
  auto sum = [&](int i) {
    float s = 0.f;
#pragma unroll
    for (int v = 0; v < RW; ++v) s += part[v][i];
    return s;
  };
  bool finite = true;
  for (int i = threadIdx.x; i < MT * NT * 256; i += 64 * RW) {
    const int n = n0 + i % (16 * NT), m = i / (16 * NT);
    const float s = sum(i);
    finite &= __builtin_isfinite(s);
    if (n < N && m < M) put(n, m, s);
  }
  if (finite) return;
#pragma unroll 1
  for (int i = threadIdx.x; i < MT * NT * 256; i += 64 * RW) {
    const int n = n0 + i % (16 * NT), m = i / (16 * NT);
    if (n < N && m < M && !__builtin_isfinite(sum(i)))
      put(n, m, expanded_dot<BITS, GRP, BF16>(x + static_cast<int64_t>(m) * K, qw + static_cast<int64_t>(n) * words, sc + static_cast<int64_t>(n) * groups,
                                              ze + static_cast<int64_t>(n) * groups, K));
  }
}

template <int BITS, int GRP, int MT>
hipError_t launch_rows(const MfmaArgs& a, bool bf16, hipStream_t s) {
#define GBX_QROWS(NT)                                                                               \
  do {                                                                                              \
    int grid = 0;                                                                                   \
    for (int g = 0; g < (a.nseg > 1 ? a.nseg : 1); ++g) grid += ((a.nseg > 1 ? a.n_seg[g] : a.N) + 16 * NT - 1) / (16 * NT); \
    if (bf16) qgemm_rows_kernel<BITS, GRP, true, MT, NT><<<grid, 64 * RW, 0, s>>>(a);               \
    else qgemm_rows_kernel<BITS, GRP, false, MT, NT><<<grid, 64 * RW, 0, s>>>(a);                   \
  } while (0)
  // 32 outputs a workgroup share the rows' image where that still leaves a workgroup for every CU (16 | 32 outputs, us, 2, 8 and 27 rows: 3 bits, group 64, 4096 x 4224
  // 6.3 7.0 10.6 | 8.8 9.3 12.8, 4112 x 4224 8.7 10.1 18.6 | 8.8 9.4 12.9, 8192 x 11008 21.1 24.8 43.8 | 19.5 21.4 30.1; 4 bits, group 32, 4096 x 11008 17.8 20.2 31.1 | 28.7
  // 31.6 53.3, 4112 x 11008 30.3 35.8 58.0 | 28.6 31.7 53.4)
  if (a.N > 4096) GBX_QROWS(2);
  else GBX_QROWS(1);
#undef GBX_QROWS
  return hipGetLastError();
}

template <int BITS, int GRP>
hipError_t launch_rows(const MfmaArgs& a, bool bf16, hipStream_t s) {
  return a.M <= 16 ? launch_rows<BITS, GRP, 1>(a, bf16, s) : launch_rows<BITS, GRP, 2>(a, bf16, s);
}

template <int BITS>
hipError_t launch_rows(const MfmaArgs& a, bool bf16, hipStream_t s) {
  return a.log2g == 7 ? launch_rows<BITS, 128>(a, bf16, s) : a.log2g == 6 ? launch_rows<BITS, 64>(a, bf16, s) : launch_rows<BITS, 32>(a, bf16, s);
}

}  // namespace

constexpr int SLAB_ROWS = 4096;             // in groups of 32

// (contractions under 1024 of up to 32 rows: see below; one row: what is left of 33, by the kernel of the other 32)
hipError_t launch_qgemm_slab(const MfmaArgs& a, int bits, bool bf16, hipStream_t s) {
  uintptr_t affine = reinterpret_cast<uintptr_t>(a.scales) | reinterpret_cast<uintptr_t>(a.zeros);
  for (int g = 1; g < a.nseg; ++g) affine |= reinterpret_cast<uintptr_t>(a.scales_x[g - 1]) | reinterpret_cast<uintptr_t>(a.zeros_x[g - 1]);
  if (a.swiglu || a.ws || a.M < 1 || a.M > (a.nseg > 1 ? 64 : SLAB_ROWS) || a.K % 128 || (a.M <= 32 && a.K < 1024) || a.log2g < 5 || a.log2g > 7 || affine % (256u >> a.log2g)) return hipErrorInvalidValue;
  return bits == 2 ? launch_slab_bits<2>(a, bf16, s) : bits == 3 ? launch_slab_bits<3>(a, bf16, s) : bits == 4 ? launch_slab_bits<4>(a, bf16, s) : hipErrorInvalidValue;
}

// Contractions off the grid of eight chunks leave some of the register-resident kernel's waves without work and give the others as much as a longer one would, while
// here every wave starts on one: few rows whose outputs fit one round stay here.  2-bit groups of 32, whose fields cost more to take apart here, do not; 3-bit ones stay with
// more rows too where two row tiles of four chunks leave the registers no room for two tiles of weights.  Here | there, us, 4096 outputs, 2, 8, 16, 17 and 32 rows: x 1152, 4
// bits, group 64 3.8 4.1 4.5 4.8 5.5 | 4.4 4.5 4.6 5.2 5.3, 3 bits, group 128 3.5 3.8 4.1 4.5 5.2 | 4.0 4.0 4.1 4.7 4.8; x 1408, 3 bits 3.6 3.9 4.3 4.8 5.5 | 4.2 4.2 4.4 4.9
// 5.1; x 1536 4.5 4.9 5.4 5.7 6.6 | 4.5 4.6 4.7 5.3 5.5 and 3.7 4.0 4.5 4.9 5.8 | 4.2 4.2 4.3 4.9 5.0; x 3200 5.4 6.0 .. | 6.3 6.4 .. and 5.0 5.4 .. | 5.5 5.5 ..; 2 bits, group
// 32, x 1152 4.7 5.1 5.9 6.8 8.1 | 4.7 4.7 4.8 5.5 5.6; 11008 outputs, x 1152 7.1 7.5 .. | 5.9 6.0 ..; there in parts of here, 3, 6, 12, 16, 17 and 32 rows: 3 bits, group 32,
// x 1152 1.18 1.18 1.16 1.09 1.04 0.97, x 1664 1.09 1.08 1.05 1.00 0.97 0.87, x 2560 0.85 0.83 0.78 0.77 0.69 0.63, x 3200 0.95 0.93 0.90 0.89 1.28 1.18; 4 bits, group 32,
// x 1152 1.08 1.05 0.99 0.96 1.01 0.92.
static bool rows_start_evenly(const MfmaArgs& a, int bits) {
  const int chunks = a.K >> 7;
  if (chunks % RW == 0 || a.N > 4096) return false;
  if (a.log2g == 5) return bits == 3 ? (chunks < 12 ? a.M <= 16 : chunks < 16 ? a.M <= 6 : chunks > 24 && a.M > 16) : bits == 4 && chunks < 12 && a.M <= 6;
  return a.M <= (chunks < 12 ? (bits == 3 ? 16 : 12) : 6);
}

// Contractions under 1024 stay with the dequantising kernel although it is the slower one (16 rows of 4096 x 512, 4 bits, group 128: 5.7 us there, 3.2
// here): models that small are held to recorded token histories, and their results keep their bits.
hipError_t launch_qgemm_rows(const MfmaArgs& a, int bits, bool bf16, hipStream_t s) {
  uintptr_t affine = reinterpret_cast<uintptr_t>(a.scales) | reinterpret_cast<uintptr_t>(a.zeros);
  for (int g = 1; g < a.nseg; ++g) affine |= reinterpret_cast<uintptr_t>(a.scales_x[g - 1]) | reinterpret_cast<uintptr_t>(a.zeros_x[g - 1]);
  if (a.swiglu || a.M < 2 || a.M > 32 || a.K % 128 || a.K < 128 * RW || a.log2g < 5 || a.log2g > 7 || affine % (256u >> a.log2g)) return hipErrorInvalidValue;
  if (!rows_start_evenly(a, bits))
    if (const hipError_t e = launch_qgemm_slab(a, bits, bf16, s); e != hipErrorInvalidValue) return e;
  return bits == 2 ? launch_rows<2>(a, bf16, s) : bits == 3 ? launch_rows<3>(a, bf16, s) : bits == 4 ? launch_rows<4>(a, bf16, s) : hipErrorInvalidValue;
}

// Where products of 33 to 4096 rows are faster as groups of up to 32 on the slab kernel than as tiles of dequantised weights (up to 64 rows: than on the other few-row kernels;
// from 1024 on: than by a 16-bit image).  Both grow with their tiles; here a tile of 16 outputs x 32 rows takes a CU 0.5 to 2.3 us, by the length of the contraction and by how dear
// the fields and scales are to take apart, behind a start of 5 us, there the chip is filled by tiles of 64 rows and more.  So the line is a number of tiles a CU.  There | here, us:
//   33 rows 4096 x 4096, 4 bits, group 128 14.8 | 8.6, 3 bits, group 64 19.1 | 9.3; 8192 x 3072 23.8 | 9.0, 24.2 | 10.9; 14336 x 4096 33.9 | 14.7, group 32 50 | 21
//   200 rows 1024 x 4096 18.6 | 8.6; 2048 x 2048 19.5 | 7.2; 4096 x 4096 28.5 | 16.3, 3 bits, group 64 29.8 | 20.8, 4 bits, group 32 29.4 | 23.6; 700 x 1280 15.2 | 5.5
//   K from 3072 on, groups of 64 and 128, 32 tiles a CU: 1000 rows 4096 x 4096 77.5 | 60.1, 512 8192 x 3072 60.0 | 49.3; more: 700 8192 x 3072 63.8 | 71.1, 450 11008 x 4096 79 | 92
//   shorter: 16 tiles 255 rows 8192 x 1536 28.8 | 19.6 to 21.5, 32 tiles 36.6 | 36.6 to 39.3; K 1152, 12 to 16 tiles 18.6 | 17.0 to 19.4, 28 tiles 30 | 33 to 38
//   K 256 and 768, 16 tiles: 100 rows of 16384 17.3 | 10.3 to 15.4, 20.4 | 12.9 to 20.0; 32 tiles 16.6 | 19.1 to 28.9, 24.6 | 24.6 to 38.1
//   3 bits, group 64, 16 tiles: 512 rows 4096 x 4096 41.5 | 39.3, 1000 2048 x 2048 32.8 | 25.7; 19 to 24 tiles 52 | 54, 55 | 67; K 1152, 12 tiles 18.6 | 20.8
//   groups of 32: 8 tiles 128 rows 8192 x 3072 27.6 | 21.1, 65 11008 x 4096 33.2 | 33.3; 10 tiles 36.6 | 38.2; 3 bits, 5 tiles 29.5 | 27.8, 8 tiles 30.3 | 32.3
//   from 1024 rows on, where few outputs leave the image's tiles few: 1024 rows 1024 x 4096 (8 tiles) 26.3 | 21.3, 2000 200 x 3072 (3) 24.7 | 13.2; 1500 1024 x 4096 (12) 31.5 | 33.4;
//   by an image that is there already, 4 bits, group 128 and 3 bits, group 64: 1024 rows 1024 x 4096 26.5 | 21.6, 25.9 | 25.4; 1024 x 1024 18.6 | 9.0, 18.6 | 10.8; 1024 x 256 9.8 |
//   5.6, 9.8 | 6.9; 4096 rows 256 x 4096 26.2 | 21.1, 25.8 | 25.0; 64 x 4096, group 32, 23.3 | 15.8, 3 bits 23.3 | 23.4
static bool groups_win(int64_t M, int N, int K, int bits, int log2g) {
  const int64_t groups = (M + 31) / 32, tiles = (N + 15) / 16;
  const int dear = log2g == 5 ? (bits == 3 ? 5 : 8) : bits == 3 && log2g == 6 ? (K >= 2048 ? 16 : 8) : K >= 3072 ? 32 : K >= 1536 ? 16 : 8;
  const int a_cu = M >= 1024 ? (log2g == 5 ? 5 : 8) : K < 1024 && (bits != 3 || log2g != 5) ? 16 : dear;
  return groups <= 2 || groups * tiles <= 256 * a_cu;
}

}  // namespace gbx

static bool groups_force_generic() {
  static const bool force = gbx::env_switch("GBX_FORCE_GENERIC") != 0;
  return force;
}

// Products of 33 to 4096 rows as groups of up to 32 that the slab kernel takes side by side, where that is the faster form (`always`: wherever it can).  1: not a call for it,
// nothing was launched.  For this package's own Python layer; not part of the public header.
extern "C" int gbx_qlinear_groups_win(int64_t M, int32_t N, int32_t K, int32_t bits, int32_t group_size) {
  return M >= 33 && M <= gbx::SLAB_ROWS && N >= 1 && K >= 128 && K <= 4096 && K % 128 == 0 && bits >= 2 && bits <= 4 && (group_size == 32 || group_size == 64 || group_size == 128) &&
         gbx::groups_win(M, N, K, bits, group_size == 32 ? 5 : group_size == 64 ? 6 : 7);
}
extern "C" int gbx_qlinear_groups(const void* x, const uint32_t* qweight, const void* scales, const void* zeros, const void* bias, void* y, int64_t M, int32_t N, int32_t K,
                                  int32_t bits, int32_t group_size, int32_t act_dtype, int32_t always, void* hip_stream) {
  if (!x || !qweight || !scales || !zeros || !y || M < 33 || M > gbx::SLAB_ROWS || N < 1 || K < 128 || K > 4096 || K % 128 || bits < 2 || bits > 4 || (group_size != 32 && group_size != 64 && group_size != 128) ||
      (act_dtype != 0 && act_dtype != 1) || reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(qweight) % 16)
    return 1;
  gbx::MfmaArgs a{};
  a.x = static_cast<const unsigned short*>(x);
  a.qweight = qweight; a.scales = static_cast<const unsigned short*>(scales); a.zeros = static_cast<const unsigned short*>(zeros);
  a.bias = static_cast<const unsigned short*>(bias); a.y = static_cast<unsigned short*>(y);
  a.M = static_cast<int>(M); a.N = N; a.K = K; a.log2g = group_size == 32 ? 5 : group_size == 64 ? 6 : 7;
  if (groups_force_generic() || (!always && !gbx::groups_win(M, N, K, bits, a.log2g))) return 1;
  const hipError_t e = gbx::launch_qgemm_slab(a, bits, act_dtype == 1, static_cast<hipStream_t>(hip_stream));
  return e == hipSuccess ? 0 : e == hipErrorInvalidValue ? 1 : 2;
}

// The same for 33 to 64 rows of two or three layers of one input (q, k, v): one launch, with the sums of a call per layer (from 65 rows on every layer is a call).  Split contraction
// of dequantised weights | here, us, 33 and 64 rows: 4096, 512 and 512 x 2048, 4 bits, group 128 9.8 9.8 | 6.0 6.3, 3 bits, group 64 12.6 12.9 | 7.0 7.5; 2048, 1024 and 1024 x 1024,
// 2 bits 8.1 8.5 | 4.1 4.3; three of 4096 x 4096, 4 bits 32.7 30.5 | 22.5 22.9; two of 12288 x 4096, 2 bits, in two passes of the batch kernel 22.0 25.6 | 23.0 23.7.
extern "C" int gbx_qlinear_groups_multi(const void* x, int32_t nseg, const void* const* qweight, const void* const* scales, const void* const* zeros, const void* const* bias,
                                        void* const* y, const int32_t* N, int64_t M, int32_t K, int32_t bits, int32_t group_size, int32_t act_dtype, void* hip_stream) {
  if (!x || nseg < 2 || nseg > 3 || M < 33 || M > 64 || K < 128 || K > 4096 || K % 128 || bits < 2 || bits > 4 || (group_size != 32 && group_size != 64 && group_size != 128) ||
      (act_dtype != 0 && act_dtype != 1) || reinterpret_cast<uintptr_t>(x) % 16 || groups_force_generic())
    return 1;
  gbx::MfmaArgs a{};
  a.x = static_cast<const unsigned short*>(x);
  a.M = static_cast<int>(M); a.N = N[0]; a.K = K; a.log2g = group_size == 32 ? 5 : group_size == 64 ? 6 : 7; a.nseg = nseg;
  for (int g = 0; g < nseg; ++g) {
    if (!qweight[g] || !scales[g] || !zeros[g] || !y[g] || N[g] < 1 || reinterpret_cast<uintptr_t>(qweight[g]) % 16) return 1;
    const auto half = [](const void* p) { return static_cast<const unsigned short*>(p); };
    const auto w = static_cast<const uint32_t*>(qweight[g]);
    a.n_seg[g] = N[g];
    if (g == 0) {
      a.qweight = w; a.scales = half(scales[0]); a.zeros = half(zeros[0]); a.bias = half(bias[0]); a.y = static_cast<unsigned short*>(y[0]);
    } else {
      a.qweight_x[g - 1] = w; a.scales_x[g - 1] = half(scales[g]); a.zeros_x[g - 1] = half(zeros[g]); a.bias_x[g - 1] = half(bias[g]); a.y_x[g - 1] = static_cast<unsigned short*>(y[g]);
    }
  }
  const hipError_t e = gbx::launch_qgemm_slab(a, bits, act_dtype == 1, static_cast<hipStream_t>(hip_stream));
  return e == hipSuccess ? 0 : e == hipErrorInvalidValue ? 1 : 2;
}
