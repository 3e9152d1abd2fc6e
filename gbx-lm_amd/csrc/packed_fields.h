// GBA-packed weights as matrix-core operands without expanding them: a field ORed under the exponent of 128.0 (bf16) or 1024.0 (fp16) IS the number C + q.
// A chunk is 128 values of the contraction in 4 steps of 16x16x32 products; inside it the order of k is free as long as both operands agree: step t of
// lane quarter f multiplies octet o(t, f) of the row, the one that lets a lane read its packed words of a group in one piece, in the pair order
// in which fields leave a word ((j, j + 8) of 16 fields of 2 bits, (j, j + 4) of 8 of 4 bits, (2 j, 2 j + 1) of 3 bits).
#pragma once
#include "mfma_common.h"

namespace gbx {

typedef unsigned packed_x2 __attribute__((ext_vector_type(2)));
typedef unsigned packed_x4 __attribute__((ext_vector_type(4)));

// A lane's four octets of a chunk of activations in the order in which fields leave a word.
template <int BITS, int GRP>
__device__ __forceinline__ void packed_order(packed_x4 (&x)[4]) {
  constexpr unsigned LO = 0x05040100u, HI = 0x07060302u;
  if constexpr (BITS == 4 || (BITS == 2 && GRP == 32)) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const packed_x4 v = x[t];
      x[t] = packed_x4{__builtin_amdgcn_perm(v.z, v.x, LO), __builtin_amdgcn_perm(v.z, v.x, HI), __builtin_amdgcn_perm(v.w, v.y, LO), __builtin_amdgcn_perm(v.w, v.y, HI)};
    }
  } else if constexpr (BITS == 2) {                        // two steps share a word
#pragma unroll
    for (int t = 0; t < 4; t += 2) {
      const packed_x4 l = x[t], h = x[t + 1];
      x[t] = packed_x4{__builtin_amdgcn_perm(h.x, l.x, LO), __builtin_amdgcn_perm(h.x, l.x, HI), __builtin_amdgcn_perm(h.y, l.y, LO), __builtin_amdgcn_perm(h.y, l.y, HI)};
      x[t + 1] = packed_x4{__builtin_amdgcn_perm(h.z, l.z, LO), __builtin_amdgcn_perm(h.z, l.z, HI), __builtin_amdgcn_perm(h.w, l.w, LO), __builtin_amdgcn_perm(h.w, l.w, HI)};
    }
  }
}

template <int BITS, int GRP, bool BF16, int TILES = 4>
struct Packed {
  static constexpr int NF = 128 / GRP;                     // groups per chunk
  static constexpr int SPG = 4 / NF;                       // product steps per group
  static constexpr int WPC = 4 * BITS;                     // packed words per row and chunk
  static constexpr int RAW = BITS == 4 ? 4 : BITS == 3 ? (GRP == 128 ? 3 : GRP == 64 ? 4 : 8) : (GRP == 32 ? 4 : 2);
  static constexpr unsigned MAGIC = BF16 ? 0x43004300u : 0x64006400u;
  static constexpr float C = BF16 ? 128.f : 1024.f;
  static constexpr unsigned MASK = BITS == 2 ? 0x00030003u : BITS == 3 ? 0x00070007u : 0x000F000Fu;

  unsigned raw[TILES][RAW];                                // per row tile: the lane's packed words of the chunk
  unsigned short sc[TILES][NF], ze[TILES][NF];

  // octet of step t and lane quarter f: f owns GRP / 4 neighbours of every group
  static __device__ __forceinline__ int step_of(int o) { return GRP == 128 ? (o & 3) : GRP == 64 ? (o >> 3) * 2 + (o & 1) : o >> 2; }
  static __device__ __forceinline__ int quarter_of(int o) { return GRP == 128 ? o >> 2 : GRP == 64 ? (o & 7) >> 1 : o & 3; }

  __device__ __forceinline__ void load(int i, const uint32_t* p, int f) {      // p: the chunk's words of the row
    if constexpr (BITS == 4 && GRP == 128) {
      const packed_x4 v = *reinterpret_cast<const packed_x4*>(p + 4 * f);
      raw[i][0] = v.x; raw[i][1] = v.y; raw[i][2] = v.z; raw[i][3] = v.w;
    } else if constexpr (BITS == 4 && GRP == 64) {
      const packed_x2 a = *reinterpret_cast<const packed_x2*>(p + 2 * f), b = *reinterpret_cast<const packed_x2*>(p + 8 + 2 * f);
      raw[i][0] = a.x; raw[i][1] = a.y; raw[i][2] = b.x; raw[i][3] = b.y;
    } else if constexpr (BITS == 4) {
#pragma unroll
      for (int t = 0; t < 4; ++t) raw[i][t] = p[4 * t + f];
    } else if constexpr (BITS == 2 && GRP == 128) {
      const packed_x2 a = *reinterpret_cast<const packed_x2*>(p + 2 * f);
      raw[i][0] = a.x; raw[i][1] = a.y;
    } else if constexpr (BITS == 2 && GRP == 64) {
      raw[i][0] = p[f]; raw[i][1] = p[4 + f];
    } else if constexpr (BITS == 2) {
#pragma unroll
      for (int t = 0; t < 4; ++t) raw[i][t] = p[2 * t + (f >> 1)];
    } else if constexpr (GRP == 128) {
#pragma unroll
      for (int q = 0; q < 3; ++q) raw[i][q] = p[3 * f + q];
    } else if constexpr (GRP == 64) {                      // 48 bits from bit 48 f (+ 192): words 3 f / 2 and the next
      const int a = (3 * f) >> 1;
      raw[i][0] = p[a]; raw[i][1] = p[a + 1]; raw[i][2] = p[6 + a]; raw[i][3] = p[7 + a];
    } else {                                               // 24 bits from bit 96 t + 24 f
      const int a = (3 * f) >> 2, b = min(a + 1, 2);
#pragma unroll
      for (int t = 0; t < 4; ++t) { raw[i][2 * t] = p[3 * t + a]; raw[i][2 * t + 1] = p[3 * t + b]; }
    }
  }
  // the same words through a buffer: `at` the first byte of the lane's row plus lane_byte(f), `chunk` the chunk's first byte in the row (uniform)
  static __device__ __forceinline__ int lane_byte(int f) {
    return BITS == 4 ? (GRP == 128 ? 16 : GRP == 64 ? 8 : 4) * f
         : BITS == 2 ? (GRP == 128 ? 8 * f : GRP == 64 ? 4 * f : 4 * (f >> 1))
                     : (GRP == 128 ? 12 * f : GRP == 64 ? 4 * ((3 * f) >> 1) : 4 * ((3 * f) >> 2));
  }
  __device__ __forceinline__ void load_buffer(int i, __amdgpu_buffer_rsrc_t r, int at, int chunk) {
    auto one = [&](int byte) { return __builtin_amdgcn_raw_buffer_load_b32(r, at + byte, chunk, 0); };
    auto two = [&](int byte, int q) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, at + byte, chunk, 0);
      raw[i][q] = v[0]; raw[i][q + 1] = v[1];
    };
    if constexpr (BITS == 4 && GRP == 128) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, at, chunk, 0);
#pragma unroll
      for (int q = 0; q < 4; ++q) raw[i][q] = v[q];
    } else if constexpr (BITS == 4 && GRP == 64) {
      two(0, 0); two(32, 2);
    } else if constexpr (BITS == 4) {
#pragma unroll
      for (int t = 0; t < 4; ++t) raw[i][t] = one(16 * t);
    } else if constexpr (BITS == 2 && GRP == 128) {
      two(0, 0);
    } else if constexpr (BITS == 2 && GRP == 64) {
      raw[i][0] = one(0); raw[i][1] = one(16);
    } else if constexpr (BITS == 2) {
#pragma unroll
      for (int t = 0; t < 4; ++t) raw[i][t] = one(8 * t);
    } else if constexpr (GRP == 128) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b96(r, at, chunk, 0);
#pragma unroll
      for (int q = 0; q < 3; ++q) raw[i][q] = v[q];
    } else if constexpr (GRP == 64) {
      two(0, 0); two(24, 2);
    } else {                                               // (quarter 3 ends with its first word: the second is the next row's, and nothing of it is used)
#pragma unroll
      for (int t = 0; t < 4; ++t) two(12 * t, 2 * t);
    }
  }
  __device__ __forceinline__ void load_affine_buffer(int i, __amdgpu_buffer_rsrc_t rs, __amdgpu_buffer_rsrc_t rz, int at, int first) {
    if constexpr (NF == 1) {
      sc[i][0] = __builtin_amdgcn_raw_buffer_load_b16(rs, at, first, 0); ze[i][0] = __builtin_amdgcn_raw_buffer_load_b16(rz, at, first, 0);
    } else if constexpr (NF == 2) {
      const unsigned a = __builtin_amdgcn_raw_buffer_load_b32(rs, at, first, 0), b = __builtin_amdgcn_raw_buffer_load_b32(rz, at, first, 0);
      sc[i][0] = a & 0xFFFF; sc[i][1] = a >> 16; ze[i][0] = b & 0xFFFF; ze[i][1] = b >> 16;
    } else {
      const auto a = __builtin_amdgcn_raw_buffer_load_b64(rs, at, first, 0), b = __builtin_amdgcn_raw_buffer_load_b64(rz, at, first, 0);
      sc[i][0] = a[0] & 0xFFFF; sc[i][1] = a[0] >> 16; sc[i][2] = a[1] & 0xFFFF; sc[i][3] = a[1] >> 16;
      ze[i][0] = b[0] & 0xFFFF; ze[i][1] = b[0] >> 16; ze[i][2] = b[1] & 0xFFFF; ze[i][3] = b[1] >> 16;
    }
  }
  __device__ __forceinline__ void load_affine(int i, const unsigned short* sp, const unsigned short* zp) {
    if constexpr (NF == 1) {
      sc[i][0] = *sp; ze[i][0] = *zp;
    } else if constexpr (NF == 2) {
      const unsigned a = *reinterpret_cast<const unsigned*>(sp), b = *reinterpret_cast<const unsigned*>(zp);
      sc[i][0] = a & 0xFFFF; sc[i][1] = a >> 16; ze[i][0] = b & 0xFFFF; ze[i][1] = b >> 16;
    } else {
      const packed_x2 a = *reinterpret_cast<const packed_x2*>(sp), b = *reinterpret_cast<const packed_x2*>(zp);
      sc[i][0] = a.x & 0xFFFF; sc[i][1] = a.x >> 16; sc[i][2] = a.y & 0xFFFF; sc[i][3] = a.y >> 16;
      ze[i][0] = b.x & 0xFFFF; ze[i][1] = b.x >> 16; ze[i][2] = b.y & 0xFFFF; ze[i][3] = b.y >> 16;
    }
  }
  // the eight operands C + q of step t (compile-time) of row tile i, in the order of the stored activations.  `mask` and `magic`: MASK and MAGIC, from a
  // caller that holds them in registers (one v_and_or_b32 a dword takes no literal: from constants the compiler makes two instructions)
  __device__ __forceinline__ packed_x4 operand(int i, int t, int f, unsigned mask = MASK, unsigned magic = MAGIC) const {
    packed_x4 r;
    if constexpr (BITS == 4) {
      const unsigned w = raw[i][t];
      r.x = (w & mask) | magic; r.y = ((w >> 4) & mask) | magic; r.z = ((w >> 8) & mask) | magic; r.w = ((w >> 12) & mask) | magic;
    } else if constexpr (BITS == 2) {
      const unsigned w = GRP == 32 ? raw[i][t] >> (8 * (f & 1)) : raw[i][t >> 1] >> (8 * (t & 1));
      r.x = (w & mask) | magic; r.y = ((w >> 2) & mask) | magic; r.z = ((w >> 4) & mask) | magic; r.w = ((w >> 6) & mask) | magic;
    } else {
      unsigned w;                                          // the octet's 24 bits from bit 0
      if constexpr (GRP == 128) {
        const int b0 = 24 * t, a = b0 >> 5;
        w = (b0 & 31) == 0 ? raw[i][a] : __builtin_amdgcn_alignbit(raw[i][a + 1 < 3 ? a + 1 : 2], raw[i][a], b0 & 31);
      } else if constexpr (GRP == 64) {
        const unsigned lo = raw[i][2 * (t >> 1)], hi = raw[i][2 * (t >> 1) + 1];
        const int sh = 16 * (f & 1);                       // (48 f mod 32)
        w = (t & 1) == 0 ? __builtin_amdgcn_alignbit(hi, lo, sh) : sh ? hi >> 8 : __builtin_amdgcn_alignbit(hi, lo, 24);
      } else {
        w = __builtin_amdgcn_alignbit(raw[i][2 * t + 1], raw[i][2 * t], (24 * f) & 31);
      }
      unsigned v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const unsigned q = (w >> (6 * j)) & 0x3F;
        v[j] = ((q | (q << 13)) & mask) | magic;
      }
      r.x = v[0]; r.y = v[1]; r.z = v[2]; r.w = v[3];
    }
    return r;
  }
};

// sum_k x[k] (s q + z), weights rounded to the activation type as the dequantising kernels have them: for the sums that the form above leaves without a
// finite number.  An infinite activation meets C + q and -C s as infinity minus infinity where its product with the weight is an infinity; one near the
// largest of its type overflows in C + q alone.  One output a thread; a sum that is no number is final.
template <int BITS, int GRP, bool BF16>
__device__ __forceinline__ float expanded_dot(const unsigned short* __restrict__ x, const uint32_t* __restrict__ w, const unsigned short* __restrict__ s,
                                              const unsigned short* __restrict__ z, int K) {
  float acc = 0.f;
#pragma unroll 1
  for (int k = 0; k < K && acc == acc; k += 32) {
    const float sf = act_to_f32<BF16>(s[k / GRP]), zf = act_to_f32<BF16>(z[k / GRP]);
#pragma unroll 8
    for (int j = k; j < k + 32; ++j) {
      const float v = act_to_f32<BF16>(f32_to_act<BF16>(fmaf(sf, static_cast<float>(field_of_row<BITS>(w, j)), zf)));
      acc = fmaf(act_to_f32<BF16>(x[j]), v, acc);
    }
  }
  return acc;
}

}  // namespace gbx
