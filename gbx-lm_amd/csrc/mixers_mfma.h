// Matrix-core helpers of libgbx_mixers.so (gfx950: 32x32x16 bf16 MFMA, transposed LDS reads).
#pragma once
#include "mixers_common.h"

namespace gbxm {

typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4v __attribute__((ext_vector_type(4)));
typedef float f32x2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

// C[32 x 32] += A[32 x 16] B[16 x 32]: lane l gives A[l % 32][8 (l / 32) ..+8] and B[8 (l / 32) ..+8][l % 32] and holds
// C[8 (e / 4) + 4 (l / 32) + e % 4][l % 32], e = 0..15.
__device__ __forceinline__ f32x16 mfma_bf16(const u32x4& a, const u32x4& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// C[16 x 16] += A[16 x 32] B[32 x 16]: lane l gives A[l % 16][8 (l / 16) ..+8] and B[8 (l / 16) ..+8][l % 16] and holds
// C[4 (l / 16) + e][l % 16], e = 0..3.
__device__ __forceinline__ f32x4v mfma_bf16_16(const u32x4& a, const u32x4& b, const f32x4v& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// two fp32 -> one packed bf16 pair, round to nearest even
__device__ __forceinline__ unsigned pack2(float a, float b) {
  f32x2v v; v.x = a; v.y = b;
  return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2v));
}
// ds_read_b64_tr_b16: per 16-lane group a 4-row x 16-column block of 16-bit elements, delivered column-major (lane i of the group:
// column i, rows 0..3); lane 4q + p of the group supplies the address of row q, columns 4p .. 4p+3.  EXEC must be full.
__device__ __forceinline__ u32x2 lds_read_tr(const unsigned char* p) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (s16x4 __attribute__((address_space(3)))*)(__attribute__((address_space(3))) unsigned char*)p));
}

// LDS as the destination of a buffer load
#define GBXM_LDSP(p) ((__attribute__((address_space(3))) void*)(p))

// How the 256 threads of a group of waves carry the rows of a key or value tile, D channels each, in pieces of 16 bytes: `LANES` neighbouring threads a row, `PER`
// pieces of it each, `ROWS` rows at a time; or, where a row's pieces do not fall into eights, piece after piece.
template <int D, int KT> struct RowPieces {
  static constexpr int C = D / 8, LANES = C % 16 == 0 ? 16 : C % 8 == 0 ? 8 : 4, PER = C / LANES, ROWS = 256 / LANES;
  static constexpr bool LINEAR = C > 4 && LANES == 4;
  static constexpr int N = LINEAR ? (KT * C + 255) / 256 : PER * ((KT + ROWS - 1) / ROWS);
  __device__ static int row(int tid, int i) { return LINEAR ? (tid + 256 * i) / C : tid / LANES + i / PER * ROWS; }
  __device__ static int piece(int tid, int i) { return LINEAR ? (tid + 256 * i) % C : tid % LANES + i % PER * LANES; }
  __device__ static bool used(int tid, int i) { return (LINEAR ? KT * C % 256 == 0 : KT % ROWS == 0) || row(tid, i) < KT; }
};

// Workgroup ids go round-robin over the 8 XCDs, each with an L2 of its own: every XCD gets a contiguous run of units (row tile, column
// block), so the column blocks of ONE row tile, which read the same activation rows, and the row tiles of one expert, which read the
// same weights, run on one XCD next to each other.  The runs are cut from the units that exist (the sort counted the tiles), not from
// the worst case that the grid is sized for: surplus workgroups would otherwise all stand in the last XCDs' runs.
__device__ __forceinline__ int xcd_unit(int units) {
  const int per = (units + 7) / 8, j = blockIdx.x >> 3, u = (blockIdx.x & 7) * per + j;
  return j < per && u < units ? u : -1;
}

// Pairs (row, choice) bucketed by expert on the device (mixers_moe_mfma.hip): offsets [E + 2] by bucket -- bucket E holds the pairs whose
// index names no expert -- then the number of row tiles; the pair ids in bucket order; per row tile (of at most `rows` pairs) its bucket
// and its first and last + 1 place in that order (surplus tiles: bucket -1).  `tiles` bounds the tiles on the host.  `ws`: expert_buckets_bytes.
struct ExpertBuckets {
  int *offsets, *sorted;
  int4* tile_tab;
  int tiles;
};
size_t expert_buckets_bytes(int64_t P, int rows, int E);
int expert_buckets(const int* idx, int P, int rows, int E, void* ws, ExpertBuckets* out, hipStream_t s);

// Steps with sequences of STATE_CHUNKS_FROM rows and more through the decayed matrix states (mixers_state_mfma.hip).  Workspace 0: not a step for it.
// left->flags: what the launches did, and left the rest of (null: nothing is left).
// One sequence of 70 | 100 | 128 | 200 rows, token by token against chunks, us: delta rule, 8 heads of 64 x 128 14 | 18 | 22 | 33 against 19 | 21 | 19 | 24; 32 of 128 x 128
// 20 | 26 | 34 | 50 against 22 | 24 | 23 | 32.
constexpr int STATE_CHUNKS_FROM = 128;
struct StateArgs;
struct StateChunks;
size_t state_chunks_workspace(int64_t T, int64_t B, int H, int dk, int dv);
int launch_state_chunks(const StateArgs& a, int64_t T, bool delta, void* ws, hipStream_t s, StateChunks* left);

}  // namespace gbxm
