// Grouped matrix-core products of routed experts for bf16 prompt portions (mechanism: mixers_moe.hip).
//
// 1. expert_sort_kernel: the step's (row, choice) pairs counted and bucketed by expert on the device (one workgroup, LDS counters):
//    offsets[E + 1], the pair ids in expert order, and the table of row tiles (expert, first pair) the two products walk.  Nothing
//    returns to the host.
// 2. expert_group_kernel, first products: act[p] = silu(gate_e h) * (up_e h) (or another form) for the pairs of expert e, 256 pairs x 128 hidden
//    channels per workgroup (256 channels where experts have no gate);
// 3. expert_group_kernel<EXPERT_DOWN>: y[pair] = down_e act[p], 256 pairs x 256 output channels per workgroup.
// Products are computed swapped -- C^T[channel, pair] = mfma(weight rows, activation rows) -- so a lane ends up with four consecutive
// channels of one pair (8-byte stores) and the gate / up pair of a channel sits in the same lane for the activation.
// What bounds it: a few hundred pairs per expert, so the weights are a stream of their own (1.2 GB at 128 experts of 3 x 2048 x 768: 0.24 ms)
// beside about as much matrix-core work; both operands therefore go memory -> LDS by DMA, stages of 64 elements, two of activations and three of
// weights (which come from memory, two stages ahead; with two of either, one ahead), and a weight row is fetched once per 256 pairs.  Eight waves, a wave 128 pairs x 64 weight rows (16 x 16 x 32 products); four phases a stage, two wave groups
// a barrier apart, so that one group multiplies while the other reads fragments and issues requests.  Stages of 64 elements, because a row
// piece is then a whole 128-byte line: 256 x 128 tiles with stages of 32 elements and two workgroups per CU spent their time on twice the L2
// requests (536 us for the first line below).  A tile is as high as its expert's pairs need, in steps of 64 (32 NR).
// Measured (us, first + second products with the sort, uniform choices, mean over four places of the weights in memory, which move these times by up to a tenth;
// two stages of weights, all from the contraction's start -> as it is now, in turn on one card):
//   27 848 pairs, 128 experts, 2048 x 768 gated:  399 -> 395 (665 TFLOP/s, 3.1 TB/s of weights)
//   18 128 pairs of the same:                     337 -> 320 (3.8 TB/s);  2 048 pairs: 262 -> 232 (5.2 TB/s)
//   16 384 pairs,  64 experts, 2048 x 2048, no gate: 421 -> 400;  2 000 pairs: 274 -> 202.  At 16 384 the weights' way from memory is a factor (one expert's for all: 150 less) and
//   the results' (kept back: 75 less), which tiles of one round write at the same time
//    8 192 pairs,   8 experts, 4096 x 2048 gated: 473 -> 480 (860 TFLOP/s): the one form that the walk of the contraction costs, by 1 %
// The table keeps a lower tile beside its expert's others.  By falling height, so that the last round is short, tiles read their weights anew: 256 pairs an
// expert 454 us against 410 (64 experts), 531 against 476 (128), 288 pairs 595 against 467.  A stage's lines ordered into L2 before gain nothing; nor does
// it matter how many rows a request spans (256 x 128 B, 64 x 512 B or 32 KB in one piece: 4.4 to 4.7 TB/s).
// An expert's tiles walk the contraction from a stage of their own (expert % stages, so that a pair's sums do not depend on the step's other pairs): rows of
// a power of two of bytes put a column of every row on the same memory channels, and workgroups that started together stayed there together.  All from the
// first stage | this, us: 64 experts of 2 x 2048 x 2048, 2 000 pairs 259 | 202 (5.3 TB/s), 64 of 3 x 2048 x 1024, 6 000 pairs 208 | 185, 128 of 3 x 2048 x
// 768, 2 048 pairs 237 | 232; offsets by column
// block as well lose the activation rows that its workgroups share in L2 (8 experts of 3 x 4096 x 2048, 8 192 pairs 7 % slower).
// The grid is sized for the worst case sum_e ceil(n_e / 256) <= P / 256 + E; surplus workgroups leave at once.
// Steps with few pairs per expert (a batch that decodes) stream weights and little else: expert_skinny_kernel takes tiles of 32 pairs, a
// wave per 32 output channels and no barrier.  A wave moves its own rows -- eight lanes to a row's 128 bytes, so an access touches eight
// cache lines instead of the 64 that loads in fragment order would -- through registers (two chunks in flight) into LDS of its own.
#include <type_traits>
#include "mixers_mfma.h"

namespace gbxm {
namespace {

constexpr int RS = 32;          // pairs per tile of the skinny form
// LDS bytes per row of a chunk; 16-byte column c of row r lies at c ^ ((r / 2) & 7), which meets no bank twice in the 16 lanes of a fragment read and lets
// three gated workgroups share a CU (rows of 144 bytes: two)
constexpr int BROW = 128;
__device__ __forceinline__ int chunk_at(int r, int c) { return r * BROW + ((c ^ (r >> 1)) & 7) * 16; }

// One workgroup; E1 = E + 1 buckets, the last for indices that name no expert.  A pair's place in its bucket is what the counting atomic returns, kept
// in registers; the order then forms in LDS and leaves in whole lines (scattered, a wave's stores take the address unit 64 cycles).  Beyond KEEP
// pairs a thread the order is written in place, the further pairs count their bucket down from its end.
// Bound by LDS atomics and trips to memory on one CU.  Two passes of atomics and scattered stores | this, us: 27 848 pairs of 128 experts 24.6 | 9.5, 16 384 of
// 64 13.5 | 6.5, 256 of 128 4.2 | 4.2, 65 536 of 128 52.5 | 43.7.  Up to FEW pairs a thread a form of their own: the other's code costs a launch 0.7 us.
constexpr int KEEP = 32, FEW = 2;         // pairs a thread keeps; few pairs: straight to their places, and no more code than that (it is read cold)
constexpr int SORT_LDS = (3 * 4097 + 5) * 4 + KEEP * 1024 * 2;           // (E <= 4096)

template <int N>
__global__ __launch_bounds__(1024) void expert_sort_kernel(const int* __restrict__ idx, int* __restrict__ offsets, int* __restrict__ sorted,
                                                          int4* __restrict__ tile_tab, int n_tiles, int rt, int P, int E1) {
  extern __shared__ int sm[];                 // counts [E1] | starts [E1 + 1] | first tile [E1] | tiles | the order, 16 bits a pair
  int* counts = sm;
  int* start = sm + E1;
  int* first = start + E1 + 1;
  unsigned short* order = reinterpret_cast<unsigned short*>(sm + ((3 * E1 + 2 + 3) & ~3));
  constexpr int STEP = N < 8 ? N : 8;
  const bool small = N > FEW && P <= N * 1024;
  const int tid = threadIdx.x;
  auto bucket = [&](int v) { return static_cast<int>(min(static_cast<unsigned>(v), static_cast<unsigned>(E1 - 1))); };
  for (int e = tid; e < E1; e += 1024) counts[e] = 0;
  __syncthreads();
  int kept[N], rank[N];
#pragma unroll
  for (int c = 0; c < N; c += STEP)
    if (c * 1024 < P) {
#pragma unroll
      for (int j = c; j < c + STEP; ++j) kept[j] = bucket(idx[min(j * 1024 + tid, P - 1)]);
#pragma unroll
      for (int j = c; j < c + STEP; ++j) rank[j] = j * 1024 + tid < P ? atomicAdd(&counts[kept[j]], 1) : 0;
    }
  __syncthreads();                             // (every kept pair has its place before a further one is counted: the kept ones come first in their bucket)
  if constexpr (N > FEW) {
    for (int i = N * 1024 + tid; i < P; i += 1024) atomicAdd(&counts[bucket(idx[i])], 1);
    __syncthreads();
  }
  if (tid < 64) {                              // one wave: running sums of pairs and tiles, 64 experts at a time
    int run = 0, tiles = 0;
    for (int e0 = 0; e0 < E1; e0 += 64) {
      const int e = e0 + tid, c = e < E1 ? counts[e] : 0, t = (c + rt - 1) / rt;
      int sc = c, st = t;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int uc = __shfl_up(sc, o, 64), ut = __shfl_up(st, o, 64);
        if (tid >= o) { sc += uc; st += ut; }
      }
      if (e < E1) {
        start[e] = run + sc - c;
        offsets[e] = run + sc - c;
        first[e] = tiles + st - t;
      }
      run += __shfl(sc, 63, 64);
      tiles += __shfl(st, 63, 64);
    }
    if (tid == 0) {
      start[E1] = run;
      offsets[E1] = run;
      offsets[E1 + 1] = tiles;
      first[E1] = tiles;
    }
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < N; c += STEP)
    if (c * 1024 < P)
#pragma unroll
      for (int j = c; j < c + STEP; ++j)
        if (j * 1024 + tid < P) {
          const int at = start[kept[j]] + rank[j];
          if (small) order[at] = j * 1024 + tid;
          else sorted[at] = j * 1024 + tid;
        }
  for (int e = tid; e < E1; e += 1024) {
    const int nt = (counts[e] + rt - 1) / rt;
    for (int t = 0; t < nt; ++t) tile_tab[first[e] + t] = int4{e, start[e] + t * rt, start[e] + min(counts[e], (t + 1) * rt), 0};
  }
  for (int t = first[E1] + tid; t < n_tiles; t += 1024) tile_tab[t] = int4{-1, 0, 0, 0};
  if constexpr (N == FEW) return;
  __syncthreads();
  if (small) {                                 // (whole groups of four: expert_buckets_bytes rounds up to them)
    for (int i = tid * 4; i < P; i += 4096) {
      const u32x2 v = *reinterpret_cast<const u32x2*>(order + i);
      *reinterpret_cast<u32x4*>(sorted + i) = u32x4{v.x & 0xFFFF, v.x >> 16, v.y & 0xFFFF, v.y >> 16};
    }
    return;
  }
  for (int e = tid; e < E1; e += 1024) counts[e] = start[e + 1];
  __syncthreads();
  for (int i = N * 1024 + tid; i < P; i += 1024) sorted[atomicSub(&counts[bucket(idx[i])], 1) - 1] = i;
}

// (the gated activations are forms of their own: a tile's epilogue repeats its activation a hundred times over)
enum { EXPERT_DOWN, EXPERT_UP, EXPERT_SILU, EXPERT_CLAMPED };

// s_waitcnt: every LDS access done, at most n vector memory accesses outstanding
__device__ __forceinline__ constexpr int lds_and_vmcnt(int n) { return (n & 0xF) | ((n >> 4) << 14) | (0x7 << 4); }

struct GroupArgs {
  const bf16_t* in;            // activation rows [.][C]
  const bf16_t* w;             // [E][N][C], gated: [E][2 N][C]
  const int* offsets;          // expert_buckets' table
  const int* sorted;
  const int4* tile_tab;
  const float* scale;
  bf16_t* out;
  int N, C, E, top, cols;
  float limit;
};

constexpr int GR = 256;                      // pairs per row tile at most
constexpr int GHALF = 128 * 128;             // LDS bytes of a half-tile: 64 elements of 128 rows
constexpr int GSTAGE = 2 * GHALF;            // a stage's activation rows of wave rows 0 | 1, or its weight rows of wave columns 0, 1 | 2, 3
constexpr int GLDS = 5 * GSTAGE;             // two stages of activations, three of weights: all of a CU's LDS
constexpr int GIDS = 256 * 32 * 16;          // behind the results, at the end: the tile's pair ids and factors
constexpr int PAST = -16;                    // byte offset (as unsigned) beyond every buffer: such lanes of a buffer load deliver zeros

// One tile of 32 NR pairs x 256 weight rows.  See the head of the file.
template <int FORM, int NR>
__device__ __forceinline__ void group_tile(const GroupArgs& a, unsigned char* lds, int e, int lo, int hi, int col, int turn) {
  constexpr bool GATED = FORM == EXPERT_SILU || FORM == EXPERT_CLAMPED;
  constexpr int PA = (NR + 3) / 4;                                      // 16-byte activation pieces per thread and half-tile
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wr = wave >> 2, wc = wave & 3;
  const int fr = lane & 15, fk = lane >> 4;
  const int N = a.N, C = a.C, n = (C + 63) >> 6;
  const int r0 = GATED ? col * 128 : col * 256;                         // the tile's first output channel
  // Start-up is one trip to memory after another (units, tile, rows, operands): the weights, which come from farthest away, are asked for first
  int ida[2][PA];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < PA; ++i) {
      const int row = h * 16 * NR + min((tid >> 3) + 64 * i, 16 * NR - 1);
      ida[h][i] = FORM == EXPERT_DOWN ? min(row, hi - lo - 1) : a.sorted[min(lo + row, hi - 1)];
    }
  const int my_id = a.sorted[min(lo + tid, hi - 1)];                    // (of the first 32 NR threads; kept for the end)
  // DMA side: piece p = tid + 512 i of a half-tile is row p / 8, slot p % 8 of its LDS image and holds 16-byte column slot ^ ((row / 2) & 7):
  // every group of 16 lanes that an LDS fragment read serves at a time then meets 16 different bank quads
  const int lcol = ((tid & 7) ^ ((tid >> 4) & 7)) * 16;
  // (down: the rows of a tile are neighbours, their offsets start at the tile; up: anywhere in the step's rows)
  const bf16_t* in0 = FORM == EXPERT_DOWN ? a.in + static_cast<int64_t>(lo) * C : a.in;
  // (the weight rows that a wave fetches lie in one matrix: in a gated tile every wave column has 32 gate rows -- fetched by waves 0 to 3 --
  //  over the up rows of the same channels -- waves 4 to 7; offsets start at the tile's first row)
  const bf16_t* w0 = a.w + (static_cast<int64_t>(e) * (GATED ? 2 : 1) * N + (GATED ? wr * N : 0) + r0) * C;
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(in0), 0, 0x7FFFFFFF, 0x00020000);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(w0), 0, 0x7FFFFFFF, 0x00020000);
  int voa[2][PA], vob[2][2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int b = h * 128 + (tid >> 3) + 64 * i;
      vob[h][i] = min(GATED ? (b >> 6) * 32 + (b & 31) : b, N - 1 - r0) * C * 2 + lcol;
    }
  }
  auto stage_of = [&](int t) { t = min(t, n - 1) + turn; return t < n ? t : t - n; };
  // half-tile h of stage t; past the end the last stage again: every wait counts the same requests
  auto stage_a = [&](int t, int h) {
    const int tc = stage_of(t);
    const bool cut = tc * 64 + 32 == C && lcol >= 64;                   // the second half of a stage that the contraction does not fill
    unsigned char* dst = lds + (t & 1) * GSTAGE + h * GHALF + wave * 1024;
#pragma unroll
    for (int i = 0; i < PA; ++i) __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, GBXM_LDSP(dst + i * 8192), 16, cut ? PAST : voa[h][i], tc * 128, 0, 0);
  };
  auto stage_b = [&](int t, int slot, int h) {
    const int tc = stage_of(t);
    const bool cut = tc * 64 + 32 == C && lcol >= 64;
    unsigned char* dst = lds + (2 + slot) * GSTAGE + h * GHALF + wave * 1024;
#pragma unroll
    for (int i = 0; i < 2; ++i) __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, GBXM_LDSP(dst + i * 8192), 16, cut ? PAST : vob[h][i], tc * 128, 0, 0);
  };
  const int sw = (fr >> 1) & 7, k0 = (fk ^ sw) * 16, k1 = ((4 + fk) ^ sw) * 16;
  const int fa_off = wr * GHALF + fr * 128, fb_off = 2 * GSTAGE + (wc >> 1) * GHALF + ((wc & 1) * 64 + fr) * 128;
  u32x4 fa[NR][2], fb[4][2];
  auto read_a = [&](const unsigned char* buf, int half) {
#pragma unroll
    for (int i = half * (NR / 2); i < (half + 1) * (NR / 2); ++i) {
      fa[i][0] = *reinterpret_cast<const u32x4*>(buf + fa_off + i * 2048 + k0);
      fa[i][1] = *reinterpret_cast<const u32x4*>(buf + fa_off + i * 2048 + k1);
    }
  };
  auto read_b = [&](const unsigned char* buf, int half) {
#pragma unroll
    for (int j = half * 2; j < half * 2 + 2; ++j) {
      fb[j][0] = *reinterpret_cast<const u32x4*>(buf + fb_off + j * 2048 + k0);
      fb[j][1] = *reinterpret_cast<const u32x4*>(buf + fb_off + j * 2048 + k1);
    }
  };
  f32x4v acc[NR][4];
#pragma unroll
  for (int i = 0; i < NR; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4v{0};
  auto quadrant = [&](int ah, int bh) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int i = ah * (NR / 2); i < (ah + 1) * (NR / 2); ++i)
#pragma unroll
      for (int j = bh * 2; j < bh * 2 + 2; ++j) {
        acc[i][j] = mfma_bf16_16(fb[j][0], fa[i][0], acc[i][j]);
        acc[i][j] = mfma_bf16_16(fb[j][1], fa[i][1], acc[i][j]);
      }
    __builtin_amdgcn_s_setprio(0);
  };
  auto bar = [] { asm volatile("s_barrier" ::: "memory"); };
  stage_b(0, 0, 0);
  stage_b(0, 0, 1);
  __builtin_amdgcn_sched_barrier(0);
  const float my_factor = FORM != EXPERT_DOWN && a.scale ? a.scale[my_id] : 1.f;
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < PA; ++i) voa[h][i] = (FORM == EXPERT_DOWN ? ida[h][i] : ida[h][i] / a.top) * C * 2 + lcol;
  stage_a(0, 0);
  stage_a(0, 1);
  stage_b(1, 1, 0);
  stage_b(1, 1, 1);
  stage_a(1, 0);
  stage_a(1, 1);
  __builtin_amdgcn_s_waitcnt(lds_and_vmcnt(4 + 2 * PA));                // stage 0 has landed (this wave's share), stage 1 may fly
  bar();
  if (wr == 1) bar();                                                   // the second wave group runs one barrier interval behind the first
  // The weights of stage t + 2 are asked for before stage t is multiplied, into the place of stage t - 1, the activations of t + 2 -- which other
  // workgroups of the XCD read too -- once stage t is in registers
  for (int t = 0, now = 0, next = 2; t < n; ++t, next = now, now = now == 2 ? 0 : now + 1) {
    const unsigned char *abuf = lds + (t & 1) * GSTAGE, *bbuf = lds + now * GSTAGE;
    read_b(bbuf, 0);
    __builtin_amdgcn_sched_barrier(0);
    read_a(abuf, 0);
    stage_b(t + 2, next, 0);
    bar();
    quadrant(0, 0);
    bar();
    read_b(bbuf, 1);
    __builtin_amdgcn_sched_barrier(0);
    read_a(abuf, 1);
    stage_b(t + 2, next, 1);
    __builtin_amdgcn_s_waitcnt(0xC07F);                                 // lgkmcnt(0): the stage is in registers before the barrier that frees its slots
    bar();
    quadrant(0, 1);
    bar();
    stage_a(t + 2, 0);
    bar();
    quadrant(1, 1);
    bar();
    stage_a(t + 2, 1);
    __builtin_amdgcn_s_waitcnt(lds_and_vmcnt(4 + 2 * PA));              // all of stage t + 1 has landed
    bar();
    quadrant(1, 0);
    bar();
  }
  if (wr == 0) bar();                                                   // the groups' barrier counts match again
  __builtin_amdgcn_s_waitcnt(lds_and_vmcnt(0));                         // no LDS-DMA outlives the workgroup
  bar();                                                                // every wave is past its last fragment: the stages' LDS is free
  int* ids = reinterpret_cast<int*>(lds + GIDS);
  float* factor = reinterpret_cast<float*>(ids + GR);
  if (tid < 32 * NR) {
    ids[tid] = my_id;
    factor[tid] = my_factor;
  }
  __builtin_amdgcn_s_waitcnt(0xC07F);
  bar();
  // The tile's results meet in LDS (16-byte column c of row r at place c ^ (r & 15): neither side meets a bank twice) and leave as whole rows of it
  constexpr int OPC = GATED ? 16 : 32;                                  // 16-byte columns of a row
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int at = wr * 16 * NR + i * 16 + fr;
    const float sc = factor[at];
#pragma unroll
    for (int j = 0; j < (GATED ? 2 : 4); ++j) {
      float v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if constexpr (FORM == EXPERT_DOWN) v[q] = acc[i][j][q];
        else if constexpr (FORM == EXPERT_UP) { const float z = fmaxf(sc * acc[i][j][q], 0.f); v[q] = z * z; }
        else v[q] = glu_act<true>(sc * acc[i][j][q], sc * acc[i][j + 2][q], FORM == EXPERT_SILU ? GBXM_GLU_SILU : GBXM_GLU_CLAMPED_SWISH, a.limit, 1.702f);
      }
      *reinterpret_cast<u32x2*>(lds + (at * OPC + ((wc * (GATED ? 4 : 8) + j * 2 + (fk >> 1)) ^ fr)) * 16 + (fk & 1) * 8) = u32x2{pack2(v[0], v[1]), pack2(v[2], v[3])};
    }
  }
  __builtin_amdgcn_s_waitcnt(0xC07F);
  bar();
  const int oc = tid & (OPC - 1), rows = min(hi - lo, 32 * NR);
  if (r0 + oc * 8 >= N) return;                                         // (N is a multiple of 32)
#pragma unroll
  for (int i = 0; i < NR * OPC / 16; ++i) {
    const int at = i * (512 / OPC) + tid / OPC;
    if (at >= rows) break;
    *reinterpret_cast<u32x4*>(a.out + static_cast<int64_t>(FORM == EXPERT_DOWN ? ids[at] : lo + at) * N + r0 + oc * 8) =
        *reinterpret_cast<const u32x4*>(lds + (at * OPC + (oc ^ (at & 15))) * 16);
  }
}

template <int FORM>
__global__ __launch_bounds__(512) void expert_group_kernel(const GroupArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int u = xcd_unit(a.offsets[a.E + 2] * a.cols);
  if (u < 0) return;                                                    // (workgroup-uniform, as everything that picks the tile)
  const int bt = u / a.cols, col = u % a.cols;
  const int4 tab = a.tile_tab[bt];
  const int e = tab.x, lo = tab.y, hi = tab.z;
  if (e >= a.E) return;                                                 // (pairs without an expert)
  const int turn = e % ((a.C + 63) >> 6);
  switch ((hi - lo + 63) / 64) {
    case 1: group_tile<FORM, 2>(a, lds, e, lo, hi, col, turn); break;
    case 2: group_tile<FORM, 4>(a, lds, e, lo, hi, col, turn); break;
    case 3: group_tile<FORM, 6>(a, lds, e, lo, hi, col, turn); break;
    default: group_tile<FORM, 8>(a, lds, e, lo, hi, col, turn); break;
  }
}

// FORM 0: out[pair] = w_e in[position in expert order] (the down product); 1: out[position] = relu(scale w_e in[row])^2; 2: gate rows over up
// rows and their gated activation.  N output channels, C contraction; both multiples of 32.
enum { SKINNY_DOWN = 0, SKINNY_UP = 1, SKINNY_GATED = 2 };

// A workgroup's row tile and column block, cut from the tiles that exist, and those first: workgroups without work in between put two with work on
// one CU and leave another idle.  The row tiles of one expert, which read the same weights, are neighbours on one XCD.  Few tiles: the XCDs share out all
// units, column block by column block; from 48 tiles on each takes a run of tiles, which loses less to its remainder than to the strides between
// experts.  (Runs cut from the grid | units | runs, us: 8 experts of 3 x 4096 x 2048, 256 pairs 198 | 128 | 174; 64 of 3 x 2048 x 2048, 256 pairs 304 | 341 | 302.)
struct SkinnyUnit { int tile, col; };
__device__ __forceinline__ SkinnyUnit skinny_unit(int tiles, int cols) {
  if (tiles < 48) {
    const int u = xcd_unit(tiles * cols);
    return u < 0 ? SkinnyUnit{-1, 0} : SkinnyUnit{u % tiles, u / tiles};
  }
  const int per = (tiles + 7) / 8, j = blockIdx.x >> 3, tile = (blockIdx.x & 7) * per + j % per, col = j / per;
  return col < cols && tile < tiles ? SkinnyUnit{tile, col} : SkinnyUnit{-1, 0};
}

template <int FORM>
__global__ __launch_bounds__(256) void expert_skinny_kernel(const bf16_t* __restrict__ in, const bf16_t* __restrict__ w, const int* __restrict__ offsets,
                                                           const int* __restrict__ sorted, const int4* __restrict__ tile_tab, const float* __restrict__ scale,
                                                           bf16_t* __restrict__ out, int N, int C, int E, int top, int kind, float limit) {
  constexpr bool TWO = FORM == SKINNY_GATED;
  const SkinnyUnit u = skinny_unit(offsets[E + 2], (N + 127) / 128);
  if (u.tile < 0) return;
  const int4 tab = tile_tab[u.tile];
  const int e = tab.x, lo = tab.y, hi = tab.z;
  if (e >= E) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 31, hb = lane >> 5;
  const int c0 = u.col * 128 + wave * 32;
  if (c0 >= N) return;
  const int row = min(lo + r, hi - 1), pair = sorted[row];
  constexpr int PARTS = TWO ? 3 : 2;                                     // weights (twice), activations
  __shared__ __attribute__((aligned(16))) unsigned char lds[4][PARTS][RS * BROW];
  unsigned char* mine = lds[wave][0];
  // this lane's pieces of a chunk: rows lane / 8 + 8 i, 16 bytes at column piece lane % 8 (a 32-element tail has four column pieces)
  const int mrow = lane >> 3, col = lane & 7;
  // (buffer loads: a lane's place is fixed, the chunk is scalar; the down product's rows are neighbours, the others lie within 2 GB)
  const bf16_t *w0 = w + (static_cast<int64_t>(e) * (TWO ? 2 : 1) * N + c0) * C, *x0 = FORM == SKINNY_DOWN ? in + static_cast<int64_t>(lo) * C : in;
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(w0), 0, 0x7FFFFFFF, 0x00020000);
  const __amdgpu_buffer_rsrc_t ru = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(w0 + static_cast<int64_t>(N) * C), 0, 0x7FFFFFFF, 0x00020000);
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(x0), 0, 0x7FFFFFFF, 0x00020000);
  const int wo = (mrow * C + col * 8) * 2;
  int xo[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int p = min(lo + mrow + 8 * i, hi - 1);
    xo[i] = ((FORM == SKINNY_DOWN ? p - lo : sorted[p] / top) * C + col * 8) * 2;
  }
  f32x16 acc = f32x16{0}, acc2 = f32x16{0};
  struct Pieces { u32x4 v[PARTS][4]; };
  auto load = [&](Pieces& f, int k0, int cols) {
    const int back = col < cols ? 0 : 64;                               // (a piece past the tail repeats one inside it; nobody reads it)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f.v[0][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, wo - back, (8 * i * C + k0) * 2, 0));
      if constexpr (TWO) f.v[1][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ru, wo - back, (8 * i * C + k0) * 2, 0));
      f.v[PARTS - 1][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, xo[i] - back, k0 * 2, 0));
    }
  };
  auto mul = [&](const Pieces& f, auto steps_c) {
    constexpr int S = decltype(steps_c)::value;
    __builtin_amdgcn_wave_barrier();                                    // (a wave's LDS accesses run in program order: its own writes and reads need
#pragma unroll                                                          //  no barrier among waves, only the compiler must keep the order)
    for (int q = 0; q < PARTS; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i) *reinterpret_cast<u32x4*>(mine + q * (RS * BROW) + chunk_at(mrow + 8 * i, col)) = f.v[q][i];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const unsigned char* p = mine + chunk_at(r, hb * S + i);
      const u32x4 x = *reinterpret_cast<const u32x4*>(p + (PARTS - 1) * (RS * BROW));
      acc = mfma_bf16(*reinterpret_cast<const u32x4*>(p), x, acc);
      if constexpr (TWO) acc2 = mfma_bf16(*reinterpret_cast<const u32x4*>(p + RS * BROW), x, acc2);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  };
  const std::integral_constant<int, 4> whole;
  const std::integral_constant<int, 2> half;
  const int full = C / 64;
  if (full) {
    Pieces f0, f1;
    // (column blocks of experts start the contraction at chunks of their own, as the tiles above)
    const int turn = (u.col + e * 5) & ((1 << (31 - __builtin_clz(full))) - 1);
    const auto chunk = [&](int i) { i = min(i, full - 1) + turn; return (i < full ? i : i - full) * 64; };
    load(f0, chunk(0), 8);
    for (int i = 0; i < full; i += 2) {                                 // (the loads past the end repeat the last chunk)
      load(f1, chunk(i + 1), 8);
      mul(f0, whole);
      load(f0, chunk(i + 2), 8);
      if (i + 1 < full) mul(f1, whole);
    }
  }
  if (C % 64) {
    Pieces f;
    load(f, full * 64, 4);
    mul(f, half);
  }
  if (lo + r >= hi) return;
  const float sc = FORM != SKINNY_DOWN && scale ? scale[pair] : 1.f;
  bf16_t* op = out + static_cast<int64_t>(FORM == SKINNY_DOWN ? pair : row) * N + c0 + 4 * hb;
#pragma unroll
  for (int q4 = 0; q4 < 4; ++q4) {
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float z = acc[4 * q4 + i];
      if constexpr (FORM == SKINNY_DOWN) v[i] = z;
      else if constexpr (FORM == SKINNY_UP) { const float p = fmaxf(sc * z, 0.f); v[i] = p * p; }
      else v[i] = glu_act<true>(sc * z, sc * acc2[4 * q4 + i], kind, limit, 1.702f);
    }
    *reinterpret_cast<u32x2*>(op + 8 * q4) = u32x2{pack2(v[0], v[1]), pack2(v[2], v[3])};
  }
}

template <int FORM>
int launch_group(const GroupArgs& g, int tiles, hipStream_t s) {
  static OncePerDevice once;                                            // (a kernel attribute belongs to the device it is set on)
  if (once.pending()) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(expert_group_kernel<FORM>), hipFuncAttributeMaxDynamicSharedMemorySize, GLDS);
    if (e != hipSuccess) return hip_fail(e, "expert_ff (grouped)");
    once.done();
  }
  const int64_t units = static_cast<int64_t>(tiles) * g.cols;
  expert_group_kernel<FORM><<<static_cast<unsigned>((units + 7) / 8 * 8), 512, GLDS, s>>>(g);
  return after_launch("expert_ff (grouped)");
}

size_t align16(size_t n) { return (n + 15) & ~static_cast<size_t>(15); }
constexpr int64_t MIN_PAIRS = 64;         // below this the weight-streaming row kernels read less
// Pairs per expert (on average) up to which the skinny form is taken.  Measured at 4 | 8 | 16 | 64 pairs per expert, skinny against grouped, us:
// 128 experts of 3 x 2048 x 768  215 | 221 | 237 | 383  against 215 | 224 | 228 | 259;  64 of 2 x 2048 x 2048  192 | 202 | 208 | 361  against
// 192 | 195 | 193 | 215;  32 of 3 x 1024 x 512  27 | 27 | 28 | 40  against 30 | 30 | 30 | 38.
constexpr int64_t SKINNY_PAIRS = 8;
// ... and, where the grouped form's first product has at most half a chip of workgroups, each of them a chain over the whole contraction, up to 64, while the skinny form's
// -- one per tile and 128 channels, about half an expert's tile more than the pairs fill -- do not come to more than one a CU of 4 096 channels: every tile reads its
// expert's weights anew.  Skinny | grouped, us: without a gate, 16 experts of 2 x 1024 x 512, 4 | 32 | 64 pairs per expert 18 | 18 | 24 against 27 | 27 | 33; 8 of 2 x 4096 x 2048,
// 16 | 48 | 64 pairs 58 | 74 | 107 against 79 | 85 | 96; 4 of 2 x 4096 x 4096, 16 | 48 | 64 67 | 69 | 120 against 97 | 105 | 121 (the line lies behind 48 in both); 16 of 2 x 2048 x 1792,
// 16 | 32 | 48 43 | 61 | 51 against 51 | 51 | 51 (many experts of one tile and a little, which the line does not see); gated, 4 of 3 x 512 x 2048, 32 | 64 pairs 26 | 27 against 37 | 45.
constexpr int64_t SKINNY_PAIRS_FEW = 64, FEW_GROUPS = 128, FEW_CHANNELS = 256 * 4096;
int rows_of(int64_t P, int E, int K, int F, bool gated) {
  const int64_t groups = (P / GR + E) * (gated ? (F + 127) / 128 : (F + 255) / 256);
  const bool few = groups <= FEW_GROUPS && (P / RS + E / 2) * ((F + 127) / 128) * K <= FEW_CHANNELS;
  return P <= (few ? SKINNY_PAIRS_FEW : SKINNY_PAIRS) * E ? RS : GR;
}


}  // namespace

int64_t expert_tiles(int64_t P, int rows, int E) { return (P / rows + E + 1 + 7) / 8 * 8; }

size_t expert_buckets_bytes(int64_t P, int rows, int E) {
  return align16(sizeof(int) * (E + 3)) + align16(sizeof(int) * P) + align16(sizeof(int4) * expert_tiles(P, rows, E));
}

int expert_buckets(const int* idx, int P, int rows, int E, void* ws, ExpertBuckets* out, hipStream_t s) {
  unsigned char* w = static_cast<unsigned char*>(ws);
  out->tiles = static_cast<int>(expert_tiles(P, rows, E));
  out->offsets = reinterpret_cast<int*>(w);
  w += align16(sizeof(int) * (E + 3));
  out->sorted = reinterpret_cast<int*>(w);
  w += align16(sizeof(int) * P);
  out->tile_tab = reinterpret_cast<int4*>(w);
  static OncePerDevice once;
  if (once.pending()) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(expert_sort_kernel<KEEP>), hipFuncAttributeMaxDynamicSharedMemorySize, SORT_LDS);
    if (e != hipSuccess) return hip_fail(e, "expert buckets");
    once.done();
  }
  const int counters = ((3 * (E + 1) + 2 + 3) & ~3) * 4;
  if (P <= FEW * 1024) expert_sort_kernel<FEW><<<1, 1024, counters, s>>>(idx, out->offsets, out->sorted, out->tile_tab, out->tiles, rows, P, E + 1);
  else expert_sort_kernel<KEEP><<<1, 1024, counters + (P <= KEEP * 1024 ? (P + 3) / 4 * 8 : 0), s>>>(idx, out->offsets, out->sorted, out->tile_tab, out->tiles, rows, P, E + 1);
  return after_launch("expert buckets");
}

size_t expert_grouped_workspace(int64_t T, int K, int F, int E, int top) {
  const int64_t P = T * top;
  if (P < MIN_PAIRS || K % 32 || F % 32 || E > 4096 || P > 0x3fffffff) return 0;
  return expert_buckets_bytes(P, RS, E) + align16(sizeof(bf16_t) * P * F);      // (the form with more tiles)
}

int launch_expert_grouped(const gbxm_expert_args& a, hipStream_t s) {
  // a tile finds its activation rows by 31-bit byte offsets: rows beyond 2 GB are steps of their own (they share nothing but the weights)
  const int64_t most = (static_cast<int64_t>(1) << 31) / (2 * static_cast<int64_t>(a.K)) - 1;
  if (a.act == GBXM_BF16 && a.K % 32 == 0 && a.T > most && most > 0) {
    for (int64_t t = 0; t < a.T; t += most) {
      gbxm_expert_args part = a;
      part.T = a.T - t < most ? a.T - t : most;
      part.h = static_cast<const bf16_t*>(a.h) + t * a.K;
      part.y = static_cast<bf16_t*>(a.y) + t * a.top * a.K;
      part.idx = a.idx + t * a.top;
      part.scale = a.scale ? a.scale + t * a.top : nullptr;
      const int rc = launch_expert_grouped(part, s);
      if (rc != GBXM_OK) return rc;
    }
    return GBXM_OK;
  }
  const int K = a.K, F = a.F, E = a.E, top = a.top;
  const size_t need = expert_grouped_workspace(a.T, K, F, E, top);
  if (need == 0) return GBXM_ERR_UNSUPPORTED;
  if (a.ws_bytes < need) return fail(GBXM_ERR_INVALID, "expert_ff: workspace of %zu bytes, %zu needed", a.ws_bytes, need);
  if ((reinterpret_cast<uintptr_t>(a.h) | reinterpret_cast<uintptr_t>(a.first) | reinterpret_cast<uintptr_t>(a.down) | reinterpret_cast<uintptr_t>(a.y) |
       reinterpret_cast<uintptr_t>(a.ws)) % 16)
    return GBXM_ERR_UNSUPPORTED;
  const int P = static_cast<int>(a.T * top);
  ExpertBuckets k;
  const bool gated = a.kind != GBXM_EXPERT_RELU2;
  const int rows = rows_of(P, E, K, F, gated);
  int rc = expert_buckets(a.idx, P, rows, E, a.ws, &k, s);
  if (rc != GBXM_OK) return rc;
  const int *offsets = k.offsets, *sorted = k.sorted, tiles = k.tiles;
  const int4* tile_tab = k.tile_tab;
  bf16_t* act = reinterpret_cast<bf16_t*>(static_cast<unsigned char*>(a.ws) + expert_buckets_bytes(P, RS, E));
  const bf16_t* h = static_cast<const bf16_t*>(a.h);
  const bf16_t* first = static_cast<const bf16_t*>(a.first);
  if (rows == RS) {
    const auto grid = [&](int n) { return static_cast<unsigned>((static_cast<int64_t>(tiles) * ((n + 127) / 128) + 7) / 8 * 8); };
    const unsigned up = grid(F), dn = grid(K);
    if (gated) expert_skinny_kernel<SKINNY_GATED><<<up, 256, 0, s>>>(h, first, offsets, sorted, tile_tab, a.scale, act, F, K, E, top, a.kind, a.limit);
    else expert_skinny_kernel<SKINNY_UP><<<up, 256, 0, s>>>(h, first, offsets, sorted, tile_tab, a.scale, act, F, K, E, top, a.kind, a.limit);
    expert_skinny_kernel<SKINNY_DOWN><<<dn, 256, 0, s>>>(act, static_cast<const bf16_t*>(a.down), offsets, sorted, tile_tab, nullptr,
                                                         static_cast<bf16_t*>(a.y), K, F, E, top, a.kind, a.limit);
    return after_launch("expert_ff (skinny groups)");
  }
  GroupArgs g{h, first, offsets, sorted, tile_tab, a.scale, act, F, K, E, top, gated ? (F + 127) / 128 : (F + 255) / 256, a.limit};
  rc = !gated ? launch_group<EXPERT_UP>(g, tiles, s) : a.kind == GBXM_GLU_SILU ? launch_group<EXPERT_SILU>(g, tiles, s) : launch_group<EXPERT_CLAMPED>(g, tiles, s);
  if (rc != GBXM_OK) return rc;
  g = GroupArgs{act, static_cast<const bf16_t*>(a.down), offsets, sorted, tile_tab, nullptr, static_cast<bf16_t*>(a.y), K, F, E, top, (K + 255) / 256, a.limit};
  return launch_group<EXPERT_DOWN>(g, tiles, s);
}

}  // namespace gbxm
