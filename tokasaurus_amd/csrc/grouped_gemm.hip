// Matrix products in which every tile of rows has a weight matrix of its own, on
// v_mfma_f32_16x16x32_bf16: the experts of a mixture (rows sorted by expert) and a matrix a head.
//
//   tk_expert_sort        pairs (token, chosen expert) sorted by expert into slots, every expert's
//                         run of slots filled up to whole tiles of GS_M slots
//   tk_grouped_gemm_bf16  C[c_row(slot), g * c_cols + n] = sum_k W[g][n][k] * A[a_row(slot), g * a_cols + k]
//                         for the slots of every tile, g the tile's group; optionally the gated form
//                         silu(gate) * up of two halves of W[g], or the gated form with clamps
//   tk_expert_sum         per token the weighted sum of its pairs' rows, identity experts, shared expert
//
// Two kernels.  A matrix a head (grouped_gemm_kernel): a wavefront owns GG_TM = 64 rows x 64 outputs: weight rows are the
// first operand of the matrix core, read straight from memory 16 bytes a lane, the rows of A the second; a lane ends up with
// 4 neighbouring outputs of one row.  The next step's operands are asked for before the current step's products.
// Experts (grouped_gemm_staged_kernel): tiles of GS_M = 128 slots x 128 weight rows through local memory, however few slots a
// tile holds (see there); experts of many rows take two such tiles as one of 256 x 256 (grouped_gemm_pairs_kernel).  Sums are 32-bit
// and run over k in ascending steps for every output: a row's result does not depend on which other rows share its tile.
#include <math.h>

#include "gemm_tile.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

#define GG_TM 64
#define GG_WAVES 4

__device__ __forceinline__ bf16x8_t gg_zero8() {
  bf16x8_t z;
#pragma unroll
  for (int e = 0; e < 8; ++e) z[e] = (__bf16)0.f;
  return z;
}

struct GroupedArgs {
  const bf16_t* A;
  int lda;
  const int* a_row;       // [slots] the row of A a slot reads, < 0: an empty slot; null: the slot's own number
  const int* c_row;       // [slots] the row of C a slot writes, < 0: none; null: the slot's own number
  const int* tile_group;  // [tiles] the group of every tile of slots, < 0: an unused tile, and [tiles] the number of used ones, which come
                          // first; null: blockIdx.z, and rows instead of slots
  int a_cols, c_cols;     // (a group a blockIdx.z) columns of A and C that a group is offset by
  const bf16_t* W;        // [groups][N (2 N in the gated form: gate rows, then up rows)][K]
  size_t w_stride;        // elements from one group's matrix to the next
  void* C;
  int ldc;
  int N, K, slots;
  const float* row_scale;  // (gated form) a factor on a slot's sums of gate and up alike, row_scale[scale_row[slot]]; null: none
  const int* scale_row;
  float limit, alpha;  // (gated form) limit > 0: the activation with clamps (clamped_glu of common.h) instead of silu
};
__device__ __forceinline__ float gg_gated(const GroupedArgs& a, float g, float u) {
  return a.limit > 0.f ? clamped_glu<bf16_t>(g, u, a.limit, a.alpha) : silu_mul_bf16(g, u);
}

// NT: blocks of 16 outputs a wavefront; F32: 32-bit output
template <int NT, bool F32>
__global__ __launch_bounds__(GG_WAVES * TK_WAVE) void grouped_gemm_kernel(GroupedArgs a) {
  constexpr int MB = GG_TM / 16;
  const int lane = threadIdx.x & (TK_WAVE - 1), wave = threadIdx.x / TK_WAVE;
  const int tile = blockIdx.x;
  const int g = (int)blockIdx.z;
  const int n0 = (blockIdx.y * GG_WAVES + wave) * NT * 16;
  if (n0 >= a.N) return;
  const int r = lane & 15, q = lane >> 4;
  const bf16_t* Wg = a.W + (size_t)g * a.w_stride;
  const bf16_t* wp[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) wp[t] = Wg + (size_t)min(n0 + t * 16 + r, a.N - 1) * a.K + q * 8;
  const bf16_t* ap[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
    ap[mb] = a.A + (size_t)min(tile * GG_TM + mb * 16 + r, a.slots - 1) * a.lda + (size_t)g * a.a_cols + q * 8;
  f32x4_t acc[NT][MB];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[t][mb] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int steps = (a.K + 31) / 32;
  bf16x8_t w[NT], av[MB];
  auto load = [&](int ks, bf16x8_t (&wv)[NT], bf16x8_t (&xv)[MB]) {
    // a step may reach past K (a multiple of 8): read a valid chunk and zero the weight
    const bool k_ok = ks * 32 + q * 8 < a.K;
    const long off = k_ok ? (long)ks * 32 : -(long)(q * 8);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      wv[t] = *(const bf16x8_t*)(wp[t] + off);
      if (!k_ok) wv[t] = gg_zero8();
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) xv[mb] = *(const bf16x8_t*)(ap[mb] + off);
  };
  load(0, w, av);
  for (int ks = 0; ks < steps; ++ks) {
    bf16x8_t wn[NT], an[MB];
    if (ks + 1 < steps) load(ks + 1, wn, an);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
        acc[t][mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[t], av[mb], acc[t][mb], 0, 0, 0);
    if (ks + 1 < steps) {
#pragma unroll
      for (int t = 0; t < NT; ++t) w[t] = wn[t];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) av[mb] = an[mb];
    }
  }
  // lane: row mb * 16 + r, outputs n0 + t * 16 + 4 q + j
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int row = tile * GG_TM + mb * 16 + r;
    if (row >= a.slots) continue;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int n = n0 + t * 16 + 4 * q;
      const size_t at = (size_t)row * a.ldc + (size_t)g * a.c_cols + n;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (n + j < a.N) {
          if (F32) ((float*)a.C)[at + j] = acc[t][mb][j];
          else ((bf16_t*)a.C)[at + j] = __float2bfloat16(acc[t][mb][j]);
        }
      }
    }
  }
}

// --------------------------------------------------------------------------
// Experts: a workgroup owns GS_M slots x 128 weight rows (in the gated form 64 of
// gate and the 64 of up that belong to them), its four wavefronts 64 x 64 each, on v_mfma_f32_32x32x16_bf16 (1.86 PFLOP/s
// in a loop of nothing else; the 16 x 16 x 32 form 1.23 to 1.57).  Steps of 32 elements of K go straight from memory to
// local memory into GS_STAGES buffers: two steps' rows are on their way while one is multiplied (48 KB a workgroup, three
// workgroups a compute unit; four buffers and two workgroups: 228 against 210 us), with one barrier a step.  16-byte pieces of a row lie exchanged by (row / 4) & 3, made on the
// side of the address, so that any 16 of the 32 rows that the lanes read at a time meet 64 different banks.
// What bounds it is memory: an expert's weights (8 MB for 2 x 1 024 rows of 2 048) pass a die's L2 once for every time that its
// tiles are taken up.  So workgroups come in the order of the runs: up to GS_TILES tiles of one group through all outputs,
// then the next, each die a stretch of that order (the hardware deals workgroups to the eight dies in turn).
// The results leave through local memory, 16 bytes a lane (8 scattered bytes a lane took 40 us of 290).
// Experts of few rows take the same tiles: their products are priced by the weights, which a tile reads once (32 experts of 2 048 x
// 1 024, 403 MB; tokens x 8 chosen, 13 / 64 / 300 tokens: 108 / 110 / 115 us for both products and the sum, 176 / 194 / 317
// with 64 slots a wavefront straight from memory).
// 2 048 tokens x 8 of 32 experts (143 tiles), gate and up: 290 us through registers into two buffers of 64
// elements with tiles taken four at a time whatever their group (634 MB past the L2), 210 us so (474 MB; 343 are needed);
// the loads alone take 180, the products alone 140.
// --------------------------------------------------------------------------
#define GS_M 128
#define GS_K 32
#define GS_STAGES 3
#define GS_DIES 8
#define GS_TILES 8
typedef __attribute__((ext_vector_type(16))) float f32x16_t;

// Tiles in a row before and behind `tile` that belong to its group `g` (both sides' first 64 asked for at once).
__device__ __forceinline__ void gg_run(const int* tile_group, int used, int tile, int& g, int& before, int& behind) {
  const int lane = threadIdx.x & (TK_WAVE - 1);
  int at[2] = {0, 0};
  bool open[2] = {true, true};
  g = tile_group[tile];
  while (open[0] || open[1]) {
    int t[2], v[2];
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      t[side] = side == 0 ? tile - 1 - at[0] - lane : tile + 1 + at[1] + lane;
      v[side] = tile_group[min(max(t[side], 0), used - 1)];
    }
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      if (!open[side]) continue;
      const unsigned long long other = ~__ballot(t[side] >= 0 && t[side] < used && v[side] == g);
      if (other != 0) {
        at[side] += __ffsll(other) - 1;
        open[side] = false;
      } else {
        at[side] += TK_WAVE;
      }
    }
  }
  before = at[0];
  behind = at[1];
}

template <bool GLU>
__global__ __launch_bounds__(256, 3) void grouped_gemm_staged_kernel(GroupedArgs a, int tiles, int n_blocks) {
  extern __shared__ __align__(16) bf16_t rows[];  // [GS_STAGES][128 slots, 128 weight rows][GS_K]; then the results [GS_M][OUT]
  constexpr int OUT = GLU ? 64 : 128;             // outputs of a workgroup
  const int used = a.tile_group[tiles];           // the tiles that hold slots come first
  const int items = used * n_blocks, per = (items + GS_DIES - 1) / GS_DIES;
  const int seq = blockIdx.x / GS_DIES, item = blockIdx.x % GS_DIES * per + seq;
  if (seq >= per || item >= items) return;
  // the run of tiles of one group that the item lies in, and in it the chunk of up to GS_TILES tiles
  const int some = item / n_blocks;
  int g, before, behind;
  gg_run(a.tile_group, used, some, g, before, behind);
  const int chunk = some - before + before / GS_TILES * GS_TILES;  // its first tile
  const int len = min(GS_TILES, some + behind + 1 - chunk);
  const int off = item - chunk * n_blocks;
  const int tile = chunk + off % len;
  const int n0 = off / len * OUT;
  const int lane = threadIdx.x & (TK_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TK_WAVE);
  // A load brings 16 rows of 32 elements; wavefront w brings slots 32 w .. 32 w + 31 and as many weight rows.  Lane l writes
  // piece l % 4 of row l / 4, which holds the row's piece (l % 4) ^ ((row / 4) & 3).
  const int lrow = lane >> 2, piece = (lane & 3) ^ (lane >> 4);
  // what this thread stores at the end: 16-byte pieces of rows, their places in C
  constexpr int PIECES = OUT / 8, PASSES = GS_M * PIECES / 256;
  const int orow = threadIdx.x / PIECES, ocol = threadIdx.x % PIECES * 8;
  const int r = lane & 31, h = lane >> 5;
  const int wm = wave & 1, wn = wave >> 1;
  // (all numbers of rows are asked for before the first is used)
  const int top = a.slots - 1;
  int from[2], crow[PASSES], filled[PASSES], frow[2] = {0, 0};
#pragma unroll
  for (int i = 0; i < 2; ++i) from[i] = tile * GS_M + wave * 32 + i * 16 + lrow;
#pragma unroll
  for (int i = 0; i < PASSES; ++i) crow[i] = filled[i] = tile * GS_M + orow + i * (256 / PIECES);
  if (a.a_row) {
#pragma unroll
    for (int i = 0; i < 2; ++i) from[i] = a.a_row[min(from[i], top)];
#pragma unroll
    for (int i = 0; i < PASSES; ++i) filled[i] = a.a_row[min(filled[i], top)];
  }
  const bool scaled = GLU && a.row_scale;
  if (scaled) {
#pragma unroll
    for (int mb = 0; mb < 2; ++mb) frow[mb] = a.scale_row[min(tile * GS_M + wm * 64 + mb * 32 + r, top)];  // (< 0: an empty slot)
  }
  if (a.c_row) {
#pragma unroll
    for (int i = 0; i < PASSES; ++i) crow[i] = a.c_row[min(crow[i], top)];
  }
  const bf16_t* src[4];  // slots, then weight rows (a row that is not stored may read any)
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = wave * 32 + i * 16 + lrow;
    const int wrow = GLU ? min(n0 + (row & 63), a.N - 1) + (row >= 64 ? a.N : 0) : min(n0 + row, a.N - 1);
    src[2 + i] = a.W + (size_t)g * a.w_stride + (size_t)wrow * a.K + piece * 8;
    src[i] = a.A + (size_t)max(tile * GS_M + row <= top ? from[i] : 0, 0) * a.lda + piece * 8;
  }
  float factor[2] = {1.f, 1.f};
  if (scaled) {
#pragma unroll
    for (int mb = 0; mb < 2; ++mb) factor[mb] = a.row_scale[max(frow[mb], 0)];
  }
#pragma unroll
  for (int i = 0; i < PASSES; ++i)
    if (tile * GS_M + orow + i * (256 / PIECES) > top || filled[i] < 0) crow[i] = -1;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (nothing but the rows' loads is counted from here on)
  const unsigned lds = (unsigned)(uintptr_t)(__attribute__((address_space(3))) bf16_t*)rows;
  const int steps = (a.K + GS_K - 1) / GS_K;
  auto ask = [&](int step) {
    const int at = (step % GS_STAGES * 256 + wave * 32) * GS_K;  // elements
    const size_t k = (size_t)step * GS_K;
    if (step * GS_K + piece * 8 < a.K) {
#pragma unroll
      for (int i = 0; i < 4; ++i) load_to_lds(src[i] + k, lds + (at + ((i >> 1) * 128 + (i & 1) * 16) * GS_K) * 2);
    } else {  // K (a multiple of 8) ends inside the step: zeros behind it (the step's first piece is always there)
#pragma unroll
      for (int i = 0; i < 4; ++i) *(bf16x8_t*)(rows + at + ((i >> 1) * 128 + (i & 1) * 16) * GS_K + lane * 8) = gg_zero8();
    }
  };
  f32x16_t acc[2][2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[t][mb][j] = 0.f;
#pragma unroll
  for (int s = 0; s < GS_STAGES - 1; ++s)
    if (s < steps) ask(s);
#pragma unroll 1
  for (int s = 0; s < steps; ++s) {
    // the step's rows are there when only those of the steps behind it (four loads each) are left, and every wavefront's are
    // behind the barrier; every wavefront is through with the step before then, whose buffer is filled again
    if (s + 1 < steps) asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (s + GS_STAGES - 1 < steps) ask(s + GS_STAGES - 1);
    const bf16_t* sa = rows + (size_t)(s % GS_STAGES) * 256 * GS_K;
    const bf16_t* sw = sa + 128 * GS_K;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      bf16x8_t w[2], x[2];
      const int swz = ((kk * 2 + h) ^ ((r >> 2) & 3)) * 8;
#pragma unroll
      for (int t = 0; t < 2; ++t) w[t] = *(const bf16x8_t*)(sw + ((GLU ? t * 64 + wn * 32 : wn * 64 + t * 32) + r) * GS_K + swz);
#pragma unroll
      for (int mb = 0; mb < 2; ++mb) x[mb] = *(const bf16x8_t*)(sa + (wm * 64 + mb * 32 + r) * GS_K + swz);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) acc[t][mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[t], x[mb], acc[t][mb], 0, 0, 0);
    }
  }
  __syncthreads();
  // A lane holds of slot wm * 64 + mb * 32 + r the outputs 8 (j / 4) + 4 h + j % 4 of a block of 32.  They pass through local
  // memory (a row's 8-byte pieces exchanged by its number) so that a slot's outputs leave 16 bytes a lane, side by side.
#pragma unroll
  for (int mb = 0; mb < 2; ++mb) {
    const int row = wm * 64 + mb * 32 + r;
#pragma unroll
    for (int t = 0; t < (GLU ? 1 : 2); ++t) {
#pragma unroll
      for (int j4 = 0; j4 < 4; ++j4) {
        union { bf16_t v[4]; uint2 raw; } o;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float y = GLU ? gg_gated(a, acc[0][mb][4 * j4 + j] * factor[mb], acc[1][mb][4 * j4 + j] * factor[mb]) : acc[t][mb][4 * j4 + j];
          o.v[j] = __float2bfloat16(y);
        }
        const int unit = (GLU ? wn * 8 : wn * 16 + t * 8) + 2 * j4 + h;  // of 4 outputs
        *(uint2*)(rows + row * OUT + ((unit >> 1) ^ (row & 7)) * 8 + (unit & 1) * 4) = o.raw;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < PASSES; ++i) {
    if (crow[i] < 0) continue;
    const int row = orow + i * (256 / PIECES);
    const uint4 v = *(const uint4*)(rows + row * OUT + ((ocol >> 3) ^ (row & 7)) * 8);
    bf16_t* dst = (bf16_t*)a.C + (size_t)crow[i] * a.ldc + n0 + ocol;
    const int left = a.N - n0 - ocol;
    if (left >= 8 && ((uintptr_t)dst & 15) == 0) {
      *(uint4*)dst = v;
    } else {
      const bf16_t* e = (const bf16_t*)&v;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (j < left) dst[j] = e[j];
    }
  }
}

// Experts of many rows: two neighbouring tiles of a group as one of 256 slots x 256 weight rows (in the gated form 128 of gate and
// 128 of up; gemm_tile.h), the odd last tile of a group in smaller ones in the same launch.  The path from the L2 to a compute
// unit bounds these products, and a tile of 256 x 256 asks for half as many bytes a product.
// us by tiles of 128 x 128 / in pairs, gate and up and down, every expert 3, 4, 5 and 6 tiles: 32 experts of 2,048 x 1,024 147 / 136 and
// 86 / 69, 185 / 141 and 109 / 75, 224 / 190 and 132 / 97, 265 / 202 and 155 / 107; 32 of 2,880 x 2,880 547 / 461 and 300 / 213 to
// 1,060 / 726 and 554 / 355.  Odd tiles as halves of a pair: 140 and 70, 199 and 100 for the first with 3 and 5.  In a launch of
// their own, which reads the experts' weights a second time: 172 and 87, 234 and 118.
template <class S, bool GLU>
__device__ __forceinline__ void wide_tile(const GroupedArgs& a, char* smem, int g, int first, int n0) {
  constexpr int OUT = GLU ? S::BN / 2 : S::BN;
  static_assert(S::BM <= 256 && S::BM * S::BN * 2 + S::BM * 4 <= S::LDS, "");
  const int lane = threadIdx.x & (TK_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TK_WAVE);
  const int wm = wave & 1, wn = wave >> 1, top = a.slots - 1;
  TileLoop<S, GLU> t;
  t.wave = wave;
  t.lds = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  t.a = (const char*)a.A;
  t.w = (const char*)(a.W + (size_t)g * a.w_stride + (size_t)n0 * a.K);
  // (all numbers of rows are asked for before the first is used)
  const int lr = lane >> 3;
  int from[S::LA], frow[2 * S::TM], to = -1;
#pragma unroll
  for (int i = 0; i < S::LA; ++i) {
    const int slot = min(first + wave * (16 * S::TM) + i * 8 + lr, top);
    from[i] = a.a_row ? a.a_row[slot] : slot;
  }
  const int own = first + (int)threadIdx.x;  // of the first BM threads
  if (threadIdx.x < S::BM && own <= top) {
    to = a.c_row ? a.c_row[own] : own;
    if (a.a_row && a.a_row[own] < 0) to = -1;
  }
  float factor[2 * S::TM];
#pragma unroll
  for (int m = 0; m < 2 * S::TM; ++m) factor[m] = 1.f;
  if (GLU && a.row_scale) {
#pragma unroll
    for (int m = 0; m < 2 * S::TM; ++m) frow[m] = a.scale_row[min(first + wm * (32 * S::TM) + m * 16 + (lane & 15), top)];  // (< 0: an empty slot)
#pragma unroll
    for (int m = 0; m < 2 * S::TM; ++m) factor[m] = a.row_scale[max(frow[m], 0)];
  }
#pragma unroll
  for (int i = 0; i < S::LA; ++i)
    t.off[i] = (unsigned)max(from[i], 0) * (unsigned)a.lda * 2 + ((lane & 7) ^ tile_swizzle(i * 8 + lr)) * 16;
#pragma unroll
  for (int i = 0; i < S::LW; ++i) {
    const int row = wave * (16 * S::TN) + i * 8 + lr;  // (a row that is not stored may read any)
    const int wrow = GLU ? min(row % OUT, a.N - 1 - n0) + (row >= OUT ? a.N : 0) : min(row, a.N - 1 - n0);
    t.off[S::LA + i] = (unsigned)wrow * (unsigned)a.K * 2 + ((lane & 7) ^ tile_swizzle(i * 8 + lr)) * 16;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (nothing but the rows' loads is counted from here on)
  t.run(smem, a.K / TILE_K, wm, wn, lane);
  __syncthreads();
  int* dst = (int*)(smem + S::BM * S::BN * 2);  // behind the results
  if (threadIdx.x < S::BM) dst[threadIdx.x] = to;
  t.deliver(smem, wm, wn, lane, n0, a.N, [&](float gate, float up, int m) { return gg_gated(a, gate * factor[m], up * factor[m]); },
            [&](int row) -> bf16_t* { return dst[row] < 0 ? nullptr : (bf16_t*)a.C + (size_t)dst[row] * a.ldc; });
}

#define WIDE_OUT(glu) ((glu) ? 128 : 256)
#define ODD_OUT(glu) ((glu) ? 64 : 128)
#define WIDE_PAIRS (GS_TILES / 2)
using PairShape = TileShape<4, 4, 2, 3>;
using HalfShape = TileShape<2, 4, 3, 3>;   // an odd tile beside its group's pairs
using OddShape = TileShape<2, 2, 5, 5>;    // an odd tile apart: half as many outputs a workgroup, so that the last round is short
using ShortShape = TileShape<1, 2, 6, 6>;  // of up to 64 rows
// A pair of neighbouring tiles of a group or an odd last tile alone: the group's first tile, the group, the number of the group's
// first pair and how many tiles it has.
struct TileRun {
  int tile, group, first, tiles;
};
// runs: the number of pairs, the odd ones with them (as the first's tile), of whole pairs (as its group), of odd tiles (as its first) and of those with up
// to ShortShape::BM rows (as its tiles);
// then room for max_pairs pairs in the order of the tiles, then the order in which they are multiplied: whole pairs from the front (tile,
// group, the group's first whole pair, how many it has), odd tiles from the back (tile, group, rows that it holds).
//
// A compute unit holds one workgroup, and a round of pairs takes all of them for one pair each.  Odd tiles are tiles of 128 x 256 among their
// group's pairs, which read the same weights; or (APART, and where the numbers of pairs and odd tiles make it pay) the whole pairs come first and the
// odd tiles, cut in two, behind them.  An expert's last tile often holds few rows: 2,048 tokens, 8 of 32 experts, are 512 rows an
// expert give or take 20, so that half of the experts have a fifth tile of some 16.
// It pays where it saves a round: a half of an odd tile counts 0.8 of a pair, of up to 64 rows 0.35, and units that the last
// round of pairs leaves idle take them beside it.  Both products, beside / apart: 32 experts of 2,048 x 1,024 with 95 pairs and one odd tile (3.0
// rounds with it, 3.0 without) 370 / 403 us, 66 and 13 (2.5, 2.1) 338 / 353, 87 and 18 (3.3, 2.7) 438 / 411, 128 and 8 (4.3, 4.0) 562 / 525; 16 of 2,048 x
// 2,048 with 33 and 7 (2.5, 2.1) 321 / 341, 64 and 3 (4.2, 4.0) 530 / 470; 8 of 2,048 x 5,632 with 8 and 8 (2.8, 1.4) 318 / 355, 32 and 3 (6.0, 5.5) 726 / 695.
__device__ __forceinline__ bool odd_tiles_apart(const TileRun& head, int n_blocks, int odd_blocks) {
  const int pairs = head.group * n_blocks, rounds = (pairs + 255) / 256;
  const int odd = (16 * (head.first - head.tiles) + 7 * head.tiles) * odd_blocks;  // in twentieths of a pair
  const int behind = max(odd - 20 * (256 * rounds - pairs), 0), beside = (head.tile * n_blocks + 255) / 256;
  return rounds * 5120 + behind + 2560 < beside * 5120;  // (a round is 256 pairs; more than half of one is to be saved)
}

template <bool GLU, bool APART>
__global__ __launch_bounds__(256, 1) void grouped_gemm_pairs_kernel(GroupedArgs a, const TileRun* __restrict__ runs, int max_pairs, int n_blocks, int odd_blocks) {
  extern __shared__ __align__(16) char smem[];
  const TileRun head = runs[0];
  const bool apart = APART && odd_tiles_apart(head, n_blocks, odd_blocks);
  const TileRun* __restrict__ order = runs + 1 + (apart ? max_pairs : 0);
  const int items = (apart ? head.group : head.tile) * n_blocks, per = (items + GS_DIES - 1) / GS_DIES;
  const int seq = blockIdx.x / GS_DIES, die = blockIdx.x % GS_DIES;
  if (seq < per) {
    const int item = die * per + seq;
    if (item >= items) return;
    const int some = item / n_blocks;
    const TileRun r = order[some];
    // the chunk of up to WIDE_PAIRS pairs of the group that the item lies in
    const int pairs = apart ? r.tiles : (r.tiles + 1) / 2;
    const int chunk = r.first + (some - r.first) / WIDE_PAIRS * WIDE_PAIRS, len = min(WIDE_PAIRS, r.first + pairs - chunk);
    const int off = item - chunk * n_blocks, pair = chunk + off % len;
    const int tile = r.tile + 2 * (pair - r.first), n0 = off / len * WIDE_OUT(GLU);
    if (apart || tile + 1 < r.tile + r.tiles) wide_tile<PairShape, GLU>(a, smem, r.group, tile * GS_M, n0);
    else wide_tile<HalfShape, GLU>(a, smem, r.group, tile * GS_M, n0);
  } else if constexpr (APART) {
    if (!apart) return;
    const int odd = head.first * odd_blocks, odd_per = (odd + GS_DIES - 1) / GS_DIES, item = die * odd_per + seq - per;
    if (seq - per >= odd_per || item >= odd) return;
    const int some = item / odd_blocks;
    const TileRun r = order[max_pairs - 1 - some];
    const int n0 = (item - some * odd_blocks) * ODD_OUT(GLU);
    if (r.first <= ShortShape::BM) wide_tile<ShortShape, GLU>(a, smem, r.group, r.tile * GS_M, n0);
    else wide_tile<OddShape, GLU>(a, smem, r.group, r.tile * GS_M, n0);
  }
}

// Whether odd tiles may go apart at all (the kernel knows how many there are): where they are at most about one round of workgroups (`odd` of
// them at the most, half of that as a rule), and reading their experts' weights once more costs little beside.  Both products and the
// sum, us, with their pairs / all apart: 128 experts of 2,048 x 768 682 / 710 and 722 / 725 at 400 rows an expert, 8 of 4,096 x 14,336 1,109 / 1,251 and
// 1,123 / 1,302 at 380.
static bool odd_may_go_apart(int odd, int n_blocks, int K) { return (long)odd * n_blocks < 512 && K <= 4096; }

template <bool GLU>
static bool launch_by_tile(const GroupedArgs& a, int tiles, const TileRun* runs, int max_pairs, hipStream_t stream) {
  const auto groups = [](long n) { return (n + GS_DIES - 1) / GS_DIES * GS_DIES; };
  const int outs = GLU ? 64 : 128, n_blocks = (a.N + outs - 1) / outs;
  if (runs) {
    const int wide_blocks = (a.N + WIDE_OUT(GLU) - 1) / WIDE_OUT(GLU);
    const int odd_blocks = (a.N + ODD_OUT(GLU) - 1) / ODD_OUT(GLU);
    // Whole pairs W and odd tiles O: 2 W + O = `tiles` at the most, and O = `odd`, what room for (tiles + O) / 2 pairs in all was made for.
    // An odd tile apart is two items, so there are W + 2 O = (2 W + O) / 2 + 3 O / 2 <= (tiles + 3 odd) / 2 (each die's stretch is rounded up).
    const int odd = min(2 * max_pairs - tiles + 1, tiles);
    const long pairs = groups((tiles + 3l * odd) / 2 * wide_blocks) + 2 * GS_DIES;
    static_assert(PairShape::BM == 2 * GS_M && OddShape::BM == GS_M && HalfShape::BM == GS_M && HalfShape::LDS <= PairShape::LDS && OddShape::LDS <= PairShape::LDS && ShortShape::LDS <= PairShape::LDS &&
                      WIDE_OUT(GLU) == 2 * ODD_OUT(GLU), "");
    auto kernel = odd_may_go_apart(odd, wide_blocks, a.K) ? grouped_gemm_pairs_kernel<GLU, true> : grouped_gemm_pairs_kernel<GLU, false>;
    if (pairs >= (1l << 31) || hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, PairShape::LDS) != hipSuccess)
      return false;
    hipLaunchKernelGGL(kernel, dim3((unsigned)pairs), dim3(256), PairShape::LDS, stream, a, runs, max_pairs, wide_blocks, odd_blocks);
    return true;
  }
  const long grid = groups((long)tiles * n_blocks);
  if (grid >= (1l << 31)) return false;
  const int lds = GS_STAGES * 256 * GS_K * (int)sizeof(bf16_t);  // 48 KB; the results' place is 32 at most
  hipLaunchKernelGGL(grouped_gemm_staged_kernel<GLU>, dim3((unsigned)grid), dim3(256), lds, stream, a, tiles, n_blocks);
  return true;
}

TK_API int tk_grouped_gemm_bf16(const void* A, int lda, const int* a_row, const int* c_row, const int* tile_group, int tiles,
                                int groups_z, int a_cols, int c_cols, const void* W, size_t w_stride, void* C, int ldc,
                                int N, int K, int slots, const TileRun* runs, int max_pairs, long a_rows, int glu, int out_f32, const float* row_scale, const int* scale_row,
                                float limit, float alpha, hipStream_t stream) {
  TK_REQUIRE(A && W && C && N > 0 && K > 0 && slots >= 0 && tiles >= 0, "grouped_gemm: bad arguments");
  TK_REQUIRE(K % 8 == 0 && lda % 8 == 0 && a_cols % 8 == 0 && w_stride % 8 == 0 && (((uintptr_t)A | (uintptr_t)W) & 15) == 0,
             "grouped_gemm: rows of A and W must start at multiples of 16 bytes (K=%d lda=%d)", K, lda);
  TK_REQUIRE((tile_group != nullptr) != (groups_z > 0), "grouped_gemm: groups come by tile or by the grid, not both");
  TK_REQUIRE(!row_scale || (glu && scale_row && a_row), "grouped_gemm: a factor a row goes with the gated form and rows by slot");
  TK_REQUIRE(!(glu && out_f32), "grouped_gemm: the gated form writes the storage type");
  if (tiles == 0 || slots == 0) return 0;
  GroupedArgs a{(const bf16_t*)A, lda, a_row, c_row, tile_group, a_cols, c_cols, (const bf16_t*)W, w_stride, C, ldc, N, K, slots,
                row_scale, scale_row, limit, alpha};
  if (tile_group) {
    TK_REQUIRE(!out_f32 && a_cols == 0 && c_cols == 0, "grouped_gemm: groups by tile write the storage type and have no columns of their own");
    TK_REQUIRE(!runs || (((uintptr_t)runs & 15) == 0 && K % TILE_K == 0 && a_rows * lda * 2 < (1l << 32) && (glu ? 2l : 1l) * N * K * 2 < (1l << 32) && max_pairs > 0),
               "grouped_gemm: pairs of tiles take whole steps of %d of K, and rows that 32-bit offsets reach", TILE_K);
    TK_REQUIRE(!runs || (2l * max_pairs >= tiles), "grouped_gemm: %d pairs are no list of the pairs of %d tiles", max_pairs, tiles);
    TK_REQUIRE(glu ? launch_by_tile<true>(a, tiles, runs, max_pairs, stream) : launch_by_tile<false>(a, tiles, runs, max_pairs, stream), "grouped_gemm: too many outputs");
    TK_CHECK_LAUNCH("grouped_gemm");
    return 0;
  }
  TK_REQUIRE(!glu && !a_row && !c_row, "grouped_gemm: groups by the grid take plain rows and have no gated form");
  const dim3 grid(tiles, (N + GG_WAVES * 64 - 1) / (GG_WAVES * 64), groups_z);
  TK_REQUIRE((long)tiles * GG_TM >= slots && grid.y < 65536 && grid.z < 65536, "grouped_gemm: too few tiles, or too many outputs or groups");
  if (out_f32)
    hipLaunchKernelGGL((grouped_gemm_kernel<4, true>), grid, dim3(GG_WAVES * TK_WAVE), 0, stream, a);
  else
    hipLaunchKernelGGL((grouped_gemm_kernel<4, false>), grid, dim3(GG_WAVES * TK_WAVE), 0, stream, a);
  TK_CHECK_LAUNCH("grouped_gemm");
  return 0;
}

// --------------------------------------------------------------------------
// Pairs (token, place) -> slots sorted by expert.  A workgroup a job: a layer's choice, or (where the choice of several layers
// is known before the first of them runs) all layers' in one launch.  Expert e's pairs take the slots
// first[e] .. first[e] + count[e] - 1 with first[e] a multiple of GS_M; the slots between a run's end and the
// next multiple are empty.  slot_pair[slot] = the pair (or -1), slot_token[slot] = its token (or -1),
// tile_group[tile] = the expert whose run the tile lies in (or -1), tile_group[max_tiles] = the tiles in use.  Pairs of identity experts (ids >= experts)
// and empty places (ids < 0) get no slot.  Which of an expert's slots a pair gets depends on the order of
// arrival and changes no result: every row is computed on its own.
// --------------------------------------------------------------------------
struct SortJob {
  const int* ids;
  int *slot_pair, *slot_token, *tile_group;
  TileRun* runs;  // (grouped_gemm_pairs_kernel: room for the numbers and twice max_pairs pairs)
  int pairs, top, experts, max_tiles, max_pairs;
};
#define SORT_JOBS 48
struct SortJobs {
  SortJob job[SORT_JOBS];
};
__global__ __launch_bounds__(1024) void expert_sort_kernel(SortJobs jobs) {
  const SortJob& jb = jobs.job[blockIdx.x];
  const int* __restrict__ ids = jb.ids;
  const int pairs = jb.pairs, top = jb.top, experts = jb.experts, max_tiles = jb.max_tiles, tm = GS_M;
  int* __restrict__ slot_pair = jb.slot_pair;
  int* __restrict__ slot_token = jb.slot_token;
  int* __restrict__ tile_group = jb.tile_group;
  extern __shared__ int sh[];  // [experts] each: counts (then the slots that are left), first slots, first pairs of tiles
  int* count = sh;
  int* first = sh + experts;
  int* first_pair = sh + 2 * experts;
  __shared__ int shorts;
  if (threadIdx.x == 0) shorts = 0;
  for (int e = threadIdx.x; e < experts; e += blockDim.x) count[e] = 0;
  for (int s = threadIdx.x; s < max_tiles * tm; s += blockDim.x) slot_pair[s] = slot_token[s] = -1;
  for (int t = threadIdx.x; t < max_tiles; t += blockDim.x) tile_group[t] = -1;
  __syncthreads();
  for (int p = threadIdx.x; p < pairs; p += blockDim.x) {
    const int e = ids[p];
    if (e >= 0 && e < experts) atomicAdd(&count[e], 1);
  }
  __syncthreads();
  int at = 0, twos = 0;
  if (threadIdx.x == 0) {
    for (int e = 0; e < experts; ++e) {
      const int n = (count[e] + tm - 1) / tm;
      first[e] = at;
      first_pair[e] = twos;
      at += n * tm;
      twos += (n + 1) / 2;
    }
    tile_group[max_tiles] = at / tm;
  } else if (threadIdx.x >= TK_WAVE) {  // beside that: odd last tiles of few rows
    for (int e = threadIdx.x - TK_WAVE; e < experts; e += blockDim.x - TK_WAVE) {
      const int over = count[e] % (2 * tm);
      if (over > 0 && over <= ShortShape::BM) atomicAdd(&shorts, 1);
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) jb.runs[0] = {twos, at / tm - twos, 2 * twos - at / tm, shorts};
  for (int e = threadIdx.x; e < experts; e += blockDim.x) {
    const int t0 = first[e] / tm, n = (count[e] + tm - 1) / tm;
    for (int t = 0; t < n; ++t) tile_group[t0 + t] = e;
    for (int p = 0; p < (n + 1) / 2; ++p) jb.runs[1 + first_pair[e] + p] = {t0, e, first_pair[e], n};
    // of the t0 tiles in front, in first_pair[e] pairs: whole pairs t0 - first_pair[e], odd tiles the rest of the pairs
    TileRun* order = jb.runs + 1 + jb.max_pairs;
    const int whole = t0 - first_pair[e];
    for (int p = 0; p < n / 2; ++p) order[whole + p] = {t0, e, whole, n / 2};
    if (n & 1) order[jb.max_pairs - 1 - (first_pair[e] - whole)] = {t0 + n - 1, e, count[e] - (n - 1) * tm, 1};
  }
  __syncthreads();
  for (int p = threadIdx.x; p < pairs; p += blockDim.x) {
    const int e = ids[p];
    if (e >= 0 && e < experts) {
      const int s = first[e] + atomicSub(&count[e], 1) - 1;
      slot_pair[s] = p;
      slot_token[s] = p / top;
    }
  }
}

TK_API int tk_expert_sort(const SortJob* jobs, int n_jobs, hipStream_t stream) {
  TK_REQUIRE(jobs && n_jobs >= 0, "expert_sort: bad arguments");
  for (int first = 0; first < n_jobs; first += SORT_JOBS) {
    SortJobs all{};
    const int n = min(SORT_JOBS, n_jobs - first);
    int most = 0;
    for (int k = 0; k < n; ++k) {
      const SortJob& j = all.job[k] = jobs[first + k];
      TK_REQUIRE(j.ids && j.slot_pair && j.slot_token && j.tile_group && j.runs && j.pairs >= 0 && j.top > 0 && j.experts > 0, "expert_sort: bad arguments");
      // (each expert that has pairs leaves at most one tile partly empty)
      TK_REQUIRE(j.max_tiles >= (j.pairs + (long)(GS_M - 1) * min(j.experts, j.pairs)) / GS_M, "expert_sort: %d tiles cannot hold %d pairs of %d experts", j.max_tiles,
                 j.pairs, j.experts);
      TK_REQUIRE(j.max_pairs >= (j.max_tiles + min(j.experts, j.max_tiles)) / 2, "expert_sort: %d pairs cannot hold those of %d tiles", j.max_pairs, j.max_tiles);
      TK_REQUIRE(3 * j.experts * sizeof(int) <= 48 * 1024, "expert_sort: too many experts");
      most = max(most, j.experts);
    }
    hipLaunchKernelGGL(expert_sort_kernel, dim3(n), dim3(1024), 3 * most * sizeof(int), stream, all);
    TK_CHECK_LAUNCH("expert_sort");
  }
  return 0;
}

// --------------------------------------------------------------------------
// out[t, c] = sum over the places k of token t, in order, of weights[t, k] * (y[t * top + k, c] for a routed expert,
// h[t, c] for an identity expert), plus shared_gate[t] * shared[t, c].  y: [pairs, width] in the storage type.
// `unit` != 0: a routed expert's row is added as it is.  weights null: equal parts, 1 / top each.
// --------------------------------------------------------------------------
__global__ __launch_bounds__(256) void expert_sum_kernel(const bf16_t* __restrict__ h, int h_stride, const bf16_t* __restrict__ y,
                                                         const int* __restrict__ ids, const float* __restrict__ weights,
                                                         const float* __restrict__ shared, const float* __restrict__ shared_gate,
                                                         float* __restrict__ out, int width, int experts, int top, int unit) {
  const int t = blockIdx.x;
  for (int c = threadIdx.x; c < width; c += blockDim.x) {
    float acc = 0.f;
    for (int k = 0; k < top; ++k) {
      const int e = ids[(size_t)t * top + k];
      if (e < 0) continue;
      const float v = e < experts ? __bfloat162float(y[((size_t)t * top + k) * width + c]) : __bfloat162float(h[(size_t)t * h_stride + c]);
      acc = fmaf(unit && e < experts ? 1.f : (weights ? weights[(size_t)t * top + k] : 1.0f / (float)top), v, acc);
    }
    if (shared) acc = fmaf(shared_gate[t], shared[(size_t)t * width + c], acc);
    out[(size_t)t * width + c] = acc;
  }
}

// The same with 16 bytes a load, a thread eight neighbouring columns, and all of a token's rows asked for before the first is
// used (EXPERT_SUM_TOP at a time).
#define EXPERT_SUM_TOP 4
__global__ __launch_bounds__(256) void expert_sum_vec_kernel(const bf16_t* __restrict__ h, int h_stride, const bf16_t* __restrict__ y,
                                                             const int* __restrict__ ids, const float* __restrict__ weights,
                                                             const float* __restrict__ shared, const float* __restrict__ shared_gate,
                                                             float* __restrict__ out, int width, int experts, int top, int unit) {
  const size_t t = blockIdx.x;
  for (int c = threadIdx.x * 8; c < width; c += blockDim.x * 8) {
    float acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = 0.f;
    for (int k0 = 0; k0 < top; k0 += EXPERT_SUM_TOP) {
      uint4 raw[EXPERT_SUM_TOP];
      float f[EXPERT_SUM_TOP];
#pragma unroll
      for (int k = 0; k < EXPERT_SUM_TOP; ++k) {
        f[k] = 0.f;
        raw[k] = make_uint4(0, 0, 0, 0);
        if (k0 + k >= top) continue;
        const int e = ids[t * top + k0 + k];
        if (e < 0) continue;
        f[k] = unit && e < experts ? 1.f : (weights ? weights[t * top + k0 + k] : 1.0f / (float)top);
        raw[k] = e < experts ? *(const uint4*)(y + (t * top + k0 + k) * width + c) : *(const uint4*)(h + t * h_stride + c);
      }
#pragma unroll
      for (int k = 0; k < EXPERT_SUM_TOP; ++k) {
        const bf16_t* v = (const bf16_t*)&raw[k];
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] = fmaf(f[k], __bfloat162float(v[j]), acc[j]);
      }
    }
    if (shared) {
      const float s = shared_gate[t];
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[j] = fmaf(s, shared[t * width + c + j], acc[j]);
    }
    *(float4*)(out + t * width + c) = make_float4(acc[0], acc[1], acc[2], acc[3]);
    *(float4*)(out + t * width + c + 4) = make_float4(acc[4], acc[5], acc[6], acc[7]);
  }
}

TK_API int tk_expert_sum(const void* h, int h_stride, const void* y, const int* ids, const float* weights, const float* shared,
                         const float* shared_gate, float* out, int tokens, int width, int experts, int top, int unit, hipStream_t stream) {
  TK_REQUIRE(h && y && ids && out && (!shared || shared_gate) && tokens >= 0 && width > 0 && top > 0 && h_stride >= width,
             "expert_sum: bad arguments");
  if (tokens == 0) return 0;
  if (width % 8 == 0 && h_stride % 8 == 0 && (((uintptr_t)h | (uintptr_t)y | (uintptr_t)out | (uintptr_t)shared) & 15) == 0) {
    hipLaunchKernelGGL(expert_sum_vec_kernel, dim3(tokens), dim3(256), 0, stream, (const bf16_t*)h, h_stride, (const bf16_t*)y, ids,
                       weights, shared, shared_gate, out, width, experts, top, unit);
    TK_CHECK_LAUNCH("expert_sum");
    return 0;
  }
  hipLaunchKernelGGL(expert_sum_kernel, dim3(tokens), dim3(256), 0, stream, (const bf16_t*)h, h_stride, (const bf16_t*)y, ids,
                     weights, shared, shared_gate, out, width, experts, top, unit);
  TK_CHECK_LAUNCH("expert_sum");
  return 0;
}
