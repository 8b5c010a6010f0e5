// A tile of a bfloat16 matrix product through local memory, for products of many rows:  C[m, n] = sum_k A[m, k] W[n, k].
//
// A workgroup of 4 wavefronts owns 64 TM rows of A and 64 TN rows of W, a wavefront 32 TM x 32 TN of them.  Two things bound it.
// The path from the L2 to a compute unit gives about 35 bytes a clock whatever the tile (32 KB take 920 clocks for a tile of
// 128 x 128, whose products take 512), so a tile is as large as the shape of the product lets it be, and the sums stay in
// registers (256 for 256 x 256: one wavefront a SIMD).  And with the whole chip at it, power: the clock falls to 1.6 GHz (2.1 on
// operands of zeros), and what counts is the energy of an operation.  v_mfma_f32_16x16x32_bf16 reads and writes its sums half as
// often as the 32 x 32 x 16 form: 4,096 x 4,096 x 14,336 rows 353 to 321 us (1.5 PFLOP/s), the same bits.
//
// Steps of 64 elements of K (128 bytes of a row, a whole cache line: steps of 32 elements in twice the buffers took 10 to 30 %
// longer) go straight from memory to local memory; of W, which comes from memory, a step more is on its way than of A, which the
// L2 holds (256 x 256: two steps of A and three of W are all of the 160 KB; with two of each a step waits for its loads, 148
// against 132 us for 2,048 x 2,048 x 8,192).  A wavefront is alone on its SIMD, so the order within a step is written down: between a
// block's products (32 elements of K) come the reads of the next block's operands and the loads of the steps ahead, a few at a
// time (all at once behind the barrier: 2 to 8 % slower); one barrier a step, in front of its second block, when all of the step's
// operands are in registers or on their way there.  Tiles of up to 128 x 256 ask for two wavefronts a SIMD (launch bounds) only
// so that their sums are kept in the ordinary registers, where the compiler does not move them between the products.
#pragma once
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 tile_bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float tile_f32x4_t;

#define TILE_K 64  // elements of K a step

template <int TM_, int TN_, int SA_, int SW_>
struct TileShape {
  static constexpr int TM = TM_, TN = TN_, SA = SA_, SW = SW_;  // steps of A and of W that local memory holds
  static_assert(SW == SA || SW == SA + 1, "");
  static constexpr int BM = 64 * TM, BN = 64 * TN;
  static constexpr int ROW = TILE_K * 2;                      // bytes of a row of a step
  static constexpr int A_STEP = BM * ROW, W_STEP = BN * ROW;  // bytes of a step
  static constexpr int W_AT = SA * A_STEP, LDS = W_AT + SW * W_STEP;
  static constexpr int LA = BM / 32, LW = BN / 32, LOADS = LA + LW;  // loads (of 8 rows) a wavefront and step
};
// place of a row's 16-byte piece c: c ^ tile_swizzle(row)
__device__ __forceinline__ int tile_swizzle(int row) { return (row ^ (row >> 3 & 1)) & 7; }

__device__ __forceinline__ void tile_load(const void* base, unsigned off, unsigned lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory", "m0");
}

template <class S, bool GLU>
struct TileLoop {
  static constexpr int TM = S::TM, TN = S::TN;
  static constexpr int XB = 2 * TM, WB = 2 * TN;  // blocks of 16 rows of A and of W that a wavefront owns
  static constexpr int UNITS = XB * WB, READS = XB + WB;
  const char *a, *w;       // first bytes, in the rows of A and W, of the steps that are asked for next (uniform)
  unsigned off[S::LOADS];  // bytes from there to this lane's piece of every load: rows of A, then of W
  unsigned lds;
  int wave;
  tile_f32x4_t acc[WB][XB];
  const char *xl[2], *wl[2];  // a lane's first row in the first step's place, per 32 elements of K
  struct Frag {
    tile_bf16x8_t x[XB], w[WB];
  };
  Frag f[2];

  template <int N, int TO>
  __device__ __forceinline__ void loads(int place) {
    if constexpr (N < TO) {
      if constexpr (N < S::LA) tile_load(a, off[N], lds + place + (wave * (16 * TM) + N * 8) * S::ROW);
      else tile_load(w, off[N], lds + S::W_AT + place + (wave * (16 * TN) + (N - S::LA) * 8) * S::ROW);
      loads<N + 1, TO>(place);
    }
  }
  // reads N .. of a block of 32 elements: w0, x0 .. , w1 ..
  template <int N, int TO>
  __device__ __forceinline__ void reads(Frag& q, const char* xp, const char* wp) {
    if constexpr (N < TO) {
      if constexpr (N >= 1 && N <= XB) {
        q.x[N - 1] = *(const tile_bf16x8_t*)(xp + (N - 1) * 16 * S::ROW);
      } else {
        constexpr int T = N == 0 ? 0 : N - XB;
        constexpr int row = GLU && T >= TN ? S::BN / 2 + (T - TN) * 16 : T * 16;
        q.w[T] = *(const tile_bf16x8_t*)(wp + row * S::ROW);
      }
      reads<N + 1, TO>(q, xp, wp);
    }
  }
  static constexpr int reads_to(int u) {
    const int n = u * READS * (UNITS < 64 ? 2 : 1) / UNITS;
    return n < READS ? n : READS;
  }
  // the products of a block; between them the reads of the next block and the loads FROM .. TO
  template <int U, bool READ, int FROM, int TO>
  __device__ __forceinline__ void units(const Frag& c, Frag& q, const char* xp, const char* wp, int place) {
    if constexpr (U < UNITS) {
      acc[U / XB][U % XB] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c.w[U / XB], c.x[U % XB], acc[U / XB][U % XB], 0, 0, 0);
      if constexpr (READ) reads<reads_to(U), reads_to(U + 1)>(q, xp, wp);
      loads<FROM + U * (TO - FROM) / UNITS, FROM + (U + 1) * (TO - FROM) / UNITS>(place);
      __builtin_amdgcn_sched_barrier(0);
      units<U + 1, READ, FROM, TO>(c, q, xp, wp, place);
    }
  }
  int a_here, a_next, w_last, w_here, w_next;  // places of a step, the next and the one before, in bytes
  // FW: the rest of the loads of the step whose rows of A were asked for last (W's), FA: the rows of A of the next such step
  template <bool FW, bool FA, bool LAST>
  __device__ __forceinline__ void step() {
    __builtin_amdgcn_sched_barrier(0);
    units<0, true, FW ? S::LA : 0, FW ? S::LOADS : 0>(f[0], f[1], xl[1] + a_here, wl[1] + w_here, w_last);
    if constexpr (!LAST) {
      w += S::ROW;
      if constexpr (FW) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((S::SA - 2) * S::LOADS + (S::SW - S::SA) * S::LW) : "memory");
      else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
    units<0, !LAST, 0, FA ? S::LA : 0>(f[1], f[0], xl[0] + a_next, wl[0] + w_next, a_here);
    a += S::ROW;
    a_here = a_next;
    a_next = a_next == (S::SA - 1) * S::A_STEP ? 0 : a_next + S::A_STEP;
    w_last = w_here;
    w_here = w_next;
    w_next = w_next == (S::SW - 1) * S::W_STEP ? 0 : w_next + S::W_STEP;
  }
  __device__ __forceinline__ void run(char* smem, int steps, int wm, int wn, int lane) {
    const int r = lane & 15, q = lane >> 4;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int place = ((4 * k + q) ^ tile_swizzle(r)) * 16;
      xl[k] = smem + (wm * (32 * TM) + r) * S::ROW + place;
      wl[k] = smem + S::W_AT + (wn * (GLU ? 16 * TN : 32 * TN) + r) * S::ROW + place;
    }
#pragma unroll
    for (int t = 0; t < WB; ++t)
#pragma unroll
      for (int m = 0; m < XB; ++m) acc[t][m] = tile_f32x4_t{0.f, 0.f, 0.f, 0.f};
    // asked for in front of the loop: SA steps of A and SW - 1 of W
#pragma unroll
    for (int st = 0; st < S::SA; ++st) {
      if (st < steps) {
        loads<0, S::LA>(st * S::A_STEP);
        a += S::ROW;
        if (st < S::SW - 1) {
          loads<S::LA, S::LOADS>(st * S::W_STEP);
          w += S::ROW;
        }
      }
    }
    if (steps >= S::SA) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((S::SA - 1) * S::LA + (S::SW - 2) * S::LW) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    reads<0, READS>(f[0], xl[0], wl[0]);
    a_here = w_here = 0;
    a_next = S::A_STEP;
    w_next = S::W_STEP;
    w_last = (S::SW - 1) * S::W_STEP;
    int s = 0;
#pragma unroll 1
    for (; s + S::SA < steps; ++s) step<true, true, false>();
    if (S::SW == S::SA && s + S::SA == steps) {
      step<true, false, false>();
      ++s;
    }
#pragma unroll 1
    for (; s + 1 < steps; ++s) step<false, false, false>();
    step<false, false, true>();
  }

  // The tile's results, rounded, through local memory (16-byte pieces exchanged by the row's number) to the rows that `dst(row)` names
  // (null: none), columns n0 .. of N; value(gate's sum, up's sum, m) in the gated form.
  template <class Value, class Dst>
  __device__ __forceinline__ void deliver(char* smem, int wm, int wn, int lane, int n0, int N, Value value, Dst dst) {
    constexpr int OUT = GLU ? S::BN / 2 : S::BN, PIECES = OUT / 8, MASK = PIECES % 16 == 0 ? 15 : (PIECES % 8 == 0 ? 7 : 3);
    bf16_t* rows = (bf16_t*)smem;
    const int r = lane & 15, q = lane >> 4;
    __syncthreads();
#pragma unroll
    for (int m = 0; m < XB; ++m) {
      const int row = wm * (32 * TM) + m * 16 + r;
#pragma unroll
      for (int t = 0; t < (GLU ? TN : WB); ++t) {
        union { bf16_t v[4]; uint2 raw; } o;
#pragma unroll
        for (int j = 0; j < 4; ++j) {  // a lane holds the outputs 4 q + 0 .. 3 of a block of 16
          const float y = GLU ? value(acc[t][m][j], acc[t + (GLU ? TN : 0)][m][j], m) : acc[t][m][j];
          o.v[j] = __float2bfloat16(y);
        }
        const int u = (wn * (GLU ? 16 * TN : 32 * TN) + t * 16) / 4 + q;  // of 4 outputs
        *(uint2*)(rows + row * OUT + ((u >> 1) ^ (row & MASK)) * 8 + (u & 1) * 4) = o.raw;
      }
    }
    __syncthreads();
#pragma unroll 4
    for (int i = threadIdx.x; i < S::BM * PIECES; i += 256) {
      const int row = i / PIECES, p = i % PIECES, left = N - n0 - p * 8;
      bf16_t* to = dst(row);
      if (to == nullptr || left <= 0) continue;
      to += n0 + p * 8;
      const uint4 v = *(const uint4*)(rows + row * OUT + (p ^ (row & MASK)) * 8);
      if (left >= 8 && ((uintptr_t)to & 15) == 0) {
        *(uint4*)to = v;
      } else {
        const bf16_t* e = (const bf16_t*)&v;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (j < left) to[j] = e[j];
      }
    }
  }
};
