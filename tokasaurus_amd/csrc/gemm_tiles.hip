// bfloat16 matrix products of many rows in tiles of gemm_tile.h, C[M, N] = A[M, K] W[N, K]^T, and the gated form
// silu(A Wg^T) * (A Wu^T) of a weight [gate | up], which saves the pass behind a plain product (a read of 2 M N and a write of M N
// numbers: 18 us for 2,048 x 8,192).
//
// Which of the tiles a product takes, and from where on the library's product is faster, says ops.tiles_choice, with the
// measurements.  Tiles come in bands of BAND tiles of rows through all outputs, each of the chip's eight dies a stretch of that order
// (the hardware deals workgroups to the dies in turn), so that the tiles a die works on at a time share rows of A and of W in its
// L2 (bands of 4 or 8: the same within 3 %; tiles of rows without bands 119 to 138 us for 2,048 rows of gate and up, 16,384 x 2,048).
#include "calls.h"
#include "gemm_tile.h"

#define TILE_DIES 8
#define BAND 4

struct TilesArgs {
  const bf16_t* A;
  int lda;
  const bf16_t* W;
  bf16_t* C;
  int ldc;
  int M, N, K;
  int m_tiles, n_tiles;
};

template <class S, bool GLU>
__global__ __launch_bounds__(256, S::TM * S::TN <= 8 ? 2 : 1) void gemm_tiles_kernel(TilesArgs a) {
  constexpr int TM = S::TM, TN = S::TN;
  extern __shared__ __align__(16) char smem[];
  constexpr int OUT = GLU ? S::BN / 2 : S::BN;
  const int items = a.m_tiles * a.n_tiles, per = (items + TILE_DIES - 1) / TILE_DIES;
  const int seq = blockIdx.x / TILE_DIES, item = blockIdx.x % TILE_DIES * per + seq;
  if (seq >= per || item >= items) return;
  const int whole = BAND * a.n_tiles, b = item / whole, in = item - b * whole;
  const int len = min(BAND, a.m_tiles - b * BAND);
  const int m0 = (b * BAND + in % len) * S::BM, n0 = in / len * OUT;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  TileLoop<S, GLU> t;
  t.wave = wave;
  t.lds = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  t.a = (const char*)(a.A + (size_t)m0 * a.lda);
  t.w = (const char*)(a.W + (size_t)n0 * a.K);
  const int lr = lane >> 3;
#pragma unroll
  for (int i = 0; i < S::LA; ++i) {
    const int row = wave * (16 * TM) + i * 8 + lr;
    t.off[i] = (unsigned)min(row, a.M - 1 - m0) * (unsigned)a.lda * 2 + ((lane & 7) ^ tile_swizzle(row)) * 16;
  }
#pragma unroll
  for (int i = 0; i < S::LW; ++i) {
    const int row = wave * (16 * TN) + i * 8 + lr;
    const int wrow = GLU ? min(row % OUT, a.N - 1 - n0) + (row >= OUT ? a.N : 0) : min(row, a.N - 1 - n0);
    t.off[S::LA + i] = (unsigned)wrow * (unsigned)a.K * 2 + ((lane & 7) ^ tile_swizzle(row)) * 16;
  }
  t.run(smem, a.K / TILE_K, wm, wn, lane);
  t.deliver(smem, wm, wn, lane, n0, a.N, [](float g, float u, int) { return silu_mul_bf16(g, u); },
            [&](int row) -> bf16_t* { return m0 + row < a.M ? a.C + (size_t)(m0 + row) * a.ldc : nullptr; });
}

template <class S, bool GLU>
static bool launch_tiles(TilesArgs a, hipStream_t stream) {
  constexpr int OUT = GLU ? S::BN / 2 : S::BN;
  a.m_tiles = (a.M + S::BM - 1) / S::BM;
  a.n_tiles = (a.N + OUT - 1) / OUT;
  auto kernel = gemm_tiles_kernel<S, GLU>;
  if (S::LDS > 64 * 1024 && hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, S::LDS) != hipSuccess) return false;
  const int items = a.m_tiles * a.n_tiles, per = (items + TILE_DIES - 1) / TILE_DIES;
  hipLaunchKernelGGL(kernel, dim3(per * TILE_DIES), dim3(256), S::LDS, stream, a);
  return true;
}

template <bool GLU>
static bool launch_shape(const TilesArgs& a, int shape, hipStream_t stream) {
  switch (shape) {
    case 0: return launch_tiles<TileShape<2, 2, 5, 5>, GLU>(a, stream);
    case 1: return launch_tiles<TileShape<3, 2, 4, 4>, GLU>(a, stream);
    case 2: return launch_tiles<TileShape<2, 4, 3, 3>, GLU>(a, stream);
  }
  if constexpr (GLU) {
    switch (shape) {
      case 3: return launch_tiles<TileShape<3, 4, 2, 3>, GLU>(a, stream);
      case 4: return launch_tiles<TileShape<4, 4, 2, 3>, GLU>(a, stream);
      case 5: return launch_tiles<TileShape<2, 1, 6, 6>, GLU>(a, stream);
    }
  }
  return false;
}

// glu: W is [gate | up], [2 N, K]; else [N, K].  shape: tiles of 128 x 128 (0), 192 x 128 and 128 x 256 rows of A and of W, and gated of
// 192 x 256 (3), 256 x 256 and 128 x 64; plain products of such tiles were behind the library's.
TK_API int tk_gemm_tiles_bf16(const void* A, int lda, const void* W, void* C, int ldc, int M, int N, int K, int glu, int shape,
                              hipStream_t stream) {
  TK_REQUIRE(A && W && C && M >= 0 && N > 0 && K > 0 && K % TILE_K == 0, "gemm_tiles: bad sizes M=%d N=%d K=%d", M, N, K);
  TK_REQUIRE(lda >= K && lda % 8 == 0 && ldc >= N && (((uintptr_t)A | (uintptr_t)W) & 15) == 0 && ((uintptr_t)C & 1) == 0,
             "gemm_tiles: rows of A and W must start at multiples of 16 bytes (lda=%d)", lda);
  // (bytes from a tile's first row of A, and of W, are 32-bit numbers)
  TK_REQUIRE(256l * lda * 2 < (1l << 32) && (glu ? N + 256l : 256l) * K * 2 < (1l << 32), "gemm_tiles: rows too long (lda=%d N=%d K=%d)", lda, N, K);
  TK_REQUIRE((long)((M + 127) / 128) * ((N + 31) / 32) < (1l << 30), "gemm_tiles: too many tiles (M=%d N=%d)", M, N);
  if (M == 0) return 0;
  const TilesArgs a{(const bf16_t*)A, lda, (const bf16_t*)W, (bf16_t*)C, ldc, M, N, K, 0, 0};
  const bool ok = glu ? launch_shape<true>(a, shape, stream) : launch_shape<false>(a, shape, stream);
  TK_REQUIRE(ok, "gemm_tiles: tile %d (0 .. 2, gated up to 5) cannot be launched", shape);
  TK_CHECK_LAUNCH("gemm_tiles");
  return 0;
}
