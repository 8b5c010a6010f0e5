// C[M,N] = A[M,K] * W[N,K]^T (+ residual[M,N]) with plain 32-bit multiply-adds:
// the matrix product of operands whose rows do not start at multiples of 16 bytes, in either
// storage type (the matrix-core kernels take the others: gemm_f32.hip, gemm_mfma.hip).
// Operands are row-major with K contiguous; any M, N, K.  A bias (one value an output, of the storage type, or null) is added
// to the product in 32-bit before it is rounded.  Two kernels: tiles of 64 x 64 through LDS, each output
// summing its K products in ascending k; and, for up to GR_MAX_ROWS rows (decode), one
// that streams the weights: a wavefront owns GR_COLS output columns, its lanes cut K
// between them and add up at the end.  In both the order of an output's additions is
// fixed by K alone, so a row's result does not depend on what else is in the batch
// beyond which of the two kernels the batch's size selects (rounding).
#include "common.h"

#define GR_COLS 4
#define GR_MAX_ROWS 32

// Four consecutive elements as 32-bit floats (k may run past K).
template <typename T>
__device__ __forceinline__ void load4(const T* row, int k, int K, float out[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) out[i] = (k + i < K) ? to_f32<T>(row[k + i]) : 0.f;
}

template <typename T, typename TO, int MB>
__global__ __launch_bounds__(256) void gemm_rows_kernel(const T* __restrict__ A, int lda,
                                                        const T* __restrict__ W,
                                                        TO* __restrict__ C, int ldc,
                                                        const T* __restrict__ residual, int ldr,
                                                        const T* __restrict__ bias, int M, int N, int K) {
  const int lane = threadIdx.x & (TK_WAVE - 1), wave = threadIdx.x / TK_WAVE;
  const int n0 = (blockIdx.x * (256 / TK_WAVE) + wave) * GR_COLS;
  const int m0 = blockIdx.y * MB;
  if (n0 >= N) return;
  float acc[MB][GR_COLS];
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int c = 0; c < GR_COLS; ++c) acc[m][c] = 0.f;
  for (int k = lane * 4; k < K; k += TK_WAVE * 4) {
    float w[GR_COLS][4];
#pragma unroll
    for (int c = 0; c < GR_COLS; ++c) load4<T>(W + (size_t)min(n0 + c, N - 1) * K, k, K, w[c]);
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      if (m0 + m < M) {  // the same for every lane
        float a[4];
        load4<T>(A + (size_t)(m0 + m) * lda, k, K, a);
#pragma unroll
        for (int c = 0; c < GR_COLS; ++c)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[m][c] = fmaf(a[i], w[c][i], acc[m][c]);
      }
    }
  }
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    if (m0 + m >= M) continue;
#pragma unroll
    for (int c = 0; c < GR_COLS; ++c) {
      float v = acc[m][c];
#pragma unroll
      for (int o = TK_WAVE / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, TK_WAVE);
      if (lane == 0 && n0 + c < N) {
        if (bias) v += to_f32<T>(bias[n0 + c]);
        if (residual) v = round_to<T>(v) + to_f32<T>(residual[(size_t)(m0 + m) * ldr + n0 + c]);
        C[(size_t)(m0 + m) * ldc + n0 + c] = from_f32<TO>(v);
      }
    }
  }
}

template <typename T, typename TO>
static void launch_rows(const T* A, int lda, const T* W, TO* C, int ldc, const T* residual, int ldr, const T* bias,
                        int M, int N, int K, hipStream_t stream) {
  const int cols_per_block = (256 / TK_WAVE) * GR_COLS;
  const unsigned gx = (unsigned)((N + cols_per_block - 1) / cols_per_block);
#define TK_ROWS_LAUNCH(MB)                                                                             \
  hipLaunchKernelGGL((gemm_rows_kernel<T, TO, MB>), dim3(gx, (M + MB - 1) / MB), dim3(256), 0, stream, \
                     A, lda, W, C, ldc, residual, ldr, bias, M, N, K)
  if (M <= 4) TK_ROWS_LAUNCH(4);
  else TK_ROWS_LAUNCH(16);
#undef TK_ROWS_LAUNCH
}

#define GT_BM 64
#define GT_BN 64
#define GT_BK 16

template <typename T, typename TO>
__global__ __launch_bounds__(256) void gemm_generic_kernel(const T* __restrict__ A, int lda,
                                                           const T* __restrict__ W,
                                                           TO* __restrict__ C, int ldc,
                                                           const T* __restrict__ residual,
                                                           int ldr, const T* __restrict__ bias, int M, int N, int K) {
  __shared__ float As[GT_BK][GT_BM + 1];
  __shared__ float Ws[GT_BK][GT_BN + 1];
  const int tid = threadIdx.x;
  const int m0 = blockIdx.y * GT_BM, n0 = blockIdx.x * GT_BN;
  const int ty = tid / 16, tx = tid % 16;
  const int lr = tid / 4, lk = (tid % 4) * 4;  // loader: row within tile, first k
  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;

  for (int k0 = 0; k0 < K; k0 += GT_BK) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int k = k0 + lk + q;
      const int am = m0 + lr, wn = n0 + lr;
      As[lk + q][lr] = (am < M && k < K) ? to_f32<T>(A[(size_t)am * lda + k]) : 0.f;
      Ws[lk + q][lr] = (wn < N && k < K) ? to_f32<T>(W[(size_t)wn * K + k]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < GT_BK; ++k) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = As[k][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = Ws[k][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + ty * 4 + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n >= N) continue;
      float v = acc[i][j];
      if (bias) v += to_f32<T>(bias[n]);
      if (residual) {
        // the product is materialised in the storage type, then added (x + proj)
        v = round_to<T>(v) + to_f32<T>(residual[(size_t)m * ldr + n]);
      }
      C[(size_t)m * ldc + n] = from_f32<TO>(v);
    }
  }
}

// out_f32: write C as 32-bit floats whatever the storage type (the logits).
TK_API int tk_gemm_generic(int dt, const void* A, int lda, const void* W, void* C, int ldc,
                               const void* residual, int ldr, const void* bias, int M, int N, int K, int out_f32,
                               hipStream_t stream) {
  TK_REQUIRE(M >= 0 && N > 0 && K > 0 && lda >= K && ldc >= N, "gemm_generic: bad sizes M=%d N=%d K=%d lda=%d ldc=%d",
             M, N, K, lda, ldc);
  TK_REQUIRE(!residual || ldr >= N, "gemm_generic: residual stride %d < N %d", ldr, N);
  if (M == 0) return 0;
  if (M <= GR_MAX_ROWS) {
    if (dt == TK_F32)
      launch_rows<float, float>((const float*)A, lda, (const float*)W, (float*)C, ldc, (const float*)residual, ldr, (const float*)bias, M, N, K, stream);
    else if (out_f32)
      launch_rows<bf16_t, float>((const bf16_t*)A, lda, (const bf16_t*)W, (float*)C, ldc, (const bf16_t*)residual, ldr, (const bf16_t*)bias, M, N, K, stream);
    else
      launch_rows<bf16_t, bf16_t>((const bf16_t*)A, lda, (const bf16_t*)W, (bf16_t*)C, ldc, (const bf16_t*)residual, ldr, (const bf16_t*)bias, M, N, K, stream);
    TK_CHECK_LAUNCH("gemm_rows");
    return 0;
  }
  dim3 grid((N + GT_BN - 1) / GT_BN, (M + GT_BM - 1) / GT_BM);
  TK_REQUIRE(grid.y < 65536, "gemm_generic: M=%d needs too many row tiles", M);
  if (dt == TK_F32) {
    hipLaunchKernelGGL((gemm_generic_kernel<float, float>), grid, dim3(256), 0, stream,
                       (const float*)A, lda, (const float*)W, (float*)C, ldc,
                       (const float*)residual, ldr, (const float*)bias, M, N, K);
  } else if (out_f32) {
    hipLaunchKernelGGL((gemm_generic_kernel<bf16_t, float>), grid, dim3(256), 0, stream,
                       (const bf16_t*)A, lda, (const bf16_t*)W, (float*)C, ldc,
                       (const bf16_t*)residual, ldr, (const bf16_t*)bias, M, N, K);
  } else {
    hipLaunchKernelGGL((gemm_generic_kernel<bf16_t, bf16_t>), grid, dim3(256), 0, stream,
                       (const bf16_t*)A, lda, (const bf16_t*)W, (bf16_t*)C, ldc,
                       (const bf16_t*)residual, ldr, (const bf16_t*)bias, M, N, K);
  }
  TK_CHECK_LAUNCH("gemm_generic");
  return 0;
}
