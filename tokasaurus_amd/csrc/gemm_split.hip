// bfloat16 matrix products for few to 256 rows (from 17 on over 2,048 inputs, 9 with the rotation behind, 5 over 8,192, 3 over 14,336:
// ops.split_from_rows) whose outputs are too narrow to give every compute unit weights of its own:  C[M,N] = A[M,K] * W[N,K]^T with K cut among workgroups, and the passes that add the cuts.
//
// The product is bound by reading W once; at these rows the output and down projections and the stacked q, k, v product have
// 32 to 64 tiles of 64 weight rows for 256 compute units, so K is cut until there is a workgroup a unit.  What a workgroup
// finds goes to memory as 32-bit sums, [cut][row][output], and the pass that reads the product anyway (the residual sum with
// the norm behind it, the rotation with the append) adds the cuts in ascending order: no workgroup waits for another and
// every output has one order of summation.
//
// Measured on an MI355X, weights from memory, us (library's product / this one, without the passes behind them): 2,048 x 8,192
// 13.4 / 8.5 at 16 rows, 22.8 / 9.5 at 64 (33.5 MB: 3.5 TB/s, a launch's floor included), 21.2 / 12.3 at 128; 2,048 x 2,048 9.0 / 4.9
// at 64; 3,072 x 2,048 11.1 / 5.5 at 64; 4,096 x 14,336 27.2 / 21.9 at 16 (5.4 TB/s), 38.5 / 25.0 at 64, 75.3 / 33.0 at 128.  Four steps
// in local memory measured best: with 8 or 9 (144 KB) 2,048 x 8,192 takes 9.7 at 16 rows, with 3 9.1.
// From 129 rows on there are two blocks of rows, which read W twice, the second time from the caches.  With the passes, library /
// this one: 2,048 x 8,192 29.4 / 22.9 at 129 rows, 30.7 / 25.9 at 256; 2,048 x 2,048 12.6 / 12.7, 13.6 / 15.6; 4,096 x 4,096 26.3 / 23.7, 27.1 /
// 25.6; 3,072 x 2,048 with the rotation 14.7 / 16.4, 16.5 / 18.9; 5,120 x 3,072 24.9 / 24.8, 40.5 / 28.5.  In whole recorded steps, where the
// weights come from memory between other products, the short ones are ahead too: 1B decode of 192 and 256 with the output projection
// the library's / split 1,968 / 1,854 and 2,194 / 2,062 us, with q, k, v 2,081 / 1,854 and 2,172 / 2,062; 3B 5,309 / 4,761 and 5,718 / 5,358.
// With three blocks it is behind (2,048 x 2,048 14.8 / 18.1 at 300 rows, 4,096 x 14,336 75 / 91).
#include "calls.h"

#include <type_traits>

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

struct SplitArgs {
  const bf16_t* A;
  int lda;
  const bf16_t* W;
  float* part;  // [cuts][M][N]
  int M, N, K, cuts;
};

#define GS_K 64      // elements of K a step
#define GS_STAGES 4  // steps that local memory holds
#define GS_ROWS 256   // rows of A (in blocks of 128, a workgroup one)

// A workgroup of 4 wavefronts owns 64 weight rows and the steps of its cut.  W and A (16 * MB rows, the last one again behind M)
// go straight from memory to local memory STAGES - 1 steps ahead, the 16-byte piece c of row r at place c ^ (r % 8): a load
// instruction writes 8 whole rows in lane order and 16 rows read at one K meet in all banks.  Up to 64 rows every wavefront
// takes 16 weight rows and all rows of A; beyond, two wavefronts take 32 weight rows and half of A each, so that local memory
// gives 6 operands for 8 products instead of 9.
template <int MB, int NB, int STAGES>
__global__ __launch_bounds__(256) void gemm_split_kernel(SplitArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int ROWS = 64 + 16 * MB, LOADS = 2 + MB / 2;  // loads a wavefront and step
  constexpr int WM = MB > 4 ? 2 : 1, TW = WM, NW = (NB + WM - 1) / WM;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, q = lane >> 4;
  // (the cut runs fastest: with 8 cuts a die reads one eighth of A)
  const int cut = blockIdx.x % a.cuts, first = blockIdx.x / a.cuts * 64, row0 = blockIdx.y * 128;
  const int all = a.K / GS_K, s0 = (int)((long)all * cut / a.cuts), steps = (int)((long)all * (cut + 1) / a.cuts) - s0;
  bf16_t* rows = (bf16_t*)smem;
  const unsigned lds = (unsigned)(uintptr_t)(__attribute__((address_space(3))) bf16_t*)rows;
  const int lr = lane >> 3, piece = ((lane & 7) ^ lr) * 8;
  const bf16_t* src[LOADS];
#pragma unroll
  for (int i = 0; i < 2; ++i) src[i] = a.W + (size_t)min(first + wave * 16 + i * 8 + lr, a.N - 1) * a.K + (size_t)s0 * GS_K + piece;
#pragma unroll
  for (int i = 0; i < MB / 2; ++i)
    src[2 + i] = a.A + (size_t)min(row0 + (wave * (MB / 2) + i) * 8 + lr, a.M - 1) * a.lda + (size_t)s0 * GS_K + piece;
  f32x4_t acc[TW][NW];
#pragma unroll
  for (int t = 0; t < TW; ++t)
#pragma unroll
    for (int mb = 0; mb < NW; ++mb) acc[t][mb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int wn = WM == 2 ? wave >> 1 : wave, wm = WM == 2 ? wave & 1 : 0;
  // LOADS: of W's rows alone for a wavefront whose rows of A are all behind the last (what lies in their place is read into results
  // that nobody stores)
  auto walk = [&](auto loads_a_step) {
    constexpr int LOADS = decltype(loads_a_step)::value;
    auto ask = [&](int step, int place) {
      const unsigned base = lds + (unsigned)(place * ROWS * GS_K * (int)sizeof(bf16_t));
      const size_t k = (size_t)step * GS_K;
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        const int row = i < 2 ? wave * 16 + i * 8 : 64 + (wave * (MB / 2) + i - 2) * 8;
        load_to_lds(src[i] + k, base + (unsigned)(row * GS_K * (int)sizeof(bf16_t)));
      }
    };
    for (int s = 0; s < STAGES - 1 && s < steps; ++s) ask(s, s);
    int at_stage = 0, next_stage = STAGES - 1;
    for (int s = 0; s < steps; ++s) {
      // the step is there when only the loads of the STAGES - 2 behind it are left; behind the barrier every wavefront's are,
      // and every wavefront is through with the step before, whose place is filled again
      if (s + STAGES - 2 < steps) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((STAGES - 2) * LOADS) : "memory");
      else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if (s + STAGES - 1 < steps) ask(s + STAGES - 1, next_stage);
      const bf16_t* at = rows + (size_t)at_stage * ROWS * GS_K;
      at_stage = at_stage + 1 == STAGES ? 0 : at_stage + 1;
      next_stage = next_stage + 1 == STAGES ? 0 : next_stage + 1;
#pragma unroll
      for (int kk = 0; kk < GS_K / 32; ++kk) {
        const int place = ((4 * kk + q) ^ (r & 7)) * 8;
        bf16x8_t wv[TW];
#pragma unroll
        for (int t = 0; t < TW; ++t) wv[t] = *(const bf16x8_t*)(at + ((wn * TW + t) * 16 + r) * GS_K + place);
#pragma unroll
        for (int mb = 0; mb < NW; ++mb) {
          const bf16x8_t av = *(const bf16x8_t*)(at + (64 + 16 * (wm * NW + mb) + r) * GS_K + place);
#pragma unroll
          for (int t = 0; t < TW; ++t) acc[t][mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[t], av, acc[t][mb], 0, 0, 0);
        }
      }
    }
  };
  if (MB > 2 || wave * (MB / 2) * 8 < a.M - row0) walk(std::integral_constant<int, 2 + MB / 2>());
  else walk(std::integral_constant<int, 2>());
  float* out = a.part + (size_t)cut * a.M * a.N;
#pragma unroll
  for (int mb = 0; mb < NW; ++mb) {
    const int token = row0 + 16 * (wm * NW + mb) + r;
    if (token >= a.M) continue;
#pragma unroll
    for (int t = 0; t < TW; ++t) {
      const int n = first + (wn * TW + t) * 16 + 4 * q;
      if (n < a.N) *(f32x4_t*)(out + (size_t)token * a.N + n) = acc[t][mb];  // (N is a multiple of 4)
    }
  }
}

template <int MB, int NB>
static bool launch_split(const SplitArgs& a, hipStream_t stream) {
  constexpr int lds = GS_STAGES * (64 + 16 * MB) * GS_K * (int)sizeof(bf16_t);
  auto kernel = gemm_split_kernel<MB, NB, GS_STAGES>;
  if (lds > 64 * 1024 && hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) return false;
  hipLaunchKernelGGL(kernel, dim3((a.N + 63) / 64 * a.cuts, (a.M + 127) / 128), dim3(256), lds, stream, a);
  return true;
}

// part [cuts][M][N] (32-bit) = A [M, K] (rows lda apart) . W [N, K]^T over each cut of K; the sum over the cuts in ascending
// order is the product.
TK_API int tk_gemm_split_bf16(const void* A, int lda, const void* W, float* part, int M, int N, int K, int cuts, hipStream_t stream) {
  TK_REQUIRE(M >= 0 && M <= GS_ROWS && N > 0 && N % 4 == 0 && K > 0 && K % GS_K == 0, "gemm_split: bad sizes M=%d N=%d K=%d", M, N, K);
  TK_REQUIRE(cuts > 0 && cuts <= K / GS_K, "gemm_split: %d cuts of K=%d", cuts, K);
  TK_REQUIRE(lda >= K && lda % 8 == 0 && (((uintptr_t)A | (uintptr_t)W | (uintptr_t)part) & 15) == 0,
             "gemm_split: rows of A, W and the sums must be 16-byte aligned (lda=%d)", lda);
  if (M == 0) return 0;
  const SplitArgs a = {(const bf16_t*)A, lda, (const bf16_t*)W, part, M, N, K, cuts};
  const bool ok = M <= 16 ? launch_split<2, 1>(a, stream)
                          : (M <= 32 ? launch_split<2, 2>(a, stream)
                                     : (M <= 64 ? launch_split<4, 4>(a, stream) : (M <= 96 ? launch_split<6, 6>(a, stream) : launch_split<8, 8>(a, stream))));
  TK_REQUIRE(ok, "gemm_split: local memory could not be reserved");
  TK_CHECK_LAUNCH("gemm_split");
  return 0;
}

// ---------------------------------------------------------------------------------
// The passes that add the cuts
// ---------------------------------------------------------------------------------

// Both passes are bound by their chain of waits: the bytes are few, a launch takes 1.6 us, and every trip to sums that other dies
// have just written 0.8 or more.  So all that a thread reads is asked for at once: the first G cuts (of cuts that are not there
// the last one again: no branch stands between the loads) beside the residual row and the norm's weight.

// the cuts' values at `at`, 4 outputs each: the first G cuts asked for together, all added in ascending order
template <int G>
struct CutSums {
  f32x4_t v[G];
  __device__ __forceinline__ void ask(const float* part, size_t apart, int cuts, size_t at) {
#pragma unroll
    for (int c = 0; c < G; ++c) v[c] = *(const f32x4_t*)(part + min(c, cuts - 1) * apart + at);
  }
  __device__ __forceinline__ f32x4_t sum(const float* part, size_t apart, int cuts, size_t at) const {
    f32x4_t s = v[0];
#pragma unroll
    for (int c = 1; c < G; ++c)
      if (c < cuts) s += v[c];
#pragma unroll 4
    for (int c = G; c < cuts; ++c) s += *(const f32x4_t*)(part + c * apart + at);
    return s;
  }
};

// stream_out = product + residual (rounded); out = RMSNorm(stream_out) * w: a workgroup a row, the arithmetic of
// rmsnorm_packed_kernel.  A thread keeps the first HELD pieces of 8 that it takes in registers.  once: the normed value is not
// rounded in front of the weight.  Rows that few go through the weight-streaming kernel round an operand of the next product
// once (x w, the row's factor on the 32-bit sums), and keep that where the split form takes its place: 8 rows of 2,048 against
// 64 bits 1.7e-3 of the norm, rounded twice 2.4e-3.
template <int HELD, int G>
__global__ __launch_bounds__(256) void split_add_rmsnorm_kernel(const float* __restrict__ part, int cuts, const bf16_t* __restrict__ residual,
                                                                const void* __restrict__ w, int w_f32, bf16_t* __restrict__ stream_out,
                                                                bf16_t* __restrict__ out, int rows, int hidden, float eps, int once) {
  __shared__ float red[4];
  const size_t base = (size_t)blockIdx.x * hidden, apart = (size_t)rows * hidden;
  const int pieces = hidden / 8;
  CutSums<G> lo[HELD], hi[HELD];
  Pack<bf16_t> res[HELD];
  struct Weights { f32x4_t a, b; } wp[HELD];  // 8 floats, or 8 of 16 bits in `a`
  auto weights = [&](int piece) {
    const char* from = (const char*)w + (size_t)piece * (w_f32 ? 32 : 16);
    Weights v;
    v.a = *(const f32x4_t*)from;
    v.b = *(const f32x4_t*)(w_f32 ? from + 16 : from);
    return v;
  };
  auto weight = [&](const Weights& v, int j) {
    const unsigned two = __float_as_uint(v.a[j / 2]);
    const float narrow = __uint_as_float(j & 1 ? two & 0xffff0000u : two << 16);
    return w_f32 ? (j < 4 ? v.a[j & 3] : v.b[j & 3]) : narrow;
  };
#pragma unroll
  for (int c = 0; c < HELD; ++c) {
    const int piece = min((int)threadIdx.x + c * 256, pieces - 1);
    const size_t at = base + (size_t)piece * 8;
    lo[c].ask(part, apart, cuts, at);
    hi[c].ask(part, apart, cuts, at + 4);
    res[c].load(residual + at);
  }
#pragma unroll
  for (int c = 0; c < HELD; ++c) wp[c] = weights(min((int)threadIdx.x + c * 256, pieces - 1));
  float held[HELD][8];
  float ss = 0.f;
  // the product rounded as one that is stored is, + the residual, rounded
  auto take = [&](int piece, f32x4_t a, f32x4_t b, const Pack<bf16_t>& r, float (&v)[8]) {
    Pack<bf16_t> s;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      v[j] = round_to<bf16_t>(round_to<bf16_t>(j < 4 ? a[j & 3] : b[j & 3]) + to_f32<bf16_t>(r.v[j]));
      s.v[j] = from_f32<bf16_t>(v[j]);
      ss += v[j] * v[j];
    }
    s.store(stream_out + base + (size_t)piece * 8);
  };
#pragma unroll
  for (int c = 0; c < HELD; ++c) {
    const int piece = threadIdx.x + c * 256;
    const size_t at = base + (size_t)piece * 8;
    if (piece < pieces) take(piece, lo[c].sum(part, apart, cuts, at), hi[c].sum(part, apart, cuts, at + 4), res[c], held[c]);
  }
  for (int piece = threadIdx.x + HELD * 256; piece < pieces; piece += 256) {
    const size_t at = base + (size_t)piece * 8;
    Pack<bf16_t> r;
    float v[8];
    r.load(residual + at);
    lo[0].ask(part, apart, cuts, at);
    hi[0].ask(part, apart, cuts, at + 4);
    take(piece, lo[0].sum(part, apart, cuts, at), hi[0].sum(part, apart, cuts, at + 4), r, v);
  }
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  const float rstd = 1.0f / sqrtf((((0.f + red[0]) + red[1]) + red[2] + red[3]) / (float)hidden + eps);
  auto give = [&](int piece, const Weights& wv, const float (&v)[8]) {
    Pack<bf16_t> o;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      o.v[j] = from_f32<bf16_t>(weight(wv, j) * (once ? v[j] * rstd : round_to<bf16_t>(v[j] * rstd)));
    o.store(out + base + (size_t)piece * 8);
  };
#pragma unroll
  for (int c = 0; c < HELD; ++c) {
    const int piece = threadIdx.x + c * 256;
    if (piece < pieces) give(piece, wp[c], held[c]);
  }
  for (int piece = threadIdx.x + HELD * 256; piece < pieces; piece += 256) {
    Pack<bf16_t> a;
    a.load(stream_out + base + (size_t)piece * 8);  // a thread reads back what it wrote
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = to_f32<bf16_t>(a.v[j]);
    give(piece, weights(piece), v);
  }
}

TK_API int tk_split_add_rmsnorm(const float* part, int cuts, const void* residual, const void* w, int w_f32, void* stream_out, void* out,
                                int rows, int hidden, float eps, int once, hipStream_t stream) {
  TK_REQUIRE(rows >= 0 && hidden > 0 && hidden % 8 == 0 && cuts > 0, "split_add_rmsnorm: bad sizes %d %d, %d cuts", rows, hidden, cuts);
  TK_REQUIRE(part && residual && w && stream_out && out, "split_add_rmsnorm: an operand is missing");
  TK_REQUIRE((((uintptr_t)part | (uintptr_t)residual | (uintptr_t)w | (uintptr_t)stream_out | (uintptr_t)out) & 15) == 0,
             "split_add_rmsnorm: operands must be 16-byte aligned");
  TK_REQUIRE(out != residual && out != stream_out && stream_out != residual, "split_add_rmsnorm: inputs and outputs must not share a buffer");
  if (rows == 0) return 0;
  const int held = hidden <= 2048 ? 1 : (hidden <= 4096 ? 2 : 4);  // (a row in registers as far as 8,192)
  auto kernel = held == 4 ? split_add_rmsnorm_kernel<4, 4>
                          : (cuts <= 4 ? (held == 1 ? split_add_rmsnorm_kernel<1, 4> : split_add_rmsnorm_kernel<2, 4>)
                                       : (held == 1 ? split_add_rmsnorm_kernel<1, 8> : split_add_rmsnorm_kernel<2, 8>));
  hipLaunchKernelGGL(kernel, dim3(rows), dim3(256), 0, stream, part, cuts, (const bf16_t*)residual, w, w_f32,
                     (bf16_t*)stream_out, (bf16_t*)out, rows, hidden, eps, once);
  TK_CHECK_LAUNCH("split_add_rmsnorm");
  return 0;
}

// The stacked q, k, v product's cuts added, q and k rotated (element j of a head with element j + d / 2; without tables they
// pass as they are), q to `q` [rows, nq * d], k and v to the token's page.  A workgroup a token and `share` of its units, a
// unit 4 neighbouring columns of one half of a head and the same 4 of the other.
template <int G>
__global__ __launch_bounds__(256) void split_rope_append_kernel(const float* __restrict__ part, int cuts, bf16_t* __restrict__ q,
                                                                const int* __restrict__ positions, const int* __restrict__ token_req,
                                                                const int* __restrict__ block_table, int table_stride,
                                                                const float* __restrict__ cos_t, const float* __restrict__ sin_t,
                                                                bf16_t* __restrict__ kcache, bf16_t* __restrict__ vcache, int rows, int nq,
                                                                int nkv, int d, int P) {
  const int t = blockIdx.x, half = d >> 1, each = half >> 2;
  const int u = blockIdx.y * 256 + threadIdx.x;
  if (u >= (nq + 2 * nkv) * each) return;
  const int h = u / each, c = (u - h * each) * 4;
  const int width = (nq + 2 * nkv) * d;
  const size_t apart = (size_t)rows * width, at = (size_t)t * width + h * d + c;
  // (positions and requests first: what they lead to is asked for while the sums are on their way)
  const int pos = positions[t], req = token_req[t];
  CutSums<G> slo, shi;
  slo.ask(part, apart, cuts, at);
  shi.ask(part, apart, cuts, at + half);
  f32x4_t cs = {1.f, 1.f, 1.f, 1.f}, sn = {0.f, 0.f, 0.f, 0.f};
  const bool rotate = h < nq + nkv && cos_t != nullptr;
  if (rotate) {
    cs = *(const f32x4_t*)(cos_t + (size_t)pos * half + c);
    sn = *(const f32x4_t*)(sin_t + (size_t)pos * half + c);
  }
  const int page = h >= nq ? block_table[(size_t)req * table_stride + pos / P] : 0;
  const f32x4_t lo = slo.sum(part, apart, cuts, at), hi = shi.sum(part, apart, cuts, at + half);
  union { bf16_t h[4]; uint2 u; } o1, o2;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float a = round_to<bf16_t>(lo[j]), b = round_to<bf16_t>(hi[j]);
    if (rotate) {
      float ra, rb;
      rotate_pair(a, b, cs[j], sn[j], ra, rb);
      a = ra;
      b = rb;
    }
    o1.h[j] = from_f32<bf16_t>(a);
    o2.h[j] = from_f32<bf16_t>(b);
  }
  const int off = pos % P;
  if (h < nq) {
    bf16_t* dst = q + (size_t)t * nq * d + h * d + c;
    *(uint2*)dst = o1.u;
    *(uint2*)(dst + half) = o2.u;
  } else if (h < nq + nkv) {
    bf16_t* dst = kcache + ((size_t)page * nkv + (h - nq)) * P * d;
    *(uint2*)(dst + key_offset(P, off, c)) = o1.u;  // (4 of a key's pieces of 8)
    *(uint2*)(dst + key_offset(P, off, c + half)) = o2.u;
  } else {
    bf16_t* dst = vcache + ((size_t)page * nkv + (h - nq - nkv)) * P * d;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      dst[value_offset(d, off, c + j)] = o1.h[j];
      dst[value_offset(d, off, c + half + j)] = o2.h[j];
    }
  }
}

TK_API int tk_split_rope_append(const float* part, int cuts, void* q, const int* positions, const int* token_req, const int* block_table,
                                int table_stride, const float* cos_t, const float* sin_t, void* kcache, void* vcache, int rows, int nq,
                                int nkv, int d, int P, hipStream_t stream) {
  TK_REQUIRE(rows >= 0 && cuts > 0 && nq > 0 && nkv > 0 && d > 0 && d % 8 == 0 && P > 0, "split_rope_append: bad sizes rows=%d nq=%d nkv=%d d=%d P=%d",
             rows, nq, nkv, d, P);
  TK_REQUIRE(part && q && positions && token_req && block_table && kcache && vcache, "split_rope_append: an operand is missing");
  TK_REQUIRE((cos_t == nullptr) == (sin_t == nullptr), "split_rope_append: cos and sin tables go together");
  TK_REQUIRE((((uintptr_t)part | (uintptr_t)q | (uintptr_t)cos_t | (uintptr_t)sin_t | (uintptr_t)kcache | (uintptr_t)vcache) & 15) == 0,
             "split_rope_append: operands must be 16-byte aligned");
  if (rows == 0) return 0;
  const int units = (nq + 2 * nkv) * (d / 8);
  auto kernel = cuts <= 4 ? split_rope_append_kernel<4> : split_rope_append_kernel<8>;
  hipLaunchKernelGGL(kernel, dim3(rows, (units + 255) / 256), dim3(256), 0, stream, part, cuts, (bf16_t*)q, positions,
                     token_req, block_table, table_stride, cos_t, sin_t, (bf16_t*)kcache, (bf16_t*)vcache, rows, nq, nkv, d, P);
  TK_CHECK_LAUNCH("split_rope_append");
  return 0;
}

// ---------------------------------------------------------------------------------
// A product and the pass behind it in one call of the host, which in steps of few tokens is what bounds them: a call from Python
// with its checks and its launch takes 8 us or more, a launch from here 2.
// ---------------------------------------------------------------------------------

TK_API int tk_split_linear_add_rmsnorm(const void* A, int lda, const void* W, float* part, int M, int N, int K, int cuts, const void* residual,
                                       const void* w, int w_f32, void* stream_out, void* out, float eps, int once, hipStream_t stream) {
  const int rc = tk_gemm_split_bf16(A, lda, W, part, M, N, K, cuts, stream);
  return rc ? rc : tk_split_add_rmsnorm(part, cuts, residual, w, w_f32, stream_out, out, M, N, eps, once, stream);
}

TK_API int tk_split_linear_rope_append(const void* A, int lda, const void* W, float* part, int M, int K, int cuts, void* q, const int* positions,
                                       const int* token_req, const int* block_table, int table_stride, const float* cos_t,
                                       const float* sin_t, void* kcache, void* vcache, int nq, int nkv, int d, int P, hipStream_t stream) {
  const int rc = tk_gemm_split_bf16(A, lda, W, part, M, (nq + 2 * nkv) * d, K, cuts, stream);
  return rc ? rc
            : tk_split_rope_append(part, cuts, q, positions, token_req, block_table, table_stride, cos_t, sin_t, kcache, vcache, M, nq, nkv, d, P,
                                   stream);
}
