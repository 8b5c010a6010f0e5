// Memory-bound kernels of the step: embedding gather, RMSNorm, SwiGLU, row
// gather, the rotary tables, and rotation fused with the append to the paged cache.
// Every kernel is a template over the storage type (float or bfloat16) and
// computes in 32-bit.
#include "calls.h"

// --------------------------------------------------------------------------
// embedding: out[t, :] = table[id_t, :]; id_t < 0 names slot -id_t-1 of `last_token`
// (the token the sampler wrote there in the step before).
// --------------------------------------------------------------------------
template <typename T>
__global__ void embed_gather_kernel(const int* __restrict__ ids, const int* __restrict__ last_token,
                                    const T* __restrict__ table, T* __restrict__ out, int hidden,
                                    int vocab) {
  const int t = blockIdx.x;
  int id = ids[t];
  if (id < 0) id = last_token[-id - 1];
  id = min(max(id, 0), vocab - 1);
  const T* src = table + (size_t)id * hidden;
  T* dst = out + (size_t)t * hidden;
  for (int i = threadIdx.x; i < hidden; i += blockDim.x) dst[i] = src[i];
}

TK_API int tk_embed_gather(int dt, const int* ids, const int* last_token, const void* table,
                               void* out, int n_tokens, int hidden, int vocab, hipStream_t stream) {
  TK_REQUIRE(n_tokens >= 0 && hidden > 0 && vocab > 0, "embed_gather: bad sizes %d %d %d", n_tokens,
             hidden, vocab);
  if (n_tokens == 0) return 0;
  if (dt == TK_F32)
    hipLaunchKernelGGL(embed_gather_kernel<float>, dim3(n_tokens), dim3(256), 0, stream, ids,
                       last_token, (const float*)table, (float*)out, hidden, vocab);
  else
    hipLaunchKernelGGL(embed_gather_kernel<bf16_t>, dim3(n_tokens), dim3(256), 0, stream, ids,
                       last_token, (const bf16_t*)table, (bf16_t*)out, hidden, vocab);
  TK_CHECK_LAUNCH("embed_gather");
  return 0;
}

static bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// --------------------------------------------------------------------------
// RMSNorm: statistics in 32-bit, the normalised value rounded to the storage
// type, then multiplied by the weight and rounded again.  The weight is of the
// storage type, or 32-bit when `w_f32` (then the product is rounded once more only).
// With ADD the rows are first x + residual (rounded), which is also written out:
// the residual stream and its norm in one pass.
// --------------------------------------------------------------------------
template <typename T, bool ADD>
__global__ void rmsnorm_kernel(const T* __restrict__ x, const T* __restrict__ residual,
                               const void* __restrict__ w, int w_f32, T* __restrict__ stream_out,
                               T* __restrict__ out, int hidden, float eps) {
  __shared__ float red[16];
  const T* row = x + (size_t)blockIdx.x * hidden;
  const T* rrow = ADD ? residual + (size_t)blockIdx.x * hidden : nullptr;
  T* srow = ADD ? stream_out + (size_t)blockIdx.x * hidden : nullptr;
  T* orow = out + (size_t)blockIdx.x * hidden;
  float ss = 0.f;
  for (int i = threadIdx.x; i < hidden; i += blockDim.x) {
    float v = to_f32<T>(row[i]);
    if (ADD) {
      v = round_to<T>(v + to_f32<T>(rrow[i]));
      srow[i] = from_f32<T>(v);
    }
    ss += v * v;
  }
  ss = block_sum(ss, red);
  const float rstd = 1.0f / sqrtf(ss / (float)hidden + eps);
  for (int i = threadIdx.x; i < hidden; i += blockDim.x) {
    float n = round_to<T>(to_f32<T>(ADD ? srow[i] : row[i]) * rstd);  // a thread reads back what it wrote
    float wi = w_f32 ? ((const float*)w)[i] : to_f32<T>(((const T*)w)[i]);
    orow[i] = from_f32<T>(wi * n);
  }
}

// The same with 16-byte accesses; a thread keeps its first HELD pieces of the row in registers.  For few rows the kernel is its chain
// of waits: all of a thread's pieces, the residual's and the weight's are asked for at once, before each piece was waited for by itself and
// the weight behind the sum (before / now, alone and with the residual: 4 rows of 2,048 in 32-bit 2.72 and 2.82 us / 2.29 and 2.36, 4
// of 4,096 in bfloat16 2.98 and 3.24 / 2.59 and 2.70).  Many rows are bound by memory (4,096 of 4,096 13.4 and 20.3 / 11.9 and 20.4; 134 MB
// with the residual, 6.6 TB/s with its share in the caches).
template <typename T, bool ADD, int HELD>
__global__ __launch_bounds__(256) void rmsnorm_packed_kernel(
    const T* __restrict__ x, const T* __restrict__ residual, const void* __restrict__ w, int w_f32,
    T* __restrict__ stream_out, T* __restrict__ out, int hidden, float eps) {
  constexpr int N = Pack<T>::N;
  __shared__ float red[16];
  const size_t base = (size_t)blockIdx.x * hidden;
  const int pieces = hidden / N;
  struct Weights { unsigned word[8]; };  // N weights of the storage type in the first four, or N floats
  auto weights = [&](int piece) {
    const char* from = (const char*)w + (size_t)piece * (w_f32 ? N * 4 : 16);
    const uint4 a = *(const uint4*)from;
    uint4 b = {};  // (a copy of `a` here would be waited for)
    if (N == 8 && w_f32) b = *(const uint4*)(from + 16);
    return Weights{{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w}};
  };
  auto weight = [&](const Weights& v, int j) {
    if (N == 4) return __uint_as_float(v.word[j]);
    const unsigned two = v.word[j / 2];
    return __uint_as_float(w_f32 ? v.word[j] : (j & 1 ? two & 0xffff0000u : two << 16));
  };
  Pack<T> xp[HELD], rp[HELD];
  Weights wp[HELD];
#pragma unroll
  for (int c = 0; c < HELD; ++c) {  // (behind the row's end: its last piece again, so that no branch stands between the loads)
    const size_t at = base + (size_t)min((int)threadIdx.x + c * 256, pieces - 1) * N;
    xp[c].load(x + at);
    if (ADD) rp[c].load(residual + at);
  }
#pragma unroll
  for (int c = 0; c < HELD; ++c) wp[c] = weights(min((int)threadIdx.x + c * 256, pieces - 1));
  float held[HELD][N];
  float ss = 0.f;
  auto take = [&](int piece, const Pack<T>& a, const Pack<T>& r, float (&v)[N]) {
    if (ADD) {
      Pack<T> s;
#pragma unroll
      for (int j = 0; j < N; ++j) {
        v[j] = round_to<T>(to_f32<T>(a.v[j]) + to_f32<T>(r.v[j]));
        s.v[j] = from_f32<T>(v[j]);
      }
      s.store(stream_out + base + (size_t)piece * N);
    } else {
#pragma unroll
      for (int j = 0; j < N; ++j) v[j] = to_f32<T>(a.v[j]);
    }
#pragma unroll
    for (int j = 0; j < N; ++j) ss += v[j] * v[j];
  };
#pragma unroll
  for (int c = 0; c < HELD; ++c) {
    const int piece = threadIdx.x + c * 256;
    if (piece < pieces) take(piece, xp[c], rp[c], held[c]);
  }
  for (int piece = threadIdx.x + HELD * 256; piece < pieces; piece += 256) {
    Pack<T> a, r;
    float v[N];
    a.load(x + base + (size_t)piece * N);
    if (ADD) r.load(residual + base + (size_t)piece * N);
    take(piece, a, r, v);
  }
  ss = block_sum(ss, red);
  const float rstd = 1.0f / sqrtf(ss / (float)hidden + eps);
  auto give = [&](int piece, const Weights& wv, const float (&v)[N]) {
    Pack<T> o;
#pragma unroll
    for (int j = 0; j < N; ++j) o.v[j] = from_f32<T>(weight(wv, j) * round_to<T>(v[j] * rstd));
    o.store(out + base + (size_t)piece * N);
  };
#pragma unroll
  for (int c = 0; c < HELD; ++c) {
    const int piece = threadIdx.x + c * 256;
    if (piece < pieces) give(piece, wp[c], held[c]);
  }
  for (int piece = threadIdx.x + HELD * 256; piece < pieces; piece += 256) {
    Pack<T> a;
    a.load((ADD ? stream_out : x) + base + (size_t)piece * N);  // a thread reads back what it wrote
    float v[N];
#pragma unroll
    for (int j = 0; j < N; ++j) v[j] = to_f32<T>(a.v[j]);
    give(piece, weights(piece), v);
  }
}

template <typename T, bool ADD>
static void launch_rmsnorm(const void* x, const void* residual, const void* w, int w_f32, void* stream_out,
                           void* out, int rows, int hidden, float eps, hipStream_t stream) {
  constexpr int N = Pack<T>::N;
  const bool packed = hidden % N == 0 && aligned16(x) && aligned16(out) && aligned16(w) &&
                      (!ADD || (aligned16(residual) && aligned16(stream_out)));
  if (packed) {
    // as many pieces as a row has: pieces that are held but not there would be asked for all the same
    auto kernel = hidden <= 256 * N ? rmsnorm_packed_kernel<T, ADD, 1> : (hidden <= 512 * N ? rmsnorm_packed_kernel<T, ADD, 2> : rmsnorm_packed_kernel<T, ADD, 4>);
    hipLaunchKernelGGL(kernel, dim3(rows), dim3(256), 0, stream, (const T*)x, (const T*)residual, w, sizeof(T) == 4 ? 1 : w_f32, (T*)stream_out,
                       (T*)out, hidden, eps);
  } else {
    hipLaunchKernelGGL((rmsnorm_kernel<T, ADD>), dim3(rows), dim3(256), 0, stream, (const T*)x,
                       (const T*)residual, w, w_f32, (T*)stream_out, (T*)out, hidden, eps);
  }
}

TK_API int tk_rmsnorm(int dt, const void* x, const void* w, int w_f32, void* out, int rows,
                          int hidden, float eps, hipStream_t stream) {
  TK_REQUIRE(rows >= 0 && hidden > 0, "rmsnorm: bad sizes %d %d", rows, hidden);
  if (rows == 0) return 0;
  if (dt == TK_F32)
    launch_rmsnorm<float, false>(x, nullptr, w, w_f32, nullptr, out, rows, hidden, eps, stream);
  else
    launch_rmsnorm<bf16_t, false>(x, nullptr, w, w_f32, nullptr, out, rows, hidden, eps, stream);
  TK_CHECK_LAUNCH("rmsnorm");
  return 0;
}

// stream_out = x + residual (rounded); out = RMSNorm(stream_out) * w.  Four buffers, none shared.
TK_API int tk_add_rmsnorm(int dt, const void* x, const void* residual, const void* w, int w_f32,
                          void* stream_out, void* out, int rows, int hidden, float eps, hipStream_t stream) {
  TK_REQUIRE(rows >= 0 && hidden > 0, "add_rmsnorm: bad sizes %d %d", rows, hidden);
  TK_REQUIRE(x && residual && stream_out && out && w, "add_rmsnorm: an operand is missing");
  TK_REQUIRE(out != x && out != residual && out != stream_out && stream_out != x && stream_out != residual,
             "add_rmsnorm: inputs and outputs must not share a buffer");
  if (rows == 0) return 0;
  if (dt == TK_F32)
    launch_rmsnorm<float, true>(x, residual, w, w_f32, stream_out, out, rows, hidden, eps, stream);
  else
    launch_rmsnorm<bf16_t, true>(x, residual, w, w_f32, stream_out, out, rows, hidden, eps, stream);
  TK_CHECK_LAUNCH("add_rmsnorm");
  return 0;
}

// --------------------------------------------------------------------------
// SwiGLU on a fused [rows, 2*inter] product laid out [gate | up]:
// out = round(round(silu(gate)) * up).
// --------------------------------------------------------------------------
template <typename T>
__global__ void swiglu_kernel(const T* __restrict__ gu, T* __restrict__ out, int inter) {
  const T* g = gu + (size_t)blockIdx.y * 2 * inter;
  const T* u = g + inter;
  T* o = out + (size_t)blockIdx.y * inter;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < inter) {
    float gv = to_f32<T>(g[i]);
    float s = round_to<T>(gv / (1.0f + expf(-gv)));
    o[i] = from_f32<T>(s * to_f32<T>(u[i]));
  }
}

template <typename T>
__global__ __launch_bounds__(256) void swiglu_packed_kernel(const T* __restrict__ gu, T* __restrict__ out, int inter) {
  constexpr int N = Pack<T>::N;
  const int piece = blockIdx.x * blockDim.x + threadIdx.x;
  if (piece >= inter / N) return;
  const T* g = gu + (size_t)blockIdx.y * 2 * inter + (size_t)piece * N;
  Pack<T> gv, uv, o;
  gv.load(g);
  uv.load(g + inter);
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const float x = to_f32<T>(gv.v[j]);
    const float s = round_to<T>(x / (1.0f + expf(-x)));
    o.v[j] = from_f32<T>(s * to_f32<T>(uv.v[j]));
  }
  o.store(out + (size_t)blockIdx.y * inter + (size_t)piece * N);
}

template <typename T>
static void launch_swiglu(const void* gate_up, void* out, int rows, int inter, hipStream_t stream) {
  constexpr int N = Pack<T>::N;
  if (inter % N == 0 && aligned16(gate_up) && aligned16(out))
    hipLaunchKernelGGL(swiglu_packed_kernel<T>, dim3((inter / N + 255) / 256, rows), dim3(256), 0, stream,
                       (const T*)gate_up, (T*)out, inter);
  else
    hipLaunchKernelGGL(swiglu_kernel<T>, dim3((inter + 255) / 256, rows), dim3(256), 0, stream,
                       (const T*)gate_up, (T*)out, inter);
}

TK_API int tk_swiglu(int dt, const void* gate_up, void* out, int rows, int inter,
                         hipStream_t stream) {
  TK_REQUIRE(rows >= 0 && inter > 0, "swiglu: bad sizes %d %d", rows, inter);
  TK_REQUIRE(rows < 65536, "swiglu: %d rows are too many for one call", rows);
  if (rows == 0) return 0;
  if (dt == TK_F32)
    launch_swiglu<float>(gate_up, out, rows, inter, stream);
  else
    launch_swiglu<bf16_t>(gate_up, out, rows, inter, stream);
  TK_CHECK_LAUNCH("swiglu");
  return 0;
}

// --------------------------------------------------------------------------
// A gated feed-forward's activation with clamps, on a fused [rows, 2*inter] product laid out
// [gate | up]:  g = min(gate, limit), u = clamp(up, -limit, limit),
//               out = g * sigmoid(alpha * g) * (u + 1), computed in 32-bit and rounded once.
// --------------------------------------------------------------------------
template <typename T>
__global__ void clamped_glu_kernel(const T* __restrict__ gu, T* __restrict__ out, int inter, float limit, float alpha) {
  const T* g = gu + (size_t)blockIdx.y * 2 * inter;
  const T* u = g + inter;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < inter) {
    const float gv = fminf(to_f32<T>(g[i]), limit);
    const float uv = fminf(fmaxf(to_f32<T>(u[i]), -limit), limit);
    out[(size_t)blockIdx.y * inter + i] = from_f32<T>(gv / (1.0f + expf(-alpha * gv)) * (uv + 1.0f));
  }
}

template <typename T>
__global__ __launch_bounds__(256) void clamped_glu_packed_kernel(const T* __restrict__ gu, T* __restrict__ out, int inter, float limit,
                                                                 float alpha) {
  constexpr int N = Pack<T>::N;
  const int piece = blockIdx.x * blockDim.x + threadIdx.x;
  if (piece >= inter / N) return;
  const T* g = gu + (size_t)blockIdx.y * 2 * inter + (size_t)piece * N;
  Pack<T> gv, uv, o;
  gv.load(g);
  uv.load(g + inter);
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const float x = fminf(to_f32<T>(gv.v[j]), limit);
    const float y = fminf(fmaxf(to_f32<T>(uv.v[j]), -limit), limit);
    o.v[j] = from_f32<T>(x / (1.0f + expf(-alpha * x)) * (y + 1.0f));
  }
  o.store(out + (size_t)blockIdx.y * inter + (size_t)piece * N);
}

template <typename T>
static void launch_clamped_glu(const void* gate_up, void* out, int rows, int inter, float limit, float alpha, hipStream_t stream) {
  constexpr int N = Pack<T>::N;
  if (inter % N == 0 && aligned16(gate_up) && aligned16(out))
    hipLaunchKernelGGL(clamped_glu_packed_kernel<T>, dim3((inter / N + 255) / 256, rows), dim3(256), 0, stream,
                       (const T*)gate_up, (T*)out, inter, limit, alpha);
  else
    hipLaunchKernelGGL(clamped_glu_kernel<T>, dim3((inter + 255) / 256, rows), dim3(256), 0, stream,
                       (const T*)gate_up, (T*)out, inter, limit, alpha);
}

// gelu(gate) * up with the tanh form of gelu, [rows, 2I] laid out [gate | up] -> [rows, I]; 32-bit arithmetic, one rounding
__device__ __forceinline__ float gelu_tanh_f32(float z) {
  return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
}
template <typename T>
__global__ void gelu_glu_kernel(const T* __restrict__ gu, T* __restrict__ out, int inter) {
  const T* g = gu + (size_t)blockIdx.y * 2 * inter;
  const T* u = g + inter;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < inter) out[(size_t)blockIdx.y * inter + i] = from_f32<T>(gelu_tanh_f32(to_f32<T>(g[i])) * to_f32<T>(u[i]));
}

// (16 bytes a load where sizes and addresses allow)
template <typename T>
__global__ __launch_bounds__(256) void gelu_glu_packed_kernel(const T* __restrict__ gu, T* __restrict__ out, int inter) {
  constexpr int N = Pack<T>::N;
  const int piece = blockIdx.x * blockDim.x + threadIdx.x;
  if (piece >= inter / N) return;
  const T* g = gu + (size_t)blockIdx.y * 2 * inter + (size_t)piece * N;
  Pack<T> gv, uv, o;
  gv.load(g);
  uv.load(g + inter);
#pragma unroll
  for (int j = 0; j < N; ++j) o.v[j] = from_f32<T>(gelu_tanh_f32(to_f32<T>(gv.v[j])) * to_f32<T>(uv.v[j]));
  o.store(out + (size_t)blockIdx.y * inter + (size_t)piece * N);
}

template <typename T>
static void launch_gelu_glu(const void* gate_up, void* out, int rows, int inter, hipStream_t stream) {
  constexpr int N = Pack<T>::N;
  if (inter % N == 0 && aligned16(gate_up) && aligned16(out))
    hipLaunchKernelGGL(gelu_glu_packed_kernel<T>, dim3((inter / N + 255) / 256, rows), dim3(256), 0, stream, (const T*)gate_up,
                       (T*)out, inter);
  else
    hipLaunchKernelGGL(gelu_glu_kernel<T>, dim3((inter + 255) / 256, rows), dim3(256), 0, stream, (const T*)gate_up, (T*)out, inter);
}

TK_API int tk_gelu_glu(int dt, const void* gate_up, void* out, int rows, int inter, hipStream_t stream) {
  TK_REQUIRE(rows >= 0 && inter > 0, "gelu_glu: bad sizes %d %d", rows, inter);
  TK_REQUIRE(rows < 65536, "gelu_glu: %d rows are too many for one call", rows);
  if (rows == 0) return 0;
  if (dt == TK_F32)
    launch_gelu_glu<float>(gate_up, out, rows, inter, stream);
  else
    launch_gelu_glu<bf16_t>(gate_up, out, rows, inter, stream);
  TK_CHECK_LAUNCH("gelu_glu");
  return 0;
}

TK_API int tk_clamped_glu(int dt, const void* gate_up, void* out, int rows, int inter, float limit, float alpha,
                          hipStream_t stream) {
  TK_REQUIRE(rows >= 0 && inter > 0 && limit > 0.f, "clamped_glu: bad sizes %d %d or limit", rows, inter);
  TK_REQUIRE(rows < 65536, "clamped_glu: %d rows are too many for one call", rows);
  if (rows == 0) return 0;
  if (dt == TK_F32)
    launch_clamped_glu<float>(gate_up, out, rows, inter, limit, alpha, stream);
  else
    launch_clamped_glu<bf16_t>(gate_up, out, rows, inter, limit, alpha, stream);
  TK_CHECK_LAUNCH("clamped_glu");
  return 0;
}

// --------------------------------------------------------------------------
// gather_rows: out[i, :] = src[idx[i], :]   (src rows `src_stride` elements apart)
// --------------------------------------------------------------------------
template <typename T>
__global__ void gather_rows_kernel(const T* __restrict__ src, int src_stride,
                                   const int* __restrict__ idx, T* __restrict__ out, int width) {
  const T* s = src + (size_t)idx[blockIdx.x] * src_stride;
  T* o = out + (size_t)blockIdx.x * width;
  for (int i = threadIdx.x; i < width; i += blockDim.x) o[i] = s[i];
}

TK_API int tk_gather_rows(int dt, const void* src, int src_stride, const int* idx, void* out,
                              int n, int width, hipStream_t stream) {
  TK_REQUIRE(n >= 0 && width > 0 && src_stride >= width, "gather_rows: bad sizes %d %d %d", n,
             width, src_stride);
  if (n == 0) return 0;
  if (dt == TK_F32)
    hipLaunchKernelGGL(gather_rows_kernel<float>, dim3(n), dim3(256), 0, stream, (const float*)src,
                       src_stride, idx, (float*)out, width);
  else
    hipLaunchKernelGGL(gather_rows_kernel<bf16_t>, dim3(n), dim3(256), 0, stream,
                       (const bf16_t*)src, src_stride, idx, (bf16_t*)out, width);
  TK_CHECK_LAUNCH("gather_rows");
  return 0;
}

// --------------------------------------------------------------------------
// Rotary tables: cos/sin[p, j] = cos/sin(p * inv_freq[j]) for j < half, 32-bit.
// --------------------------------------------------------------------------
__global__ void rope_table_kernel(const float* __restrict__ inv_freq, float* __restrict__ cos_t,
                                  float* __restrict__ sin_t, int n_pos, int half) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_pos * half) return;
  const int p = i / half, j = i % half;
  const float angle = (float)p * inv_freq[j];
  cos_t[i] = cosf(angle);
  sin_t[i] = sinf(angle);
}

TK_API int tk_rope_table(const float* inv_freq, float* cos_t, float* sin_t, int n_pos, int half,
                             hipStream_t stream) {
  TK_REQUIRE(n_pos > 0 && half > 0, "rope_table: bad sizes %d %d", n_pos, half);
  const long total = (long)n_pos * half;
  TK_REQUIRE(total < (1l << 31), "rope_table: table of %ld entries is too large", total);
  hipLaunchKernelGGL(rope_table_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream,
                     inv_freq, cos_t, sin_t, n_pos, half);
  TK_CHECK_LAUNCH("rope_table");
  return 0;
}

// --------------------------------------------------------------------------
// rope_append: for each token rotate its query heads in place, rotate its key
// heads and store them, and store its value heads, in the token's page.
//   qkv row: [nq*d | nkv*d | nkv*d]  (only the first part when !write_cache)
//   K pages: [page][kv head][d / 8][P][8]    V pages: [page][kv head][P / 4][d][4]
//   (key_offset and value_offset of common.h)
// The first `rot` elements of a head are rotated (rot = d: the whole head): element j pairs with
// element j + rot/2, and the tables have rot/2 entries a position; the elements from `rot` on
// pass as they are.  The rotation is computed in 32-bit.
// When cos_t is null the heads are stored unrotated (no position encoding).
// One workgroup a token, an element (pair) a thread: a variant that moved 16 bytes a thread
// was measured no faster (12.5 against 11.5 us for 2,048 tokens of the 1B shape): the
// kernel waits for its chain of loads (position, table entry, row), not for its bytes.
// --------------------------------------------------------------------------
template <typename T>
__global__ void rope_append_kernel(T* __restrict__ qkv, int row_stride,
                                   const int* __restrict__ positions,
                                   const int* __restrict__ token_req,
                                   const int* __restrict__ block_table, int table_stride,
                                   const float* __restrict__ cos_t, const float* __restrict__ sin_t,
                                   T* __restrict__ kcache, T* __restrict__ vcache, int nq, int nkv,
                                   int d, int rot, int P, int write_cache) {
  const int t = blockIdx.x;
  const int pos = positions[t];
  const int half = rot / 2;
  T* row = qkv + (size_t)t * row_stride;
  const float* c = cos_t ? cos_t + (size_t)pos * half : nullptr;
  const float* s = sin_t ? sin_t + (size_t)pos * half : nullptr;

  // queries, in place
  for (int i = threadIdx.x; i < nq * half; i += blockDim.x) {
    const int h = i / half, j = i % half;
    T* x = row + h * d;
    const float x1 = to_f32<T>(x[j]), x2 = to_f32<T>(x[j + half]);
    const float cj = c ? c[j] : 1.f, sj = s ? s[j] : 0.f;
    float o1, o2;
    rotate_pair(x1, x2, cj, sj, o1, o2);
    x[j] = from_f32<T>(o1);
    x[j + half] = from_f32<T>(o2);
  }
  if (!write_cache) return;

  const int page = block_table[(size_t)token_req[t] * table_stride + pos / P];
  const int p = pos % P;
  const T* krow = row + nq * d;
  const T* vrow = krow + nkv * d;
  for (int i = threadIdx.x; i < nkv * half; i += blockDim.x) {
    const int h = i / half, j = i % half;
    const float x1 = to_f32<T>(krow[h * d + j]), x2 = to_f32<T>(krow[h * d + j + half]);
    const float cj = c ? c[j] : 1.f, sj = s ? s[j] : 0.f;
    T* dst = kcache + ((size_t)page * nkv + h) * P * d;
    float o1, o2;
    rotate_pair(x1, x2, cj, sj, o1, o2);
    dst[key_offset(P, p, j)] = from_f32<T>(o1);
    dst[key_offset(P, p, j + half)] = from_f32<T>(o2);
  }
  for (int i = threadIdx.x; i < nkv * (d - rot); i += blockDim.x) {  // the part of a key that is not rotated
    const int h = i / (d - rot), e = rot + i % (d - rot);
    kcache[((size_t)page * nkv + h) * P * d + key_offset(P, p, e)] = krow[h * d + e];
  }
  for (int i = threadIdx.x; i < nkv * d; i += blockDim.x) {
    const int h = i / d, e = i % d;
    vcache[((size_t)page * nkv + h) * P * d + value_offset(d, p, e)] = vrow[i];
  }
}

TK_API int tk_rope_append(int dt, void* qkv, int row_stride, const int* positions,
                              const int* token_req, const int* block_table, int table_stride,
                              const float* cos_t, const float* sin_t, void* kcache, void* vcache,
                              int n_tokens, int nq, int nkv, int d, int rot, int P, int write_cache,
                              hipStream_t stream) {
  TK_REQUIRE(n_tokens >= 0 && nq > 0 && nkv >= 0 && d > 0 && d % 2 == 0 && P > 0,
             "rope_append: bad sizes tokens=%d nq=%d nkv=%d d=%d P=%d", n_tokens, nq, nkv, d, P);
  TK_REQUIRE(rot >= 0 && rot <= d && rot % 2 == 0, "rope_append: %d rotated elements of a head of %d", rot, d);
  TK_REQUIRE(row_stride >= (write_cache ? (nq + 2 * nkv) * d : nq * d),
             "rope_append: row stride %d is shorter than the heads it holds", row_stride);
  TK_REQUIRE(!write_cache || (kcache && vcache && block_table),
             "rope_append: cache pointers missing");
  if (n_tokens == 0) return 0;
  if (dt == TK_F32)
    hipLaunchKernelGGL(rope_append_kernel<float>, dim3(n_tokens), dim3(256), 0, stream,
                       (float*)qkv, row_stride, positions, token_req, block_table, table_stride,
                       cos_t, sin_t, (float*)kcache, (float*)vcache, nq, nkv, d, rot, P, write_cache);
  else
    hipLaunchKernelGGL(rope_append_kernel<bf16_t>, dim3(n_tokens), dim3(256), 0, stream,
                       (bf16_t*)qkv, row_stride, positions, token_req, block_table, table_stride,
                       cos_t, sin_t, (bf16_t*)kcache, (bf16_t*)vcache, nq, nkv, d, rot, P, write_cache);
  TK_CHECK_LAUNCH("rope_append");
  return 0;
}

// --------------------------------------------------------------------------
// head_rmsnorm: RMSNorm of every head's d elements in place, for `heads` heads of each row that
// start at column `first_col` (the query heads, or the key heads, of a stacked q|k|v row before
// the rotation); one weight [d] for all heads.  A wavefront a (row, head); the arithmetic of
// rmsnorm_kernel (statistics in 32-bit, the normalised value rounded before the weight).
// --------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void head_rmsnorm_kernel(T* __restrict__ x, int row_stride, const void* __restrict__ w,
                                                           int w_f32, int rows, int first_col, int heads, int d, float eps) {
  const int lane = threadIdx.x & (TK_WAVE - 1);
  const long unit = (long)blockIdx.x * (blockDim.x / TK_WAVE) + threadIdx.x / TK_WAVE;
  if (unit >= (long)rows * heads) return;
  const int row = (int)(unit / heads), head = (int)(unit % heads);
  T* p = x + (size_t)row * row_stride + first_col + (size_t)head * d;
  float ss = 0.f;
  for (int i = lane; i < d; i += TK_WAVE) {
    const float v = to_f32<T>(p[i]);
    ss += v * v;
  }
  ss = wave_sum(ss);
  const float rstd = 1.0f / sqrtf(ss / (float)d + eps);
  for (int i = lane; i < d; i += TK_WAVE) {
    const float n = round_to<T>(to_f32<T>(p[i]) * rstd);
    const float wi = w_f32 ? ((const float*)w)[i] : to_f32<T>(((const T*)w)[i]);
    p[i] = from_f32<T>(wi * n);
  }
}

TK_API int tk_head_rmsnorm(int dt, void* x, int row_stride, const void* w, int w_f32, int rows, int first_col, int heads,
                           int d, float eps, hipStream_t stream) {
  TK_REQUIRE(rows >= 0 && heads > 0 && d > 0 && first_col >= 0 && row_stride >= first_col + heads * d,
             "head_rmsnorm: bad sizes rows=%d first_col=%d heads=%d d=%d stride=%d", rows, first_col, heads, d, row_stride);
  const long units = (long)rows * heads;
  if (units == 0) return 0;
  TK_REQUIRE(units < (1l << 31), "head_rmsnorm: too many heads to norm");
  const unsigned blocks = (unsigned)((units + 3) / 4);
  if (dt == TK_F32)
    hipLaunchKernelGGL(head_rmsnorm_kernel<float>, dim3(blocks), dim3(256), 0, stream, (float*)x, row_stride, w, w_f32, rows,
                       first_col, heads, d, eps);
  else
    hipLaunchKernelGGL(head_rmsnorm_kernel<bf16_t>, dim3(blocks), dim3(256), 0, stream, (bf16_t*)x, row_stride, w, w_f32, rows,
                       first_col, heads, d, eps);
  TK_CHECK_LAUNCH("head_rmsnorm");
  return 0;
}

// --------------------------------------------------------------------------
// add_bias: out[m][n] += bias[n] for 32-bit rows (the bias of a head whose product a library
// computed; every other product adds its bias in its own epilogue)
// --------------------------------------------------------------------------
template <typename T>
__global__ void add_bias_kernel(float* __restrict__ out, const T* __restrict__ bias, size_t total, int cols) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < total) out[i] += to_f32<T>(bias[i % cols]);
}

TK_API int tk_add_bias(int dt, float* out, const void* bias, int rows, int cols, hipStream_t stream) {
  TK_REQUIRE(rows >= 0 && cols > 0, "add_bias: bad sizes %d %d", rows, cols);
  const size_t total = (size_t)rows * cols;
  if (total == 0) return 0;
  const unsigned blocks = (unsigned)((total + 255) / 256);
  if (dt == TK_F32)
    hipLaunchKernelGGL(add_bias_kernel<float>, dim3(blocks), dim3(256), 0, stream, out, (const float*)bias, total, cols);
  else
    hipLaunchKernelGGL(add_bias_kernel<bf16_t>, dim3(blocks), dim3(256), 0, stream, out, (const bf16_t*)bias, total, cols);
  TK_CHECK_LAUNCH("add_bias");
  return 0;
}

// --------------------------------------------------------------------------
// fill: used instead of a memset so that it may be recorded into a HIP graph.
// --------------------------------------------------------------------------
__global__ void fill_u32_kernel(uint32_t* p, uint32_t v, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

TK_API int tk_fill_u32(void* p, uint32_t value, size_t n, hipStream_t stream) {
  if (n == 0) return 0;
  TK_REQUIRE(n < ((size_t)1 << 40), "fill: too many elements");
  hipLaunchKernelGGL(fill_u32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream,
                     (uint32_t*)p, value, n);
  TK_CHECK_LAUNCH("fill_u32");
  return 0;
}

// --------------------------------------------------------------------------
// add: out = x + y, both rounded operands added in 32-bit and rounded once (the residual
// sum behind a product that a library computed)
// --------------------------------------------------------------------------
template <typename T>
__global__ void add_rows_kernel(const T* __restrict__ x, const T* __restrict__ y, T* __restrict__ out, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = from_f32<T>(to_f32<T>(x[i]) + to_f32<T>(y[i]));
}

TK_API int tk_add(int dt, const void* x, const void* y, void* out, size_t n, hipStream_t stream) {
  if (n == 0) return 0;
  TK_REQUIRE(n < ((size_t)1 << 40), "add: too many elements");
  const unsigned blocks = (unsigned)((n + 255) / 256);
  if (dt == TK_F32)
    hipLaunchKernelGGL(add_rows_kernel<float>, dim3(blocks), dim3(256), 0, stream, (const float*)x,
                       (const float*)y, (float*)out, n);
  else
    hipLaunchKernelGGL(add_rows_kernel<bf16_t>, dim3(blocks), dim3(256), 0, stream, (const bf16_t*)x,
                       (const bf16_t*)y, (bf16_t*)out, n);
  TK_CHECK_LAUNCH("add");
  return 0;
}
