// Shared helpers of the gfx950 kernel library: element types, reductions over a
// 64-wide wavefront, error reporting to the Python side.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <stdint.h>

#define TK_WAVE 64

enum TkDtype { TK_F32 = 0, TK_BF16 = 1 };

typedef __hip_bfloat16 bf16_t;

// Entry points are the only symbols a library exports.
#define TK_API extern "C" __attribute__((visibility("default")))

// Every entry point returns 0 or a negative code; the text is read with tk_last_error().
void tk_set_error(const char* fmt, ...);

#define TK_REQUIRE(cond, ...)        \
  do {                               \
    if (!(cond)) {                   \
      tk_set_error(__VA_ARGS__);     \
      return -1;                     \
    }                                \
  } while (0)

#define TK_CHECK_LAUNCH(name)                                                \
  do {                                                                       \
    hipError_t e__ = hipGetLastError();                                      \
    if (e__ != hipSuccess) {                                                 \
      tk_set_error("%s: launch failed: %s", name, hipGetErrorString(e__));   \
      return -2;                                                             \
    }                                                                        \
  } while (0)

// Layout of a page of the cache (P tokens of one kv head, head size d), chosen so that
// the lanes of a wavefront that feed the matrix cores read consecutive memory:
//   keys   [d / 8][P][8]   the 8-element pieces of the P keys, piece by piece
//   values [P / 4][d][4]   groups of 4 tokens, for each the d rows of 4 values
// A page of kv head h of page `page` starts at ((page * nkv + h) * P * d).
#define TK_KEY_PIECE 8
#define TK_VALUE_QUAD 4
__host__ __device__ __forceinline__ size_t key_offset(int P, int in_page, int e) {
  return ((size_t)(e / TK_KEY_PIECE) * P + in_page) * TK_KEY_PIECE + (e % TK_KEY_PIECE);
}
// Elements a page of P keys of size d takes: a key whose size is no multiple of the piece has
// its last piece padded (the matrix-core kernels take multiples of 16 only and never see one).
__host__ __device__ __forceinline__ size_t key_page_elems(int P, int d) {
  return (size_t)((d + TK_KEY_PIECE - 1) / TK_KEY_PIECE) * TK_KEY_PIECE * P;
}
__host__ __device__ __forceinline__ size_t value_offset(int d, int in_page, int e) {
  return ((size_t)(in_page / TK_VALUE_QUAD) * d + e) * TK_VALUE_QUAD + (in_page % TK_VALUE_QUAD);
}

// One rotation of a pair by (cos, sin) in 32-bit, written out in fused multiply-adds so that
// every kernel that rotates gets the same bits whatever the compiler would contract.
__device__ __forceinline__ void rotate_pair(float x1, float x2, float c, float s, float& o1, float& o2) {
  o1 = __fmaf_rn(x1, c, -__fmul_rn(x2, s));
  o2 = __fmaf_rn(x2, c, __fmul_rn(x1, s));
}

// log(1 + exp(x)), also -(logarithm of a sigmoid) of -x: max(x, 0) + log(1 + y) with y = exp(-|x|) <= 1.  log(1 + y) is log 2 (or 0, y below a half) and
// f - f^2 / 2 + f^3 q(f) of f = (y - 1) / 2 (or y), with q of the least greatest error on [-1/4, 1/2], 9e-10 of the result.  The greater terms are
// added with what each sum leaves, so that one rounding remains.  Some 50 instructions where log1pf(expf()) takes 150, in kernels bound by
// them: the first kernel of the delta rule in chunks took 80 us for prompts of 562 and 938 tokens with 35 of them, their parts added plainly, and 87 with log1pf; the call of
// those prompts takes the same with 50 as with 35 (2,983 us).  Errors from 64 bits, root mean square (largest), with
// log1pf(expf(x)) / so: |x| <= 12 1.291e-7 (5.54e-7) / 1.279e-7 (4.77e-7), |x| <= 2 2.93e-8 (1.67e-7) / 2.66e-8 (1.29e-7), in [-1, 0] 1.610e-8 (5.78e-8) / 1.610e-8
// (5.75e-8), the rest there being expf's; of a logarithm of a sigmoid over |x| <= 2 2.94e-8 (1.36e-7) / 2.66e-8 (1.29e-7); of decays exp(-softplus) 1.356e-8 / 1.349e-8
// over |x| <= 12, 1.638e-8 / 1.607e-8 over |x| <= 2.
__device__ __forceinline__ float softplus(float x) {
  const float y = expf(-fabsf(x));
  const bool upper = y >= 0.5f;
  const float f = upper ? fmaf(y, 0.5f, -0.5f) : y;
  const float log2_hi = upper ? 0.693147182f : 0.f, log2_lo = upper ? -1.90465421e-9f : 0.f;
  float q = 0.037672464f;
  q = fmaf(q, f, -0.09116142f);
  q = fmaf(q, f, 0.11700654f);
  q = fmaf(q, f, -0.12727785f);
  q = fmaf(q, f, 0.14276241f);
  q = fmaf(q, f, -0.16655296f);
  q = fmaf(q, f, 0.19999605f);
  q = fmaf(q, f, -0.25000164f);
  q = fmaf(q, f, 0.3333334f);
  const float h = -0.5f * f, s = log2_hi + f, s_left = f - (s - log2_hi);
  const float l = fmaf(h, f, s), l_left = fmaf(h, f, s - l);
  const float left = fmaf(f * f, f * q, (s_left + l_left) + log2_lo);
  const float line = fmaxf(x, 0.f), hi = fmaxf(line, l), lo = fminf(line, l), t = hi + lo;
  return t + ((hi < 64.f ? lo - (t - hi) : 0.f) + left);  // (no difference of infinities)
}

template <typename T>
__device__ __forceinline__ float to_f32(T v);
template <>
__device__ __forceinline__ float to_f32<float>(float v) { return v; }
template <>
__device__ __forceinline__ float to_f32<bf16_t>(bf16_t v) { return __bfloat162float(v); }

template <typename T>
__device__ __forceinline__ T from_f32(float v);
template <>
__device__ __forceinline__ float from_f32<float>(float v) { return v; }
template <>
__device__ __forceinline__ bf16_t from_f32<bf16_t>(float v) { return __float2bfloat16(v); }

// Round a 32-bit value to the storage type and back: the place where the
// reference's tensors are materialised in the engine dtype.
template <typename T>
__device__ __forceinline__ float round_to(float v) { return to_f32<T>(from_f32<T>(v)); }

// x / (1 + exp(-x)) of a bfloat16 number, to be rounded to one: the hardware's exponential and reciprocal, a correction of the quotient
// and the hardware's repair of its special cases; both sides scaled, so that no reciprocal leaves the normal numbers.  Rounded, it is what
// expf and the division give for every one of the 65,536 numbers, in 9 instructions where those take some 25, in epilogues that have nothing
// beside them (a tile of 256 x 256 of gate and up: 128 a thread, one wavefront a SIMD).  us of gate and up in tiles, with those / with
// this: 16,384 x 2,048 101 rows 19.2 / 18.8, 512 36.8 / 35.4, 1,045 78.6 / 75.0, 2,048 120 / 114; 16,384 x 3,072 1,045 rows 109 / 105; 28,672 x 4,096
// 512 rows 99.1 / 96.6, 4,096 697 / 686.
__device__ __forceinline__ float silu_of_bf16(float x) {
  const float d = fmaf(__builtin_amdgcn_exp2f(x * -1.44269504f), 0.0625f, 0.0625f);
  const float u = x * 0.0625f, r = __builtin_amdgcn_rcpf(d), q = u * r;
  return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, q, u), r, q), d, u);
}

// silu(gate) * up as the engine's storage type sees it: both operands and the activation
// rounded to bfloat16, the product left in 32-bit for the caller to round.
__device__ __forceinline__ float silu_mul_bf16(float g, float u) {
  const float gr = round_to<bf16_t>(g), ur = round_to<bf16_t>(u);
  const float s = round_to<bf16_t>(silu_of_bf16(gr));
  return s * ur;
}

// A gated activation with clamps, g sigmoid(alpha g) (u + 1) with g = min(gate, limit) and u = clamp(up, -limit, limit), as the
// engine's storage type sees it: the operands rounded to it, 32-bit arithmetic, the result left for the caller to round.
template <typename T>
__device__ __forceinline__ float clamped_glu(float gate, float up, float limit, float alpha) {
  const float g = fminf(round_to<T>(gate), limit), u = fminf(fmaxf(round_to<T>(up), -limit), limit);
  return g / (1.0f + expf(-alpha * g)) * (u + 1.0f);
}

// Accesses that are coherent across the chip's dies (each has an L2 of its own): relaxed
// atomics of agent scope, which the compiler turns into loads that go around, and stores that
// write through, the caches.  Data that one workgroup of a running kernel writes and another
// reads moves through these; no cache-wide write-back or invalidation is needed then.
__device__ __forceinline__ uint64_t shared_load64(const void* p) {
  return __hip_atomic_load((const uint64_t*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void shared_store64(void* p, uint64_t v) {
  __hip_atomic_store((uint64_t*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void shared_store16(void* p, uint16_t v) {
  __hip_atomic_store((uint16_t*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// What the lanes of one wavefront have written to local memory is there for its other lanes (a wavefront's accesses to
// local memory are in order; the compiler must keep them so).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Every lane's value meets its partners' 32, 16, 8, 4, 2 and 1 lanes away, in this order, through the lanes' own data paths: a step
// takes a few clocks, through local memory (a shuffle) fifty, and these chains stand between two trips to memory.  After the
// step of 8 a row of 16 lanes holds its 8 values twice, so that a turn by 4 is an exchange.
template <typename Op>
__device__ __forceinline__ float wave_reduce(float v, Op op) {
  const auto h = __builtin_amdgcn_permlane32_swap(__float_as_int(v), __float_as_int(v), false, false);
  v = op(__int_as_float(h[0]), __int_as_float(h[1]));
  const auto q = __builtin_amdgcn_permlane16_swap(__float_as_int(v), __float_as_int(v), false, false);
  v = op(__int_as_float(q[0]), __int_as_float(q[1]));
  v = op(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xF, 0xF, true)));  // row_ror:8
  v = op(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xF, 0xF, true)));  // row_ror:4
  v = op(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, true)));   // quad_perm:[2,3,0,1]
  return op(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, true)));  // quad_perm:[1,0,3,2]
}

__device__ __forceinline__ float wave_sum(float v) {
  return wave_reduce(v, [](float a, float b) { return a + b; });
}

__device__ __forceinline__ float wave_max(float v) {
  return wave_reduce(v, [](float a, float b) { return fmaxf(a, b); });
}

// Sum over a workgroup of up to 1024 threads; every thread gets the result.
// `scratch` holds at least 16 floats of LDS; the order of the additions is fixed.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  const int lane = threadIdx.x & (TK_WAVE - 1);
  const int wave = threadIdx.x / TK_WAVE;
  const int nwaves = (blockDim.x + TK_WAVE - 1) / TK_WAVE;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float total = 0.f;
  for (int w = 0; w < nwaves; ++w) total += scratch[w];
  return total;
}

__device__ __forceinline__ float block_max(float v, float* scratch) {
  const int lane = threadIdx.x & (TK_WAVE - 1);
  const int wave = threadIdx.x / TK_WAVE;
  const int nwaves = (blockDim.x + TK_WAVE - 1) / TK_WAVE;
  v = wave_max(v);
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float total = scratch[0];
  for (int w = 1; w < nwaves; ++w) total = fmaxf(total, scratch[w]);
  return total;
}

// Sums over the 16 lanes of a row of the wavefront through the lanes' own data paths (no LDS): partners
// exchange and add, so every lane ends with the same bits, in an order that depends on nothing.
__device__ __forceinline__ float dpp_quad_xor1(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, true));
}
__device__ __forceinline__ float dpp_quad_xor2(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, true));
}
__device__ __forceinline__ float dpp_half_mirror(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xF, 0xF, true));
}
__device__ __forceinline__ float dpp_row_mirror(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xF, 0xF, true));
}
// the sum over the 16 lanes of a row, in every lane
__device__ __forceinline__ float row_sum16(float v) {
  v += dpp_quad_xor1(v);
  v += dpp_quad_xor2(v);
  v += dpp_half_mirror(v);
  v += dpp_row_mirror(v);
  return v;
}

// --------------------------------------------------------------------------
// 16 bytes of the storage type at a time, where sizes and addresses allow it
// --------------------------------------------------------------------------
template <typename T>
struct Pack {
  static constexpr int N = 16 / sizeof(T);
  union { uint4 raw; T v[N]; };
  __device__ __forceinline__ void load(const T* p) { raw = *(const uint4*)p; }
  __device__ __forceinline__ void store(T* p) const { *(uint4*)p = raw; }
};

// 16 bytes a lane from memory to local memory, lane l to `lds` (the same for the wavefront) + 16 l.  Counted in vmcnt, which
// the caller waits for: the compiler knows nothing of the load.
__device__ __forceinline__ void load_to_lds(const bf16_t* src, unsigned lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(src) : "memory", "m0");
}
