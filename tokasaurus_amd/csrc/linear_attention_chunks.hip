// Linear attention in chunks of 64 tokens as products on the matrix cores, for the forms whose decays are at most one and
// come with a portion's tokens: LA_CHANNEL and LA_MEMORY of linear_attention.hip, whose sums these are in another order.
// Every product is one of 32-bit numbers (v_mfma_f32_16x16x4_f32), in either storage type.
//
// Inside a chunk let A_t be the sum of the decays' logarithms from the chunk's first token to token t (a number per row of S,
// or in LA_MEMORY one for all rows), w_s the factor on what token s writes (1, or exp(i - m)), and S the state in front of it:
//     o_t = (exp(A_t) q_t)^T S + sum_{s <= t} P_ts v_s          P_ts = sum_i q_t,i k_s,i exp(A_t,i - A_s,i) w_s
//     S  <- exp(A_last) S + sum_s (exp(A_last - A_s) w_s k_s) v_s^T
// No exponent is positive as it stands, and none becomes so: P is computed in blocks of 16 x 16 tokens, off the diagonal as a
// product of q_t exp(A_t - R) and k_s exp(R - A_s) with R the sum in front of the block of t (s <= R's token < t).  On the
// diagonal the second exponent is positive; where it stays below LC_REACH in every channel (the decays of 16 tokens leave
// more than 2^-LC_REACH) both factors and their product are numbers as good as any, else the block is summed pair by pair.
//
// Three kernels.  The first works on all (chunk, head) at once: decays, their sums, and the factors of the products above, in
// `rec`.  The second walks a request's chunks for a tile of 16 x 16 of a head's state in a wavefront, and leaves the state in front
// of every chunk in `rec`.  The third makes the results from those, all (chunk, head) at once.
// The walk is the only chain, and it is as short as it can be: 16 products a chunk.  Walked together with the results (one kernel, 16 columns of
// a head a workgroup, the state handed round through local memory) a chunk took 2.3 us on as few workgroups as a prompt has heads and
// blocks of columns.  us, all kernels of a layer, walked together / apart, heads of 128 x 128: LA_MEMORY, 8 heads: 2,048 tokens 95 / 52, 8,192 tokens
// 329 / 165, 300 and 1,200 tokens 66 / 49, 100 tokens 20 / 19, six of 500 66 / 67; LA_CHANNEL, 16 heads: 114 / 75, 462 / 334, 87 / 73, 35 / 28, four
// of 500 88 / 80; 4 heads of 256 x 256, 1,000 tokens 121 / 61.
#include "linear_attention.h"
#include <algorithm>
#include <type_traits>

typedef float v4f __attribute__((ext_vector_type(4)));

#define LC_CHUNK 64
#define LC_SLAB 64       // rows of S (key channels) that the first kernel works on at a time
#define LC_LD 68         // a row of a slab in LDS: 64 numbers and the padding that spreads rows over the banks
#define LC_RANK 16       // low-rank sums staged at a time
#define LC_MAX_SLABS 4   // key heads of up to 256 channels
#define LC_FROM 32       // tokens of a step's longest portion from which on it goes in chunks
#define LC_REACH 60.f
#define LC_LOG2E 1.44269504088896341f

__device__ __forceinline__ float lc_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// What a (chunk, head) leaves in `rec`: the factors of q and of k, P, the decay of S over the chunk [dkp], the state in front of the chunk
// and the values (with ones in the column that sums the keys).  All but the decay lie as the lanes of the second and third kernel
// read them, 64 lanes' four numbers side by side: lane 16 c + col of block
//     q [w][m]   has token 16 w + col, channels 16 m + 4 c + e
//     k [n][T]   has channel 16 n + col, tokens 16 T + 4 c + e
//     P [w][T]   has token 16 w + col, tokens s = 16 T + 4 c + e
//     S [z][m]   has column 16 z + col, rows 16 m + 4 c + e
//     v [z][T]   has column 16 z + col, tokens 16 T + 4 c + e
__host__ __device__ __forceinline__ size_t lc_k_at(int dkp) { return (size_t)LC_CHUNK * dkp; }
__host__ __device__ __forceinline__ size_t lc_p_at(int dkp) { return (size_t)2 * LC_CHUNK * dkp; }
__host__ __device__ __forceinline__ size_t lc_d_at(int dkp) { return lc_p_at(dkp) + LC_CHUNK * LC_CHUNK; }
__host__ __device__ __forceinline__ size_t lc_s_at(int dkp) { return lc_d_at(dkp) + dkp; }
__host__ __device__ __forceinline__ size_t lc_v_at(int dkp, int blocks) { return lc_s_at(dkp) + (size_t)dkp * 16 * blocks; }
__host__ __device__ __forceinline__ size_t lc_words(int dkp, int blocks) { return lc_v_at(dkp, blocks) + (size_t)LC_CHUNK * 16 * blocks; }
template <int MODE>
__host__ __device__ __forceinline__ int lc_blocks(int dv) { return (la_columns<MODE>(dv) + 15) / 16; }

bool la_chunks_take(int mode, int dk, int longest) {
  return (mode == LA_CHANNEL || mode == LA_MEMORY) && dk <= LC_SLAB * LC_MAX_SLABS && longest >= LC_FROM;
}

// --------------------------------------------------------------------------
// The first kernel.  A workgroup a (chunk, head); wavefront g owns tokens 16 g .. 16 g + 15: as a channel a lane for loading and
// summing, as rows of a block of P for the products.  Tokens beyond the request's end have q = k = 0 and no decay.
// --------------------------------------------------------------------------
template <int MODE>
__global__ __launch_bounds__(256) void la_chunk_factors_kernel(LaArgs a, int dkp, const float* __restrict__ proj,
                                                               const float2* __restrict__ gates, float* __restrict__ rec) {
  constexpr bool CHANNEL = MODE == LA_CHANNEL;
  __shared__ __align__(16) float qs[LC_CHUNK * LC_LD], ks[LC_CHUNK * LC_LD], as[CHANNEL ? LC_CHUNK * LC_LD : LC_CHUNK];
  __shared__ __align__(16) float low[CHANNEL ? LC_RANK * LC_LD : 4], sums[CHANNEL ? 4 * LC_SLAB : 4], ws[CHANNEL ? 4 : LC_CHUNK];
  const int chunk = blockIdx.x, h = blockIdx.y;
  const int r = a.chunk_req[chunk], row0 = a.chunk_row0[chunk], last = a.q_start[r + 1];
  const int lane = threadIdx.x & (TK_WAVE - 1), g = __builtin_amdgcn_readfirstlane(threadIdx.x / TK_WAVE);
  const int col = lane & 15, c = lane >> 4;
  const int blocks = lc_blocks<MODE>(a.dv);
  float* out = rec + ((size_t)chunk * a.H + h) * lc_words(dkp, blocks);
  const int t0 = row0 + 16 * g;
  // the values, as the products' operands lie (zeros behind the last token; 1 in the column that sums the keys)
#pragma unroll 4
  for (int zc = 0; zc < blocks; ++zc) {
    const int j = zc * 16 + col;
    const float* src = proj + a.v_off + h * a.dv + min(j, a.dv - 1);
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int t = t0 + 4 * c + e;
      v[e] = src[(size_t)min(t, last - 1) * a.ld];
      if (!CHANNEL && j == a.dv) v[e] = 1.f;
      if (t >= last || j >= la_columns<MODE>(a.dv)) v[e] = 0.f;
    }
    ((float4*)(out + lc_v_at(dkp, blocks)))[(zc * 4 + g) * TK_WAVE + lane] = make_float4(v[0], v[1], v[2], v[3]);
  }
  if (!CHANNEL && g == 0) {
    const int t = row0 + lane;
    const float2 e = t < last ? gates[(size_t)t * a.H + h] : make_float2(0.f, 0.f);
    float l = e.x;
#pragma unroll
    for (int o = 1; o < LC_CHUNK; o <<= 1) {
      const float up = __shfl_up(l, o, TK_WAVE);
      if (lane >= o) l += up;
    }
    as[lane] = l * LC_LOG2E;
    ws[lane] = e.y;
  }
  v4f acc[4];
#pragma unroll
  for (int J = 0; J < 4; ++J) acc[J] = (v4f){0.f, 0.f, 0.f, 0.f};
  float diag[4] = {0.f, 0.f, 0.f, 0.f};  // (of diagonal blocks that are summed pair by pair)
  auto stage = [&](int r0, int nr) {  // the chunk's low-rank sums r0 .. r0 + nr - 1
    for (int i = threadIdx.x; i < LC_CHUNK * nr; i += 256) {
      const int t = i / nr, k = i % nr;
      low[k * LC_LD + t] = proj[(size_t)min(row0 + t, last - 1) * a.ld + a.low_off + r0 + k];
    }
  };
  if (CHANNEL) stage(0, min(LC_RANK, a.rank));
  __syncthreads();

  for (int n0 = 0; n0 < dkp; n0 += LC_SLAB) {
    const int ch = n0 + lane, x = h * a.dk + ch;
    const bool in = ch < a.dk;
    float A[16], qv[16], kv[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const float* row = proj + (size_t)min(t0 + j, last - 1) * a.ld + (in ? x : 0);
      qv[j] = row[a.q_off];
      kv[j] = row[a.k_off];
    }
    bool near = true;  // the diagonal block goes as a product
    if (CHANNEL) {
      const int width = a.H * a.dk;
#pragma unroll
      for (int j = 0; j < 16; ++j) A[j] = 0.f;
      for (int r0 = 0; r0 < a.rank; r0 += LC_RANK) {
        const int nr = min(LC_RANK, a.rank - r0);
        float up[LC_RANK];
#pragma unroll
        for (int k = 0; k < LC_RANK; ++k) up[k] = in && k < nr ? a.low_up[(size_t)(r0 + k) * width + x] : 0.f;
        if (a.rank > LC_RANK) {
          __syncthreads();
          stage(r0, nr);
          __syncthreads();
        }
#pragma unroll
        for (int k = 0; k < LC_RANK; ++k) {
          if (k >= nr) break;
          const float4* lt = (const float4*)(low + k * LC_LD + 16 * g);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float4 l4 = lt[j];
            A[4 * j] = fmaf(l4.x, up[k], A[4 * j]); A[4 * j + 1] = fmaf(l4.y, up[k], A[4 * j + 1]);
            A[4 * j + 2] = fmaf(l4.z, up[k], A[4 * j + 2]); A[4 * j + 3] = fmaf(l4.w, up[k], A[4 * j + 3]);
          }
        }
      }
      const float bias = in ? a.low_bias[x] : 0.f;
      float sum = 0.f;
      const float per_tau = 1.f / a.tau;
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        // the quotient by tau, corrected as a division does it (a product alone would be off to one side, 64 times over in a chunk's sum), then in units of log 2
        const float x = la_log_sigmoid(A[j] + bias), y = x * per_tau;
        A[j] = __builtin_amdgcn_div_fixupf(fmaf(fmaf(-y, a.tau, x), per_tau, y), a.tau, x) * LC_LOG2E;
        asm volatile("" : "+v"(A[j]));  // (all of them, side by side: no branch around each)
      }
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        sum += in && t0 + j < last ? A[j] : 0.f;
        A[j] = sum;
      }
      sums[g * LC_SLAB + lane] = sum;
      near = __all(sum > -LC_REACH);
    }
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const bool valid = in && t0 + j < last;
      qs[(16 * g + j) * LC_LD + lane] = valid ? qv[j] * a.q_scale : 0.f;
      kv[j] = valid ? kv[j] : 0.f;
      ks[(16 * g + j) * LC_LD + lane] = kv[j];
    }
    float end;
    if (CHANNEL) {
      __syncthreads();
      float before = 0.f;
      end = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float s = sums[w * LC_SLAB + lane];
        if (w < g) before += s;
        end += s;
      }
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        A[j] += before;
        as[(16 * g + j) * LC_LD + lane] = A[j];
      }
    } else {
      end = as[LC_CHUNK - 1];
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        A[j] = as[16 * g + j];
        kv[j] *= ws[16 * g + j];
      }
    }
    // the factors of the products that the other kernels make (those of q below)
    {
      float4* kt = (float4*)(out + lc_k_at(dkp)) + ((ch / 16) * 4 + g) * TK_WAVE + col;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        kt[16 * j] = make_float4(kv[4 * j] * lc_exp2(end - A[4 * j]), kv[4 * j + 1] * lc_exp2(end - A[4 * j + 1]),
                            kv[4 * j + 2] * lc_exp2(end - A[4 * j + 2]), kv[4 * j + 3] * lc_exp2(end - A[4 * j + 3]));
    }
    if (g == 0) out[lc_d_at(dkp) + ch] = lc_exp2(end);
    __syncthreads();
    // rows 16 g .. of P, transposed: a lane has row 16 J + col of the first operand (k) and column 16 g + col of the second (q),
    // and of every 16 channels the four from 4 c on; it ends up with P of token 16 g + col and tokens s = 16 J + 4 c + i.
#pragma unroll
    for (int m = 0; m < LC_SLAB / 16; ++m) {
      const int at = 16 * m + 4 * c;
      float4 q4 = *(const float4*)(qs + (16 * g + col) * LC_LD + at);
      float4 a4, ref = make_float4(0.f, 0.f, 0.f, 0.f);
      if (CHANNEL) {
        a4 = *(const float4*)(as + (16 * g + col) * LC_LD + at);
      } else {
        const float l = as[16 * g + col];
        a4 = make_float4(l, l, l, l);
      }
      ((float4*)out)[(g * (dkp / 16) + n0 / 16 + m) * TK_WAVE + lane] =
          make_float4(q4.x * lc_exp2(a4.x), q4.y * lc_exp2(a4.y), q4.z * lc_exp2(a4.z), q4.w * lc_exp2(a4.w));
      if (CHANNEL) {
        if (g > 0) ref = *(const float4*)(as + (16 * g - 1) * LC_LD + at);
        q4.x *= lc_exp2(a4.x - ref.x); q4.y *= lc_exp2(a4.y - ref.y); q4.z *= lc_exp2(a4.z - ref.z); q4.w *= lc_exp2(a4.w - ref.w);
      }
      float4 kj[4], bj[4];  // (asked for together, those not used too)
#pragma unroll
      for (int J = 0; J < 4; ++J) {
        kj[J] = *(const float4*)(ks + (16 * J + col) * LC_LD + at);
        if (CHANNEL) bj[J] = *(const float4*)(as + (16 * J + col) * LC_LD + at);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int J = 0; J < 4; ++J) {
        if (J > g || (J == g && !near)) continue;  // (the same for all lanes)
        float4 k4 = kj[J];
        if (CHANNEL) {
          const float4 b4 = bj[J];
          k4.x *= lc_exp2(ref.x - b4.x); k4.y *= lc_exp2(ref.y - b4.y); k4.z *= lc_exp2(ref.z - b4.z); k4.w *= lc_exp2(ref.w - b4.w);
        }
        acc[J] = __builtin_amdgcn_mfma_f32_16x16x4f32(k4.x, q4.x, acc[J], 0, 0, 0);
        acc[J] = __builtin_amdgcn_mfma_f32_16x16x4f32(k4.y, q4.y, acc[J], 0, 0, 0);
        acc[J] = __builtin_amdgcn_mfma_f32_16x16x4f32(k4.z, q4.z, acc[J], 0, 0, 0);
        acc[J] = __builtin_amdgcn_mfma_f32_16x16x4f32(k4.w, q4.w, acc[J], 0, 0, 0);
      }
    }
    if (CHANNEL && !near) {
      // the block on the diagonal: the lane's four pairs (token 16 g + col, tokens s = 16 g + 4 c + i), as a product leaves them
#pragma unroll 4
      for (int m = 0; m < LC_SLAB / 4; ++m) {
        const float4 q4 = *(const float4*)(qs + (16 * g + col) * LC_LD + 4 * m), a4 = *(const float4*)(as + (16 * g + col) * LC_LD + 4 * m);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float4 k4 = *(const float4*)(ks + (16 * g + 4 * c + i) * LC_LD + 4 * m);
          const float4 b4 = *(const float4*)(as + (16 * g + 4 * c + i) * LC_LD + 4 * m);
          // (pairs with s behind the token are dropped below: their exponents are kept from overflowing)
          diag[i] = fmaf(q4.x * k4.x, lc_exp2(fminf(a4.x - b4.x, 0.f)), diag[i]);
          diag[i] = fmaf(q4.y * k4.y, lc_exp2(fminf(a4.y - b4.y, 0.f)), diag[i]);
          diag[i] = fmaf(q4.z * k4.z, lc_exp2(fminf(a4.z - b4.z, 0.f)), diag[i]);
          diag[i] = fmaf(q4.w * k4.w, lc_exp2(fminf(a4.w - b4.w, 0.f)), diag[i]);
        }
      }
    }
    __syncthreads();  // the slab is used up
  }
  // P as far as the third kernel uses it: up to the diagonal block's end
#pragma unroll
  for (int J = 0; J < 4; ++J) {
    if (J > g) continue;
    float p[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = 16 * g + col, s = 16 * J + 4 * c + i;
      p[i] = CHANNEL ? acc[J][i] + (J == g ? diag[i] : 0.f) : acc[J][i] * (lc_exp2(fminf(as[t] - as[s], 0.f)) * ws[s]);
      if (s > t) p[i] = 0.f;
    }
    ((float4*)(out + lc_p_at(dkp)))[(g * 4 + J) * TK_WAVE + lane] = make_float4(p[0], p[1], p[2], p[3]);
  }
}

// --------------------------------------------------------------------------
// The second kernel: the state in front of every chunk.  A wavefront owns 16 rows x 16 columns of a head's state of a request and
// walks its chunks; nothing passes between wavefronts, so a chunk costs its 16 products, one chain.  What a chunk needs (its
// factors of k, its decay, its values) is asked for LC_SETS - 1 chunks ahead, into sets of registers in turn.
// --------------------------------------------------------------------------
#define LC_SETS 5

struct LcStep {
  float4 k[4], v[4], d;
};

template <int MODE>
__global__ __launch_bounds__(TK_WAVE) void la_chunk_states_kernel(LaArgs a, int dkp, float* __restrict__ rec) {
  const int h = blockIdx.x, r = blockIdx.y;
  const int c0 = a.first_chunk[r], chunks = a.first_chunk[r + 1] - c0;
  if (chunks <= 0) return;
  const int lane = threadIdx.x, col = lane & 15, c = lane >> 4;
  const int zc = blockIdx.z / (dkp / 16), n = blockIdx.z % (dkp / 16);  // columns 16 zc .., rows 16 n ..
  const int columns = la_columns<MODE>(a.dv), blocks = lc_blocks<MODE>(a.dv), j = zc * 16 + col;
  const bool live = j < columns;
  float* s_col = a.state + (size_t)a.slots[r] * a.state_stride + ((size_t)h * columns + (live ? j : 0)) * a.dk + 16 * n + 4 * c;
  v4f s;
#pragma unroll
  for (int i = 0; i < 4; ++i) s[i] = live && 16 * n + 4 * c + i < a.dk ? s_col[i] : 0.f;
  const size_t words = lc_words(dkp, blocks), step = (size_t)a.H * words;
  float* own = rec + ((size_t)c0 * a.H + h) * words;
  const float* k_at = own + lc_k_at(dkp) + (n * 4 * TK_WAVE + lane) * 4;
  const float* v_at = own + lc_v_at(dkp, blocks) + (zc * 4 * TK_WAVE + lane) * 4;
  const float* d_at = own + lc_d_at(dkp) + 16 * n + 4 * c;
  float* s_at = own + lc_s_at(dkp) + ((size_t)zc * dkp + 16 * n) * 16 + lane * 4;
  // of the request's chunk i: T < 4 (factors of k and values, and with the first the decay)
  auto ask = [&](LcStep& x, int i, int T) {
    const size_t at = (size_t)i * step;
    x.k[T] = *(const float4*)(k_at + at + T * TK_WAVE * 4);
    x.v[T] = *(const float4*)(v_at + at + T * TK_WAVE * 4);
    if (T == 0) x.d = *(const float4*)(d_at + at);
    __builtin_amdgcn_sched_barrier(0);  // (asked for here, chunks ahead of their use)
  };
  // (the loads stand between the products, which wait for each other)
  auto take = [&](const LcStep& x, int i, LcStep& next, auto more) {
    const int ahead = min(i + LC_SETS - 1, chunks - 1);  // (behind the last chunk that one again)
    *(float4*)(s_at + (size_t)i * step) = make_float4(s[0], s[1], s[2], s[3]);
    s[0] *= x.d.x; s[1] *= x.d.y; s[2] *= x.d.z; s[3] *= x.d.w;
#pragma unroll
    for (int T = 0; T < 4; ++T) {
      s = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[T].x, x.v[T].x, s, 0, 0, 0);
      if constexpr (decltype(more)::value) ask(next, ahead, T);
      s = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[T].y, x.v[T].y, s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[T].z, x.v[T].z, s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[T].w, x.v[T].w, s, 0, 0, 0);
    }
  };
  LcStep x[LC_SETS];
#pragma unroll
  for (int i = 0; i < LC_SETS - 1; ++i)
#pragma unroll
    for (int T = 0; T < 4; ++T) ask(x[i], min(i, chunks - 1), T);
  // (whole turns of the sets, and what is left behind them: with a way out of the middle of a turn the compiler moves what was asked for
  // between registers at its end, and waits for all of it there)
  int i = 0;
#pragma unroll 1
  for (; i + LC_SETS <= chunks; i += LC_SETS) {
#pragma unroll
    for (int u = 0; u < LC_SETS; ++u) take(x[u], i + u, x[(u + LC_SETS - 1) % LC_SETS], std::true_type{});
  }
#pragma unroll
  for (int u = 0; u < LC_SETS - 1; ++u)
    if (i + u < chunks) take(x[u], i + u, x[u], std::false_type{});
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (live && 16 * n + 4 * c + i < a.dk) s_col[i] = s[i];
}

// --------------------------------------------------------------------------
// The third kernel: the results, all (chunk, head) at once.  Wavefront w has tokens 16 w .. of a chunk, whose factors of q and
// rows of P stay in its registers while it goes through the workgroup's blocks of 16 columns: the state in front of the chunk times
// the factors of q, and P times the chunk's values.  A block of the state and of the values goes straight to local memory, two
// ahead, and is read there by all four wavefronts: the path from the L2 to a compute unit gives some 35 bytes a cycle.  NP: slabs of 64
// rows of S.
// --------------------------------------------------------------------------
#define LC_PLACES 3

template <int MODE, int NP>
__global__ __launch_bounds__(256) void la_chunk_outputs_kernel(LaArgs a, int share, const float* __restrict__ rec, float* __restrict__ o) {
  constexpr int DKP = LC_SLAB * NP, PIECES = 4 * NP + 4, LOADS = PIECES / 4;  // of 1 KB: a block of the state, then of the values
  __shared__ __align__(16) float4 lds[LC_PLACES][PIECES * TK_WAVE];
  const int chunk = blockIdx.x, h = blockIdx.y;
  const int lane = threadIdx.x & (TK_WAVE - 1), w = __builtin_amdgcn_readfirstlane(threadIdx.x / TK_WAVE);
  const int col = lane & 15, c = lane >> 4;
  const int columns = la_columns<MODE>(a.dv), blocks = lc_blocks<MODE>(a.dv);
  const int z0 = blockIdx.z * share, z1 = min(blocks, z0 + share);
  const float* src = rec + ((size_t)chunk * a.H + h) * lc_words(DKP, blocks);
  const unsigned base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) float4*)lds;
  auto ask = [&](int zc, int place) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int piece = w * LOADS + i;
      const float* from = piece < 4 * NP ? src + lc_s_at(DKP) + ((size_t)zc * 4 * NP + piece) * TK_WAVE * 4
                                         : src + lc_v_at(DKP, blocks) + ((size_t)zc * 4 + piece - 4 * NP) * TK_WAVE * 4;
      load_to_lds((const bf16_t*)(from + lane * 4), base + (unsigned)((place * PIECES + piece) * TK_WAVE * sizeof(float4)));
    }
  };
  ask(z0, 0);
  if (z0 + 1 < z1) ask(z0 + 1, 1);
  float4 q[4 * NP], p[4];
#pragma unroll
  for (int m = 0; m < 4 * NP; ++m) q[m] = ((const float4*)src)[(w * (DKP / 16) + m) * TK_WAVE + lane];
#pragma unroll
  for (int T = 0; T < 4; ++T)
    if (T <= w) p[T] = ((const float4*)(src + lc_p_at(DKP)))[(w * 4 + T) * TK_WAVE + lane];
  const int row0 = a.chunk_row0[chunk], last = a.q_start[a.chunk_req[chunk] + 1];
  const int t0 = row0 + 16 * w + 4 * c;
  float* dst = o + ((size_t)t0 * a.H + h) * a.o_head + col;
  v4f y0, y1;
  auto deliver = [&](int zc) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (zc * 16 + col < columns && t0 + i < last) dst[(size_t)i * a.H * a.o_head + zc * 16] = y0[i] + y1[i];
  };
  int place = 0;
#pragma unroll 1
  for (int zc = z0; zc < z1; ++zc) {
    // the block is there when only the loads of the one behind it are left; behind the barrier every wavefront's are, and every
    // wavefront is through with the block before, whose place is filled again
    if (zc + 1 < z1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(LOADS) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (zc > z0) deliver(zc - 1);
    if (zc + 2 < z1) ask(zc + 2, place == 0 ? 2 : place - 1);
    y0 = y1 = (v4f){0.f, 0.f, 0.f, 0.f};
    const float4* x = lds[place] + lane;
    float4 sm[4 * NP], vm[4];
#pragma unroll
    for (int m = 0; m < 4 * NP; ++m) sm[m] = x[m * TK_WAVE];
#pragma unroll
    for (int T = 0; T < 4; ++T)
      if (T <= w) vm[T] = x[(4 * NP + T) * TK_WAVE];  // (the same for all lanes)
#pragma unroll
    for (int m = 0; m < 4 * NP; ++m) {
      y0 = __builtin_amdgcn_mfma_f32_16x16x4f32(q[m].x, sm[m].x, y0, 0, 0, 0);
      y1 = __builtin_amdgcn_mfma_f32_16x16x4f32(q[m].y, sm[m].y, y1, 0, 0, 0);
      y0 = __builtin_amdgcn_mfma_f32_16x16x4f32(q[m].z, sm[m].z, y0, 0, 0, 0);
      y1 = __builtin_amdgcn_mfma_f32_16x16x4f32(q[m].w, sm[m].w, y1, 0, 0, 0);
    }
#pragma unroll
    for (int T = 0; T < 4; ++T) {
      if (T > w) continue;
      y0 = __builtin_amdgcn_mfma_f32_16x16x4f32(p[T].x, vm[T].x, y0, 0, 0, 0);
      y1 = __builtin_amdgcn_mfma_f32_16x16x4f32(p[T].y, vm[T].y, y1, 0, 0, 0);
      y0 = __builtin_amdgcn_mfma_f32_16x16x4f32(p[T].z, vm[T].z, y0, 0, 0, 0);
      y1 = __builtin_amdgcn_mfma_f32_16x16x4f32(p[T].w, vm[T].w, y1, 0, 0, 0);
    }
    place = place == LC_PLACES - 1 ? 0 : place + 1;
  }
  deliver(z1 - 1);
}

// 32-bit words of working memory that a chunk of a step takes for all heads, and a token beside that (the gates).
TK_API int tk_linear_attention_chunk_words(int mode, int H, int dk, int dv, int longest) {
  if (!la_chunks_take(mode, dk, longest)) return 0;
  const int dkp = (dk + LC_SLAB - 1) / LC_SLAB * LC_SLAB;
  return (int)(H * lc_words(dkp, mode == LA_MEMORY ? lc_blocks<LA_MEMORY>(dv) : lc_blocks<LA_CHANNEL>(dv)));
}
TK_API int tk_linear_attention_chunk_tokens() { return LC_CHUNK; }

template <int MODE>
static int lc_run(const LaArgs& a, hipStream_t stream) {
  const int slabs = (a.dk + LC_SLAB - 1) / LC_SLAB, dkp = slabs * LC_SLAB;
  const int blocks = lc_blocks<MODE>(a.dv);
  float2* gates = nullptr;
  if (MODE == LA_MEMORY) {
    gates = (float2*)(a.rec + (size_t)a.n_chunks * a.H * lc_words(dkp, blocks));
    la_launch_gates(a, gates, 1, stream);
  }
  if (a.n_singles > 0) la_launch_singles(MODE, a, stream);
  hipLaunchKernelGGL(la_chunk_factors_kernel<MODE>, dim3(a.n_chunks, a.H), dim3(256), 0, stream, a, dkp, a.proj, gates, a.rec);
  hipLaunchKernelGGL(la_chunk_states_kernel<MODE>, dim3(a.H, a.n_requests, blocks * (dkp / 16)), dim3(TK_WAVE), 0, stream, a, dkp, a.rec);
  // blocks of columns a workgroup: as many as leave two workgroups for each of 256 compute units, one of which reads its block while
  // the other multiplies
  const long parts = std::min<long>(blocks, std::max(1l, 512 / ((long)a.n_chunks * a.H)));
  const int share = (int)((blocks + parts - 1) / parts);
  const dim3 grid(a.n_chunks, a.H, (blocks + share - 1) / share);
#define LC_OUTPUTS(NP) hipLaunchKernelGGL((la_chunk_outputs_kernel<MODE, NP>), grid, dim3(256), 0, stream, a, share, a.rec, a.o)
  if (slabs == 1) LC_OUTPUTS(1);
  else if (slabs == 2) LC_OUTPUTS(2);
  else if (slabs == 3) LC_OUTPUTS(3);
  else LC_OUTPUTS(4);
#undef LC_OUTPUTS
  TK_CHECK_LAUNCH("linear_attention");
  return 0;
}

int la_run_chunks(int mode, const LaArgs& a, hipStream_t stream) {
  TK_REQUIRE(a.H < 65536 && a.n_chunks <= a.n_tokens, "linear_attention: bad sizes in chunks");
  return mode == LA_CHANNEL ? lc_run<LA_CHANNEL>(a, stream) : lc_run<LA_MEMORY>(a, stream);
}
