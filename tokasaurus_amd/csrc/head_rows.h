// Rows [q | k | v] of bfloat16 heads on their way from the projection to attention: an RMSNorm (of every head, or of a row's queries and of
// its keys), the rotation of whole heads, keys and values to their pages.  What the general kernel of
// attention_prepare.hip does element by element, for heads of one size d = 16, 32, 64 or 128, 16 bytes at a time: a wavefront has a
// token, a lane pieces of 8 elements, d / 8 neighbouring lanes a head.  All of a row is asked for at once, with the position, so that
// the chain of waits is two trips to memory (the position, then the page and the angles); nothing goes through local memory, no barrier.
// Bound by those trips and the launch up to a few hundred tokens, then by memory.  us, the general kernel / this one, norms of every head, pairs of
// neighbours and of halves, 32 + 8 heads of 64: 16 tokens 7.3 / 5.2 and 7.3 / 6.4, 101 7.5 / 5.5 and 7.5 / 6.7, 500 9.1 / 6.6 and 8.9 / 7.8, 2,048
// 22.0 / 12.2 and 20.3 / 13.6, 8,192 63 / 38.6 and 57 / 40.5; 24 + 8 heads of 128, 1,045 tokens 19.2 / 14.5 and 17.4 / 16.1 (by workgroups of 4 tokens 18.4,
// too few of them).
#pragma once

#include "common.h"

#define HR_TOKENS 2  // a workgroup, a wavefront each
enum { HR_PLAIN = 0, HR_PER_HEAD = 1, HR_PER_ROW = 2 };

struct HeadRows {
  bf16_t* qkv;
  int row_stride;
  const int *positions, *token_req, *block_table;
  int table_stride;
  const float *q_weight, *k_weight;  // [d] (HR_PER_HEAD) or [heads * d] (HR_PER_ROW); null: not normed
  float eps;
  const float* freq;           // [d / 2]
  float rot_scale;
  bf16_t *kcache, *vcache;
  int n_tokens, nq, nkv, d, P, write_cache;
};

// 8 neighbouring elements as four words, and one of them
typedef uint32_t hr_piece_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float hr_element(hr_piece_t x, int e) {
  return __uint_as_float(e & 1 ? x[e >> 1] & 0xffff0000u : x[e >> 1] << 16);
}

// HALVES: pairs (m, m + d / 2), else (2 m, 2 m + 1).  NI: pieces a lane has at most.
template <int NORM, bool HALVES, int NI>
__global__ __launch_bounds__(64 * HR_TOKENS) void head_rows_kernel(HeadRows a) {
  const int lane = threadIdx.x & 63, t = blockIdx.x * HR_TOKENS + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (t >= a.n_tokens) return;
  const int d = a.d, per = d >> 3, half = d >> 1;  // lanes a head, pairs of one
  const int j = lane & (per - 1);                   // this lane's piece of a head, the same in all its pieces
  const int q_end = a.nq * per, k_end = q_end + (a.write_cache ? a.nkv * per : 0), end = k_end + (a.write_cache ? a.nkv * per : 0);
  bf16_t* row = a.qkv + (size_t)t * a.row_stride;
  hr_piece_t x[NI > 8 ? NI : 9];  // (of 128 bytes and less the compiler makes one vector, which it then indexes in 254 registers)
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    x[i] = hr_piece_t{0, 0, 0, 0};
    if (i * 64 + lane < end) x[i] = *(const hr_piece_t*)(row + (i * 64 + lane) * 8);
  }
  const int pos = a.positions[t];
  const int page = a.write_cache ? a.block_table[(size_t)a.token_req[t] * a.table_stride + pos / a.P] : 0, p = pos % a.P;
  // cosines and sines of this lane's pairs
  constexpr int PAIRS = HALVES ? 8 : 4;
  const int first = HALVES ? (j * 8) & (half - 1) : j * 4;
  float cs[PAIRS], sn[PAIRS];
  {  // a lane an angle, handed round
    float s, c;
    sincosf(__fmul_rn((float)pos, a.freq[lane & (half - 1)]), &s, &c);
    c *= a.rot_scale;
    s *= a.rot_scale;
#pragma unroll
    for (int m = 0; m < PAIRS; ++m) {
      cs[m] = __shfl(c, first + m, 64);
      sn[m] = __shfl(s, first + m, 64);
    }
  }
  float rq = 1.f, rk = 1.f;
  if (NORM == HR_PER_ROW) {
    float sq = 0.f, sk = 0.f;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int item = i * 64 + lane;
      float ss = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float v = hr_element(x[i], e);
        ss = fmaf(v, v, ss);
      }
      sq += item < q_end ? ss : 0.f;
      sk += item >= q_end && item < k_end ? ss : 0.f;
    }
    if (a.q_weight) rq = 1.0f / sqrtf(wave_sum(sq) / (float)(a.nq * d) + a.eps);
    if (a.k_weight && a.write_cache) rk = 1.0f / sqrtf(wave_sum(sk) / (float)(a.nkv * d) + a.eps);
  }
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int item = i * 64 + lane;
    if (i * 64 >= end) continue;  // (the same for all lanes)
    const bool is_q = item < q_end, is_k = !is_q && item < k_end;
    const float* weight = is_q ? a.q_weight : (is_k ? a.k_weight : nullptr);
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = hr_element(x[i], e);
    if (NORM != HR_PLAIN) {
      float r = is_q ? rq : rk;
      if (NORM == HR_PER_HEAD) {
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fmaf(v[e], v[e], ss);
        // (a head's lanes are neighbours, from a multiple of their number on; the same number for all lanes)
        ss += dpp_quad_xor1(ss);
        if (per >= 4) ss += dpp_quad_xor2(ss);
        if (per >= 8) ss += dpp_half_mirror(ss);
        if (per >= 16) ss += dpp_row_mirror(ss);
        r = 1.0f / sqrtf(ss / (float)d + a.eps);
      }
      if (weight) {
        const float* w = weight + (NORM == HR_PER_HEAD ? j * 8 : (item - (is_q ? 0 : q_end)) * 8);
        const float4 w0 = *(const float4*)w, w1 = *(const float4*)(w + 4);
        v[0] = v[0] * r * w0.x; v[1] = v[1] * r * w0.y; v[2] = v[2] * r * w0.z; v[3] = v[3] * r * w0.w;
        v[4] = v[4] * r * w1.x; v[5] = v[5] * r * w1.y; v[6] = v[6] * r * w1.z; v[7] = v[7] * r * w1.w;
      }
    }
    union { bf16_t v[8]; hr_piece_t raw; } y;
    if (HALVES) {
      const bool low = j * 8 < half;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float other = __shfl_xor(v[e], per >> 1, 64);
        float u = low ? v[e] : other, w = low ? other : v[e];
        rotate_pair(u, w, cs[e], sn[e], u, w);
        y.v[e] = __float2bfloat16(low ? u : w);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        float u, w;
        rotate_pair(v[e], v[e + 1], cs[e / 2], sn[e / 2], u, w);
        y.v[e] = __float2bfloat16(u);
        y.v[e + 1] = __float2bfloat16(w);
      }
    }
    if (is_q) {
      *(hr_piece_t*)(row + item * 8) = y.raw;
    } else if (is_k) {
      const int h = (item - q_end) / per;
      *(hr_piece_t*)(a.kcache + ((size_t)page * a.nkv + h) * key_page_elems(a.P, d) + ((size_t)j * a.P + p) * 8) = y.raw;
    } else if (item < end) {
      const int h = (item - k_end) / per;
      bf16_t* dst = a.vcache + ((size_t)page * a.nkv + h) * a.P * d + value_offset(d, p, j * 8);
#pragma unroll
      for (int e = 0; e < 8; ++e) ((uint16_t*)dst)[e * TK_VALUE_QUAD] = (uint16_t)(x[i][e >> 1] >> (16 * (e & 1)));
    }
  }
}

// Whether the kernel takes these rows: heads of a size whose lanes divide a wavefront, 16-byte pieces, weights at multiples of 16.
static bool head_rows_take(const HeadRows& a) {
  const bool size = a.d == 16 || a.d == 32 || a.d == 64 || a.d == 128;
  const uintptr_t at = (uintptr_t)a.qkv | (uintptr_t)a.kcache | (uintptr_t)a.q_weight | (uintptr_t)a.k_weight;
  return size && a.row_stride % 8 == 0 && (at & 15) == 0 && a.freq &&
         (a.nq + (a.write_cache ? 2 * a.nkv : 0)) * (a.d >> 3) <= 64 * 16;
}

template <int NORM, bool HALVES>
static void launch_head_rows(const HeadRows& a, hipStream_t stream) {
  const int pieces = (a.nq + (a.write_cache ? 2 * a.nkv : 0)) * (a.d >> 3), ni = (pieces + 63) / 64;
  const dim3 grid((a.n_tokens + HR_TOKENS - 1) / HR_TOKENS), block(64 * HR_TOKENS);
  if (ni <= 4) hipLaunchKernelGGL((head_rows_kernel<NORM, HALVES, 4>), grid, block, 0, stream, a);
  else if (ni <= 8) hipLaunchKernelGGL((head_rows_kernel<NORM, HALVES, 8>), grid, block, 0, stream, a);
  else if (ni <= 12) hipLaunchKernelGGL((head_rows_kernel<NORM, HALVES, 12>), grid, block, 0, stream, a);
  else hipLaunchKernelGGL((head_rows_kernel<NORM, HALVES, 16>), grid, block, 0, stream, a);
}
