// The gated delta rule with one decay per head and key channel, as a recurrence over the
// tokens of each request, and what stands around it: the short causal convolutions of q, k
// and v with their activation, the unit norms, the write strength and the decays (before), the
// per-head norm with its gate (after).  Everything that enters the recurrence is 32-bit.
//
// Per request a state row of 32-bit floats lives in the request's slot:
//   [ S: heads x dv x dk ][ tail: (taps - 1) x channels ]
// S is kept transposed (a value column's dk numbers lie together); the tail holds the last
// taps - 1 inputs of the convolutions, oldest first, channels = 2 * kv_heads * dk + heads * dv
// in the order q | k | v.  A slot's row is all zeros when a request takes it.
//
// Per token and head, with decay g (dk), write strength beta, unit k, scaled unit q, value v:
//   S <- diag(g) S;  u = beta * (v - S^T k);  S <- S + k u^T;  o = S^T q.
// The columns of S (one a value channel) do not meet: a column is owned by DR_LANES lanes that
// cut dk between them and add up through the wavefront, always in the same order: among the tokens that
// run here a result does not depend on how its request's tokens were cut into steps or what shares the batch.
// Portions of many tokens run in delta_rule_chunks.hip instead, whose sums stand in another order: a prompt's
// results depend in their last bits on how it was cut, single tokens' on nothing.
#include "delta_rule.h"

#define DR_LANES 16    // lanes that share a column of the state (a row of the wavefront's data paths)
#define DR_TOKENS 16   // most tokens staged in LDS at a time

// --------------------------------------------------------------------------
// Before the recurrence.  A token's work is cut into units, one a wavefront: a q head or a k head
// (convolution, silu, unit norm), a v head (convolution, silu), a head's decays, and the write
// strengths of all heads.
//   proj row (T): [q | k | v] (channels) ... and the write strength's `heads` numbers at col_b
//   a_pre (32-bit) [tokens, heads * dk]: the decay's projection before bias and softplus
//   rec row (32-bit): [q: G*dk | k: G*dk | v: H*dv | decay: H*dk | beta: H]
// FUSE_TAIL (every request of the step brings one token): the lane that convolves a channel also
// moves the channel's tail on, which it alone reads; else the kernel below does it afterwards.
// `below` > 0: only the tokens from `first_row` on, of requests that bring fewer than `below`; rec starts at that row.
// --------------------------------------------------------------------------
#define DP_MAX_PER_LANE 8  // dk, dv <= 512

template <typename T, bool FUSE_TAIL>
__global__ __launch_bounds__(256) void delta_prepare_kernel(
    const T* __restrict__ proj, int ld, int col_b, const float* __restrict__ a_pre, int ld_a,
    const float* __restrict__ conv_w, int taps, const float* __restrict__ a_log,
    const float* __restrict__ dt_bias, float* __restrict__ state, size_t state_stride,
    size_t tail_off, const int* __restrict__ q_start, const int* __restrict__ token_req,
    const int* __restrict__ slots, float* __restrict__ rec, int ld_rec, int H, int G, int dk, int dv, int first_row, int below) {
  const int t = first_row + blockIdx.x;
  if (below > 0) {
    const int r = token_req[t];
    if (q_start[r + 1] - q_start[r] >= below) return;
  }
  const int lane = threadIdx.x & (TK_WAVE - 1);
  const int unit = blockIdx.y * (blockDim.x / TK_WAVE) + threadIdx.x / TK_WAVE;
  const int n_units = 2 * G + 2 * H + 1;
  if (unit >= n_units) return;
  const int C = 2 * G * dk + H * dv;
  float* out = rec + (size_t)blockIdx.x * ld_rec;
  const int v_off = 2 * G * dk, decay_off = v_off + H * dv, beta_off = decay_off + H * dk;
  if (unit < 2 * G + H) {
    // a head's channels through the convolution: q head, k head or v head
    const bool is_v = unit >= 2 * G;
    const int width = is_v ? dv : dk;
    const int c0 = is_v ? v_off + (unit - 2 * G) * dv : unit * dk;
    const int r = token_req[t];
    const int first = q_start[r];
    const int local = t - first;
    float* tail = state + (size_t)slots[r] * state_stride + tail_off;
    float y[DP_MAX_PER_LANE];
    float ss = 0.f;
#pragma unroll
    for (int n = 0; n < DP_MAX_PER_LANE; ++n) {
      const int i = lane + n * TK_WAVE;
      y[n] = 0.f;
      if (i < width) {
        const int c = c0 + i;
        float acc = 0.f;
        for (int j = 0; j < taps; ++j) {
          const int src = local - (taps - 1) + j;
          const float x = src >= 0 ? to_f32<T>(proj[(size_t)(first + src) * ld + c])
                                   : tail[(size_t)(src + taps - 1) * C + c];
          acc = fmaf(conv_w[(size_t)c * taps + j], x, acc);
          if (FUSE_TAIL && j >= 1) tail[(size_t)(j - 1) * C + c] = x;  // (local is 0: entry j - 1 was read a tap ago)
        }
        y[n] = silu_f32(acc);
        ss = fmaf(y[n], y[n], ss);
      }
    }
    float mul = 1.f;
    if (!is_v) {  // unit vectors; the queries also times dk^-1/2
      mul = 1.0f / sqrtf(wave_sum(ss) + 1e-6f);
      if (unit < G) mul *= 1.0f / sqrtf((float)dk);
    }
#pragma unroll
    for (int n = 0; n < DP_MAX_PER_LANE; ++n) {
      const int i = lane + n * TK_WAVE;
      if (i < width) out[c0 + i] = y[n] * mul;
    }
  } else if (unit < 2 * G + 2 * H) {
    const int h = unit - 2 * G - H;
    const float rate = expf(a_log[h]);
    for (int i = lane; i < dk; i += TK_WAVE) {
      const int x = h * dk + i;
      out[decay_off + x] = expf(-rate * softplus(a_pre[(size_t)t * ld_a + x] + dt_bias[x]));
    }
  } else {
    for (int i = lane; i < H; i += TK_WAVE)
      out[beta_off + i] = sigmoid_f32(to_f32<T>(proj[(size_t)t * ld + col_b + i]));
  }
}

// The convolutions' tails after the step: the last taps - 1 inputs of every request, taken
// from this step's rows and, where the step brought fewer, from the old tail.  A thread a
// (request, channel); it reads all it needs before it writes.
template <typename T>
__global__ void delta_tail_kernel(const T* __restrict__ proj, int ld, int taps, float* __restrict__ state,
                                  size_t state_stride, size_t tail_off, const int* __restrict__ q_start,
                                  const int* __restrict__ slots, int C) {
  const int r = blockIdx.y;
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= C) return;
  const int first = q_start[r], n = q_start[r + 1] - first;
  float* tail = state + (size_t)slots[r] * state_stride + tail_off;
  float keep[DR_MAX_TAPS];
#pragma unroll
  for (int s = 0; s < DR_MAX_TAPS - 1; ++s) {
    if (s < taps - 1) {
      const int src = n - (taps - 1) + s;
      keep[s] = src >= 0 ? to_f32<T>(proj[(size_t)(first + src) * ld + c]) : tail[(size_t)(src + taps - 1) * C + c];
    }
  }
#pragma unroll
  for (int s = 0; s < DR_MAX_TAPS - 1; ++s)
    if (s < taps - 1) tail[(size_t)s * C + c] = keep[s];
}

// --------------------------------------------------------------------------
// The recurrence.  Workgroup (head, request, block of value columns); a column of the state is
// owned by DR_LANES neighbouring lanes: lane holds rows 4 * (lane + DR_LANES * n) + e, n < NQ,
// e < 4.  Per token, with the decayed column sd = g * s:
//     dot = k . sd,  qs = q . sd   (one round of sums through the lanes for both)
//     u = beta * (v - dot);  s = sd + k * u;  o = qs + u * (q . k)
// (o = q . s written out: the read-out sees the token's own write).  q . k does not depend on
// the column but costs little beside the other two sums.  The tokens' rows come through LDS
// in chunks: DR_LOADERS threads of the workgroup do nothing but move the next chunk in while
// the others compute this one, and meet them at a barrier a chunk.
// The sums through the lanes use the lanes' own data paths (no LDS): partners exchange and
// add, so every lane ends with the same bits, in an order that depends on nothing.
// --------------------------------------------------------------------------
// Rows of tokens t0 .. t0 + nt - 1 into a buffer [nt][q | k | decay (dkp each) | v (cols) | beta | padding], by
// `nmove` threads of which this is `me`.  Several loads are in flight a thread before the first is stored.
// VEC: the three long pieces move 16 bytes at a time (the caller found sizes and offsets to be multiples of 4).
template <bool VEC>
__device__ __forceinline__ void delta_move_rows(float* buf, const float* __restrict__ rec, int ld_rec, int t0, int nt,
                                                int me, int nmove, int row_floats, int dkp, int dk, int dv, int cols,
                                                int col0, int q_off, int k_off, int g_off, int v_off, int b_off) {
  constexpr int B = 8;
  if constexpr (VEC) {
    const int per_row = 3 * dkp / 4;
    for (int x0 = me; x0 < nt * per_row; x0 += B * nmove) {
      float4 v[B];
#pragma unroll
      for (int j = 0; j < B; ++j) {
        const int x = x0 + j * nmove;
        v[j] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (x < nt * per_row) {
          const int tt = x / per_row, rem = x % per_row, which = rem / (dkp / 4), i = 4 * (rem % (dkp / 4));
          if (i < dk)
            v[j] = *(const float4*)(rec + (size_t)(t0 + tt) * ld_rec + (which == 0 ? q_off : (which == 1 ? k_off : g_off)) + i);
        }
      }
#pragma unroll
      for (int j = 0; j < B; ++j) {
        const int x = x0 + j * nmove;
        if (x < nt * per_row) *(float4*)(buf + (x / per_row) * row_floats + 4 * (x % per_row)) = v[j];
      }
    }
  }
  const int first = VEC ? 3 * dkp : 0;  // what is left to move one by one
  const int per_row = row_floats - first;
  for (int x0 = me; x0 < nt * per_row; x0 += B * nmove) {
    float v[B];
#pragma unroll
    for (int j = 0; j < B; ++j) {
      const int x = x0 + j * nmove;
      v[j] = 0.f;
      if (x < nt * per_row) {
        const int tt = x / per_row, rem = first + x % per_row;
        const float* row = rec + (size_t)(t0 + tt) * ld_rec;
        if (rem < 3 * dkp) {
          const int which = rem / dkp, i = rem % dkp;
          if (i < dk) v[j] = row[(which == 0 ? q_off : (which == 1 ? k_off : g_off)) + i];
        } else if (rem < 3 * dkp + cols) {
          const int c = rem - 3 * dkp;
          if (col0 + c < dv) v[j] = row[v_off + col0 + c];
        } else if (rem == 3 * dkp + cols) {
          v[j] = row[b_off];
        }
      }
    }
#pragma unroll
    for (int j = 0; j < B; ++j) {
      const int x = x0 + j * nmove;
      if (x < nt * per_row) buf[(x / per_row) * row_floats + first + x % per_row] = v[j];
    }
  }
}

#define DR_LOADERS 128  // threads of a workgroup that only move the next chunk's rows into LDS

template <int NQ, bool VEC>
__global__ __launch_bounds__(NQ > 2 ? 384 : 1024) void delta_rule_kernel(
    const float* __restrict__ rec, int ld_rec, float* __restrict__ state, size_t state_stride,
    const int* __restrict__ q_start, const int* __restrict__ slots, float* __restrict__ o, int H, int G,
    int dk, int dv, int cols, int tok, int below) {
  // two buffers of [tok][3][dkp] q, k, decay; [tok][cols] v; [tok] beta
  extern __shared__ __align__(16) float stage[];
  const int h = blockIdx.x, r = blockIdx.y;
  const int col0 = blockIdx.z * cols;
  const int ncompute = cols * DR_LANES;
  const bool loader = (int)threadIdx.x >= ncompute;
  const int lane = threadIdx.x % DR_LANES, grp = threadIdx.x / DR_LANES;
  const int col = col0 + grp;
  const bool live = !loader && col < dv;
  constexpr int dkp = NQ * DR_LANES * 4;  // dk rounded up to what the lanes of a column hold
  const int gk = h / (H / G);
  const int first = q_start[r], last = q_start[r + 1];
  if (below > 0 && last - first >= below) return;  // the same for the whole workgroup
  float* s_col = state + (size_t)slots[r] * state_stride + ((size_t)h * dv + (live ? col : 0)) * dk;

  float s[NQ][4];
#pragma unroll
  for (int n = 0; n < NQ; ++n)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = 4 * (lane + DR_LANES * n) + e;
      s[n][e] = (live && i < dk) ? s_col[i] : 0.f;
    }

  const int row_floats = 3 * dkp + (cols + 1 + 3) / 4 * 4;
  const int buf_floats = tok * row_floats;
  const int q_off = gk * dk, k_off = G * dk + gk * dk, v_off = 2 * G * dk + h * dv;
  const int g_off = 2 * G * dk + H * dv + h * dk, b_off = 2 * G * dk + H * dv + H * dk + h;

#define move(BUF, T0, NT, ME, NMOVE) \
  delta_move_rows<VEC>(BUF, rec, ld_rec, T0, NT, ME, NMOVE, row_floats, dkp, dk, dv, cols, col0, q_off, k_off, g_off, v_off, b_off)
  if (first < last) move(stage, first, min(tok, last - first), threadIdx.x, blockDim.x);
  __syncthreads();
  int chunk = 0;
#pragma unroll 1
  for (int t0 = first; t0 < last; t0 += tok, ++chunk) {
    const int nt = min(tok, last - t0);
    const float* buf = stage + (chunk & 1) * buf_floats;
    if (loader) {
      const int next = t0 + tok;
      if (next < last) move(stage + ((chunk + 1) & 1) * buf_floats, next, min(tok, last - next), threadIdx.x - ncompute, DR_LOADERS);
    } else {
#pragma unroll 1
      for (int tt = 0; tt < nt; ++tt) {
        const float* row = buf + tt * row_floats;
        const float4* q4 = (const float4*)row;
        const float4* k4 = (const float4*)(row + dkp);
        const float4* g4 = (const float4*)(row + 2 * dkp);
        float kk[NQ][4];
        float dot[2] = {0.f, 0.f}, qs[2] = {0.f, 0.f}, kq[2] = {0.f, 0.f};
#pragma unroll
        for (int n = 0; n < NQ; ++n) {
          const float4 g = g4[lane + DR_LANES * n], k = k4[lane + DR_LANES * n], q = q4[lane + DR_LANES * n];
          kk[n][0] = k.x; kk[n][1] = k.y; kk[n][2] = k.z; kk[n][3] = k.w;
          s[n][0] *= g.x; s[n][1] *= g.y; s[n][2] *= g.z; s[n][3] *= g.w;
          dot[0] = fmaf(k.x, s[n][0], dot[0]); dot[1] = fmaf(k.y, s[n][1], dot[1]);
          dot[0] = fmaf(k.z, s[n][2], dot[0]); dot[1] = fmaf(k.w, s[n][3], dot[1]);
          qs[0] = fmaf(q.x, s[n][0], qs[0]); qs[1] = fmaf(q.y, s[n][1], qs[1]);
          qs[0] = fmaf(q.z, s[n][2], qs[0]); qs[1] = fmaf(q.w, s[n][3], qs[1]);
          kq[0] = fmaf(q.x, k.x, kq[0]); kq[1] = fmaf(q.y, k.y, kq[1]);
          kq[0] = fmaf(q.z, k.z, kq[0]); kq[1] = fmaf(q.w, k.w, kq[1]);
        }
        const float d = row_sum16(dot[0] + dot[1]);
        const float qsum = row_sum16(qs[0] + qs[1]);
        const float kqsum = row_sum16(kq[0] + kq[1]);
        const float u = row[3 * dkp + cols] * (row[3 * dkp + grp] - d);
#pragma unroll
        for (int n = 0; n < NQ; ++n)
#pragma unroll
          for (int e = 0; e < 4; ++e) s[n][e] = fmaf(kk[n][e], u, s[n][e]);
        if (live && lane == 0) o[(size_t)(t0 + tt) * H * dv + (size_t)h * dv + col] = fmaf(u, kqsum, qsum);
      }
    }
    __syncthreads();
  }
#undef move
  if (live) {
#pragma unroll
    for (int n = 0; n < NQ; ++n)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 4 * (lane + DR_LANES * n) + e;
        if (i < dk) s_col[i] = s[n][e];
      }
  }
}

// --------------------------------------------------------------------------
// After the recurrence: every head's dv outputs divided by their root mean square, times a
// weight [dv] shared by the heads, times sigmoid(gate); rounded once to T.  A wavefront a
// (token, head).
// --------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void gated_head_norm_kernel(const float* __restrict__ o, const float* __restrict__ gate,
                                                              int ld_gate, int H, const float* __restrict__ w, float eps,
                                                              T* __restrict__ out, long units, int dv) {
  const int lane = threadIdx.x & (TK_WAVE - 1);
  const long unit = (long)blockIdx.x * (blockDim.x / TK_WAVE) + threadIdx.x / TK_WAVE;
  if (unit >= units) return;
  const float* x = o + (size_t)unit * dv;
  const float* g = gate + (size_t)(unit / H) * ld_gate + (size_t)(unit % H) * dv;
  float ss = 0.f;
  for (int i = lane; i < dv; i += TK_WAVE) ss = fmaf(x[i], x[i], ss);
  ss = wave_sum(ss);
  const float rstd = 1.0f / sqrtf(ss / (float)dv + eps);
  for (int i = lane; i < dv; i += TK_WAVE)
    out[(size_t)unit * dv + i] = from_f32<T>(x[i] * rstd * w[i] * sigmoid_f32(g[i]));
}

// --------------------------------------------------------------------------
// A step of single tokens (every request one, as many kv heads as heads): all of the above for a (head, request) in one workgroup, with
// the bits of the three kernels, every sum in their order.  A column of the state is owned by DR_LANES lanes as above, a thread has
// NC of them, DS_GROUPS apart; they are asked for in front of all else, so that the convolutions, norms and decays (a
// channel a thread, through local memory) are made while the state is on its way.  What bounds it: two trips to memory, the convolution's
// inputs and the state beside each other and the slot's number in front, and the state's bytes (128 KB read and
// written a head of 128 x 128).  us a layer, 16 heads of 128 x 128, three kernels / this one, states from memory: 1 request 11.1 / 5.0, 8 requests
// 21.6 / 7.2, 64 requests 67.5 / 35.2 (3.8 TB/s); 16 heads of 256 x 256, 8 requests 56.4 / 20.2; a decode step of 8 requests, eight layers, 735 / 635.
// --------------------------------------------------------------------------
#define DS_THREADS 1024
#define DS_GROUPS (DS_THREADS / DR_LANES)
#define DS_MAX 256  // dk, dv

struct DeltaSingleArgs {
  const void* proj;
  int ld, col_b;
  const float* a_pre;
  int ld_a;
  const float* conv_w;
  int taps;
  const float *a_log, *dt_bias;
  float* state;
  size_t state_stride, tail_off;
  const int *q_start, *slots;
  const float* gate;
  int ld_gate;
  const float* norm_w;
  float eps;
  void* out;
  int H, dk, dv;
};

template <typename T, int NQ, int NC>
__global__ __launch_bounds__(DS_THREADS) void delta_single_kernel(DeltaSingleArgs a) {
  constexpr int DKP = NQ * DR_LANES * 4;
  __shared__ __align__(16) float qs[DKP], ks[DKP], gs[DKP], vs[DS_MAX], os[DS_MAX], mul[2], beta;
  const int h = blockIdx.x, r = blockIdx.y, tid = threadIdx.x, dk = a.dk, dv = a.dv;
  const int t = a.q_start[r];
  if (a.q_start[r + 1] <= t) return;
  const int lane = tid % DR_LANES, grp = tid / DR_LANES;
  float* row = a.state + (size_t)a.slots[r] * a.state_stride;
  float* s_at = row + (size_t)h * dv * dk;
  float4 s[NC][NQ];
#pragma unroll
  for (int j = 0; j < NC; ++j)
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
      const int col = grp + j * DS_GROUPS, i = 4 * (lane + DR_LANES * n);
      s[j][n] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (col < dv && i < dk) s[j][n] = *(const float4*)(s_at + (size_t)col * dk + i);
    }
  const T* x_row = (const T*)a.proj + (size_t)t * a.ld;
  const int conv = 2 * dk + dv, C = a.H * conv;
  for (int c = tid; c < conv + dk + 1; c += DS_THREADS) {
    if (c < conv) {  // a channel of q, k or v through the convolution and silu, its tail moved on
      const int which = c < dk ? 0 : (c < 2 * dk ? 1 : 2), x = c - which * dk;
      const int ch = (which == 2 ? 2 * a.H * dk + h * dv : (which * a.H + h) * dk) + x;
      float* tail = row + a.tail_off + ch;
      const float* w = a.conv_w + (size_t)ch * a.taps;
      const float own = to_f32<T>(x_row[ch]);
      float acc = 0.f;
      if (a.taps == 4) {  // (all of them asked for before the first is moved)
        const float x0 = tail[0], x1 = tail[C], x2 = tail[2 * (size_t)C];
        acc = fmaf(w[0], x0, acc);
        acc = fmaf(w[1], x1, acc);
        acc = fmaf(w[2], x2, acc);
        acc = fmaf(w[3], own, acc);
        tail[0] = x1;
        tail[C] = x2;
        tail[2 * (size_t)C] = own;
      } else {
        for (int j = 0; j < a.taps; ++j) {
          const float in = j < a.taps - 1 ? tail[(size_t)j * C] : own;
          acc = fmaf(w[j], in, acc);
          if (j >= 1) tail[(size_t)(j - 1) * C] = in;
        }
      }
      (which == 0 ? qs : (which == 1 ? ks : vs))[x] = silu_f32(acc);
    } else if (c < conv + dk) {
      const int x = c - conv;
      const float rate = expf(a.a_log[h]);
      gs[x] = expf(-rate * softplus(a.a_pre[(size_t)t * a.ld_a + h * dk + x] + a.dt_bias[h * dk + x]));
    } else {
      beta = sigmoid_f32(to_f32<T>(x_row[a.col_b + h]));
    }
  }
  if (tid < DKP - dk) qs[dk + tid] = ks[dk + tid] = gs[dk + tid] = 0.f;  // (lanes beyond the head's channels)
  __syncthreads();
  const int wave = tid / TK_WAVE, wl = tid % TK_WAVE;
  if (wave < 2) {  // unit vectors; the queries also times dk^-1/2
    const float* y = wave == 0 ? qs : ks;
    float ss = 0.f;
    for (int i = wl; i < dk; i += TK_WAVE) ss = fmaf(y[i], y[i], ss);
    float m = 1.0f / sqrtf(wave_sum(ss) + 1e-6f);
    if (wave == 0) m *= 1.0f / sqrtf((float)dk);
    if (wl == 0) mul[wave] = m;
  }
  __syncthreads();
  const float mq = mul[0], mk = mul[1], b = beta;
  float4 q[NQ], k[NQ], g[NQ];
#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    const int i = lane + DR_LANES * n;
    q[n] = ((const float4*)qs)[i];
    k[n] = ((const float4*)ks)[i];
    g[n] = ((const float4*)gs)[i];
    q[n].x *= mq; q[n].y *= mq; q[n].z *= mq; q[n].w *= mq;
    k[n].x *= mk; k[n].y *= mk; k[n].z *= mk; k[n].w *= mk;
  }
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    const int col = grp + j * DS_GROUPS;
    float dot[2] = {0.f, 0.f}, qd[2] = {0.f, 0.f}, kq[2] = {0.f, 0.f};
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
      float4& z = s[j][n];
      z.x *= g[n].x; z.y *= g[n].y; z.z *= g[n].z; z.w *= g[n].w;
      dot[0] = fmaf(k[n].x, z.x, dot[0]); dot[1] = fmaf(k[n].y, z.y, dot[1]);
      dot[0] = fmaf(k[n].z, z.z, dot[0]); dot[1] = fmaf(k[n].w, z.w, dot[1]);
      qd[0] = fmaf(q[n].x, z.x, qd[0]); qd[1] = fmaf(q[n].y, z.y, qd[1]);
      qd[0] = fmaf(q[n].z, z.z, qd[0]); qd[1] = fmaf(q[n].w, z.w, qd[1]);
      kq[0] = fmaf(q[n].x, k[n].x, kq[0]); kq[1] = fmaf(q[n].y, k[n].y, kq[1]);
      kq[0] = fmaf(q[n].z, k[n].z, kq[0]); kq[1] = fmaf(q[n].w, k[n].w, kq[1]);
    }
    const float d = row_sum16(dot[0] + dot[1]), qsum = row_sum16(qd[0] + qd[1]), kqsum = row_sum16(kq[0] + kq[1]);
    const float u = b * ((col < dv ? vs[col] : 0.f) - d);
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
      float4& z = s[j][n];
      z.x = fmaf(k[n].x, u, z.x); z.y = fmaf(k[n].y, u, z.y); z.z = fmaf(k[n].z, u, z.z); z.w = fmaf(k[n].w, u, z.w);
      const int i = 4 * (lane + DR_LANES * n);
      if (col < dv && i < dk) *(float4*)(s_at + (size_t)col * dk + i) = z;
    }
    if (col < dv && lane == 0) os[col] = fmaf(u, kqsum, qsum);
  }
  __syncthreads();
  if (wave > 0) return;
  const float* gate = a.gate + (size_t)t * a.ld_gate + (size_t)h * dv;
  float ss = 0.f;
  for (int i = wl; i < dv; i += TK_WAVE) ss = fmaf(os[i], os[i], ss);
  const float rstd = 1.0f / sqrtf(wave_sum(ss) / (float)dv + a.eps);
  T* out = (T*)a.out + ((size_t)t * a.H + h) * dv;
  for (int i = wl; i < dv; i += TK_WAVE) out[i] = from_f32<T>(os[i] * rstd * a.norm_w[i] * sigmoid_f32(gate[i]));
}

template <typename T, int NQ>
static void launch_delta_single(const DeltaSingleArgs& a, int n_requests, hipStream_t stream) {
  const dim3 grid(a.H, n_requests);
  if (a.dv <= DS_GROUPS) hipLaunchKernelGGL((delta_single_kernel<T, NQ, 1>), grid, dim3(DS_THREADS), 0, stream, a);
  else if (a.dv <= 2 * DS_GROUPS) hipLaunchKernelGGL((delta_single_kernel<T, NQ, 2>), grid, dim3(DS_THREADS), 0, stream, a);
  else hipLaunchKernelGGL((delta_single_kernel<T, NQ, 4>), grid, dim3(DS_THREADS), 0, stream, a);
}

// Whether tk_delta_single takes these heads and this state: pieces of 16 bytes.
TK_API int tk_delta_single_takes(int H, int G, int dk, int dv, const float* state, size_t state_stride) {
  return H == G && dk > 0 && dk <= DS_MAX && dk % 4 == 0 && dv > 0 && dv <= DS_MAX && state_stride % 4 == 0 && ((uintptr_t)state & 15) == 0 ? 1 : 0;
}

// A step of one token a request: tk_delta_prepare, tk_delta_rule and tk_gated_head_norm in one launch (their arguments; out [tokens][H * dv]).
TK_API int tk_delta_single(int dt, const void* proj, int ld, int col_b, const float* a_pre, int ld_a, const float* conv_w, int taps,
                           const float* a_log, const float* dt_bias, float* state, size_t state_stride, size_t tail_off, const int* q_start,
                           const int* slots, const float* gate, int ld_gate, const float* norm_w, float eps, void* out, int n_requests, int H,
                           int dk, int dv, hipStream_t stream) {
  TK_REQUIRE(n_requests >= 0 && n_requests < 65536 && H > 0 && tk_delta_single_takes(H, H, dk, dv, state, state_stride),
             "delta_single: bad sizes requests=%d heads=%d dk=%d dv=%d", n_requests, H, dk, dv);
  TK_REQUIRE(taps >= 1 && taps <= DR_MAX_TAPS, "delta_single: %d taps (1..%d)", taps, DR_MAX_TAPS);
  const int C = H * (2 * dk + dv);
  TK_REQUIRE(ld >= C && col_b >= 0 && col_b + H <= ld && ld_a >= H * dk && ld_gate >= H * dv, "delta_single: row strides %d, %d, %d too short", ld, ld_a, ld_gate);
  TK_REQUIRE((size_t)H * dv * dk <= tail_off && tail_off + (size_t)(taps - 1) * C <= state_stride, "delta_single: the state row is too short");
  if (n_requests == 0) return 0;
  const DeltaSingleArgs a = {proj, ld, col_b, a_pre, ld_a, conv_w, taps, a_log, dt_bias, state, state_stride, tail_off, q_start, slots,
                             gate, ld_gate, norm_w, eps, out, H, dk, dv};
#define DS_CASE(T)                                                       \
  do {                                                                   \
    if (dk <= 64) launch_delta_single<T, 1>(a, n_requests, stream);      \
    else if (dk <= 128) launch_delta_single<T, 2>(a, n_requests, stream); \
    else launch_delta_single<T, 4>(a, n_requests, stream);               \
  } while (0)
  if (dt == TK_F32) DS_CASE(float);
  else DS_CASE(bf16_t);
#undef DS_CASE
  TK_CHECK_LAUNCH("delta_single");
  return 0;
}

// The tails of `C` channels moved on by the step's rows (after whoever reads the old ones).
TK_API int tk_delta_tail(int dt, const void* proj, int ld, int taps, float* state, size_t state_stride, size_t tail_off,
                         const int* q_start, const int* slots, int n_requests, int C, hipStream_t stream) {
  TK_REQUIRE(taps >= 1 && taps <= DR_MAX_TAPS && ld >= C && tail_off + (size_t)(taps - 1) * C <= state_stride && n_requests < 65536,
             "delta_tail: bad sizes taps=%d channels=%d requests=%d", taps, C, n_requests);
  if (taps == 1 || n_requests <= 0) return 0;
  const dim3 grid((C + 255) / 256, n_requests);
  if (dt == TK_F32)
    hipLaunchKernelGGL(delta_tail_kernel<float>, grid, dim3(256), 0, stream, (const float*)proj, ld, taps, state, state_stride,
                       tail_off, q_start, slots, C);
  else
    hipLaunchKernelGGL(delta_tail_kernel<bf16_t>, grid, dim3(256), 0, stream, (const bf16_t*)proj, ld, taps, state, state_stride,
                       tail_off, q_start, slots, C);
  TK_CHECK_LAUNCH("delta_tail");
  return 0;
}

// below > 0: only the rows from first_row on, of requests that bring fewer tokens; the tails stay as they are (tk_delta_tail
// moves them on afterwards).  rec: [n_tokens - first_row] rows.
TK_API int tk_delta_prepare(int dt, const void* proj, int ld, int col_b, const float* a_pre, int ld_a,
                            const float* conv_w, int taps, const float* a_log, const float* dt_bias,
                            float* state, size_t state_stride, size_t tail_off, const int* q_start,
                            const int* token_req, const int* slots, float* rec, int ld_rec, int n_tokens,
                            int n_requests, int H, int G, int dk, int dv, int first_row, int below, hipStream_t stream) {
  TK_REQUIRE(first_row >= 0 && below >= 0 && (below > 0 || first_row == 0) && first_row <= n_tokens,
             "delta_prepare: rows from %d on of requests of fewer than %d tokens", first_row, below);
  TK_REQUIRE(n_tokens >= 0 && n_requests >= 0 && H > 0 && G > 0 && H % G == 0 && dk > 0 && dv > 0,
             "delta_prepare: bad sizes tokens=%d heads=%d kv heads=%d dk=%d dv=%d", n_tokens, H, G, dk, dv);
  TK_REQUIRE(taps >= 1 && taps <= DR_MAX_TAPS, "delta_prepare: %d taps (1..%d)", taps, DR_MAX_TAPS);
  const int C = 2 * G * dk + H * dv;
  TK_REQUIRE(ld >= C && col_b >= 0 && col_b + H <= ld, "delta_prepare: row stride %d too short", ld);
  TK_REQUIRE(ld_a >= H * dk, "delta_prepare: the decay projection's stride %d is too short", ld_a);
  TK_REQUIRE(ld_rec >= C + H * dk + H, "delta_prepare: output stride %d too short", ld_rec);
  TK_REQUIRE(tail_off + (size_t)(taps - 1) * C <= state_stride, "delta_prepare: the state row is too short");
  TK_REQUIRE(dk <= DP_MAX_PER_LANE * TK_WAVE && dv <= DP_MAX_PER_LANE * TK_WAVE, "delta_prepare: head sizes %d, %d (at most %d)",
             dk, dv, DP_MAX_PER_LANE * TK_WAVE);
  if (n_tokens == first_row) return 0;
  const int units = 2 * G + 2 * H + 1;
  const dim3 grid(n_tokens - first_row, (units + 3) / 4);
  TK_REQUIRE(grid.y < 65536, "delta_prepare: too many heads");
  // every request brings one token: the convolving lane moves its channel's tail on itself
  const bool fuse_tail = n_tokens == n_requests && taps > 1 && below == 0;
#define DP_LAUNCH(T, FUSE)                                                                                         \
  hipLaunchKernelGGL((delta_prepare_kernel<T, FUSE>), grid, dim3(256), 0, stream, (const T*)proj, ld, col_b, a_pre, ld_a, \
                     conv_w, taps, a_log, dt_bias, state, state_stride, tail_off, q_start, token_req, slots, rec,  \
                     ld_rec, H, G, dk, dv, first_row, below)
  if (dt == TK_F32) {
    if (fuse_tail) DP_LAUNCH(float, true); else DP_LAUNCH(float, false);
  } else {
    if (fuse_tail) DP_LAUNCH(bf16_t, true); else DP_LAUNCH(bf16_t, false);
  }
#undef DP_LAUNCH
  TK_CHECK_LAUNCH("delta_prepare");
  if (taps > 1 && !fuse_tail && below == 0) return tk_delta_tail(dt, proj, ld, taps, state, state_stride, tail_off, q_start, slots, n_requests, C, stream);
  return 0;
}

// rec, o: of the step's first row.  below > 0: only the requests that bring fewer tokens.
TK_API int tk_delta_rule(const float* rec, int ld_rec, float* state, size_t state_stride, const int* q_start,
                         const int* slots, float* o, int n_requests, int H, int G, int dk, int dv, int cols,
                         int below, hipStream_t stream) {
  TK_REQUIRE(n_requests >= 0 && H > 0 && G > 0 && H % G == 0 && dk > 0 && dv > 0,
             "delta_rule: bad sizes heads=%d kv heads=%d dk=%d dv=%d", H, G, dk, dv);
  TK_REQUIRE(dk <= 512, "delta_rule: key size %d (at most 512)", dk);
  TK_REQUIRE(cols > 0 && cols % (TK_WAVE / DR_LANES) == 0 && cols * DR_LANES <= 1024,
             "delta_rule: %d columns a workgroup", cols);
  TK_REQUIRE(ld_rec >= 2 * G * dk + H * dv + H * dk + H, "delta_rule: input stride %d too short", ld_rec);
  TK_REQUIRE((size_t)H * dv * dk <= state_stride, "delta_rule: the state row is too short");
  TK_REQUIRE(n_requests < 65536, "delta_rule: too many requests");
  if (n_requests == 0) return 0;
  int nq = (dk + DR_LANES * 4 - 1) / (DR_LANES * 4);
  nq = nq <= 2 ? nq : (nq <= 4 ? 4 : 8);  // the kernel's instances
  const int dkp = nq * DR_LANES * 4;
  const int threads = cols * DR_LANES + DR_LOADERS;
  TK_REQUIRE(threads <= (nq > 2 ? 384 : 1024), "delta_rule: %d columns a workgroup are too many for key size %d", cols, dk);
  const int row_floats = 3 * dkp + (cols + 1 + 3) / 4 * 4;
  int tok = 8192 / row_floats;  // two buffers of 32 KB at most
  tok = tok > DR_TOKENS ? DR_TOKENS : tok;
  TK_REQUIRE(tok >= 1, "delta_rule: key size %d with %d columns a workgroup", dk, cols);
  const size_t smem = sizeof(float) * 2 * (size_t)tok * row_floats;
  const dim3 grid(H, n_requests, (dv + cols - 1) / cols), block(threads);
  const bool vec = dk % 4 == 0 && (H * dv) % 4 == 0 && ld_rec % 4 == 0 && ((uintptr_t)rec & 15) == 0;
#define DR_CASE(NQ)                                                                                              \
  do {                                                                                                           \
    if (vec)                                                                                                     \
      hipLaunchKernelGGL((delta_rule_kernel<NQ, true>), grid, block, smem, stream, rec, ld_rec, state,           \
                         state_stride, q_start, slots, o, H, G, dk, dv, cols, tok, below);                            \
    else                                                                                                         \
      hipLaunchKernelGGL((delta_rule_kernel<NQ, false>), grid, block, smem, stream, rec, ld_rec, state,          \
                         state_stride, q_start, slots, o, H, G, dk, dv, cols, tok, below);                            \
  } while (0)
  if (nq == 1) DR_CASE(1);
  else if (nq == 2) DR_CASE(2);
  else if (nq == 4) DR_CASE(4);
  else DR_CASE(8);
#undef DR_CASE
  TK_CHECK_LAUNCH("delta_rule");
  return 0;
}

TK_API int tk_gated_head_norm(int dt, const float* o, const float* gate, int ld_gate, const float* w, float eps, void* out,
                              int n_tokens, int H, int dv, hipStream_t stream) {
  TK_REQUIRE(ld_gate >= H * dv, "gated_head_norm: the gate's stride %d is too short", ld_gate);
  TK_REQUIRE(n_tokens >= 0 && H > 0 && dv > 0, "gated_head_norm: bad sizes %d %d %d", n_tokens, H, dv);
  if (n_tokens == 0) return 0;
  const long units = (long)n_tokens * H;
  const long blocks = (units + 3) / 4;
  TK_REQUIRE(blocks < (1l << 31), "gated_head_norm: too many rows");
  if (dt == TK_F32)
    hipLaunchKernelGGL(gated_head_norm_kernel<float>, dim3((unsigned)blocks), dim3(256), 0, stream, o, gate, ld_gate, H, w, eps,
                       (float*)out, units, dv);
  else
    hipLaunchKernelGGL(gated_head_norm_kernel<bf16_t>, dim3((unsigned)blocks), dim3(256), 0, stream, o, gate, ld_gate, H, w, eps,
                       (bf16_t*)out, units, dv);
  TK_CHECK_LAUNCH("gated_head_norm");
  return 0;
}
