// The gated delta rule over portions of many tokens, in chunks of 16 as products on the matrix cores' 32-bit multiply-adds
// (v_mfma_f32_16x16x4_f32): the sums of delta_rule.hip in another order, everything 32-bit as there.
//
// Inside a chunk let a_t be the product of the decays of its tokens up to t (a number per row of S), S the state in front of it,
// L the strictly lower triangle of beta_t M_ts and T = (1 + L)^-1:
//     M_ts = sum_i k_t,i k_s,i prod_{s < j <= t} g_j,i        P_ts = the same with q_t, s <= t
//     u_t  = beta_t (v_t - (a_t k_t)^T S - sum_{s < t} M_ts u_s)    =>    U = V' - W S,  V' = T beta V,  W = T beta (a k)
//     o_t  = (a_t q_t)^T S + sum_{s <= t} P_ts u_s                   =>    O = P V' + (a q - P W) S
//     S   <- a_last S + sum_s (k_s prod_{j > s} g_j) u_s^T
// Every decay appears in products of at most the chunk's decays, as the recurrence multiplies them: no logarithms, no
// exponents, no quotients, whatever the decays are.
//
// Two kernels.  The first takes all (chunk, head) at once, from the projections (convolutions, unit norms, decays, write
// strengths are made there: nothing of delta_prepare's rows goes through memory), and leaves W, a q - P W, the factors of k, the
// chunk's decay, V' and P V'.  The second walks a request's chunks for 16 columns of a head's state in a workgroup, whose four
// wavefronts hold a quarter of S's rows each in registers: two products on what the first left (their quarters added
// through local memory, one barrier a chunk) and one update.  The result of a product lies in the lanes as the next needs
// its operand (row 4 * (lane / 16) + j of column lane % 16), so S never leaves the registers.
// A step's portions of many tokens come here (delta_portions_in_chunks in ops.py), its other requests run in delta_rule.hip: how a
// request is cut into portions changes the order of the sums.
// The recurrence token by token is one chain of 270 ns a token; here it is one of about 1 us a chunk of 16, and the first
// kernel, bound by its vector instructions, has no chain.  Two prompts of 562 and 938 tokens, 16 heads of 128 x 128: 72 us of
// delta_prepare and 256 us of delta_rule before, 80 and 53 us now (93 and 55 with sizes that the first kernel learned as it ran and walks that waited
// for all of a chunk's operands, us of a layer with what surrounds it: these two prompts 142 / 121, one of 1,500 168 / 148, eight of 200 133 / 131).
#include "delta_rule.h"

typedef float v4f __attribute__((ext_vector_type(4)));

#define DC_CHUNK 16
#define DC_MAX_DK 256
#define DC_MAX_DV 256
#define DC_LD 20  // floats a row of the chunk's 16 x 16 matrices takes in local memory (read 16 bytes at a time)

// What a (chunk, head) leaves, in floats, as the lanes of the second kernel read it (64 lanes' four numbers side by side), for
// dkp rows (a multiple of 64) and dvp columns (a multiple of 16): lane 16 q + r of block m holds
//   W, Q  token r, rows 16 m + 4 q + e          K  row 16 m + r, tokens 4 q + e        D  the decay of every row, plain
//   V, O  column 16 m + r, tokens 4 q + e
__host__ __device__ __forceinline__ size_t dc_q_at(int dkp) { return (size_t)16 * dkp; }
__host__ __device__ __forceinline__ size_t dc_k_at(int dkp) { return (size_t)32 * dkp; }
__host__ __device__ __forceinline__ size_t dc_d_at(int dkp) { return (size_t)48 * dkp; }
__host__ __device__ __forceinline__ size_t dc_v_at(int dkp) { return (size_t)49 * dkp; }
__host__ __device__ __forceinline__ size_t dc_o_at(int dkp, int dvp) { return dc_v_at(dkp) + (size_t)16 * dvp; }
__host__ __device__ __forceinline__ size_t dc_words(int dkp, int dvp) { return dc_o_at(dkp, dvp) + (size_t)16 * dvp; }

struct DeltaChunkArgs {
  const void* proj;
  int ld, col_b;
  const float* a_pre;
  int ld_a;
  const float* conv_w;
  int taps;
  const float* a_log;
  const float* dt_bias;
  float* state;
  size_t state_stride, tail_off;
  const int* q_start;
  const int* slots;
  const int* chunk_req;
  const int* chunk_row0;
  const int* chunk_first;
  float* rec;
  float* o;
  int H, G, dk, dv, dkp, dvp;
};

template <typename T, int DKP>
__global__ __launch_bounds__(256, 4) void delta_chunk_factors_kernel(DeltaChunkArgs a) {
  extern __shared__ __align__(16) float sh[];
  constexpr int dkp = DKP;
  const int dvp = a.dvp, dk = a.dk, dv = a.dv;
  float* qs = sh;                      // [16][dkp]
  float* ks = qs + DC_CHUNK * dkp;     // [16][dkp]
  float* gs = ks + DC_CHUNK * dkp;     // [16][dkp]
  float* vs = gs + DC_CHUNK * dkp;     // [16][dvp]
  float* Ms = vs + DC_CHUNK * dvp;      // [16][DC_LD]
  float* Ps = Ms + DC_CHUNK * DC_LD;    // [16][DC_LD]
  float* Ts = Ps + DC_CHUNK * DC_LD;    // [16][DC_LD] T beta
  float* beta = Ts + DC_CHUNK * DC_LD;  // [16]
  const T* proj = (const T*)a.proj;
  const int chunk = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int r = a.chunk_req[chunk], row0 = a.chunk_row0[chunk], first = a.q_start[r];
  const int n = min(DC_CHUNK, a.q_start[r + 1] - row0), local0 = row0 - first;
  const int gk = h / (a.H / a.G), C = 2 * a.G * dk + a.H * dv;
  const float* tail = a.state + (size_t)a.slots[r] * a.state_stride + a.tail_off;

  // what the decays are made from, asked for in front of all else
  constexpr int DECAYS = DC_CHUNK * DKP / 256;
  const float* pre = a.a_pre + (size_t)row0 * a.ld_a + h * dk;
  float z[DECAYS];
#pragma unroll
  for (int u = 0; u < DECAYS; ++u) {
    const int t = (u * 256 + tid) / DKP, x = (u * 256 + tid) % DKP;
    z[u] = pre[(unsigned)(min(t, n - 1) * a.ld_a + min(x, dk - 1))] + a.dt_bias[(unsigned)(h * dk + min(x, dk - 1))];
  }
  // a channel's 16 tokens through the convolution and silu, a thread a channel of q, k or v; zeros behind the last token
  for (int c = tid; c < 2 * dkp + dvp; c += 256) {
    const int which = c < dkp ? 0 : (c < 2 * dkp ? 1 : 2);
    const int x = c - which * dkp;  // channel within the head
    const bool in = x < (which == 2 ? dv : dk);
    const int ch = which == 2 ? 2 * a.G * dk + h * dv + x : which * a.G * dk + gk * dk + x;
    float* dst = (which == 0 ? qs : (which == 1 ? ks : vs)) + x;
    const int pitch = which == 2 ? dvp : dkp;
    if (!in) {
#pragma unroll
      for (int t = 0; t < DC_CHUNK; ++t) dst[t * pitch] = 0.f;
      continue;
    }
    const float* w = a.conv_w + (size_t)ch * a.taps;
    auto row_of = [&](int row) { return to_f32<T>((proj + (size_t)row * a.ld)[(unsigned)ch]); };
    auto input = [&](int src) {  // of place `src` among the step's tokens of the request, or from the tail before them
      return src >= 0 ? row_of(first + src) : tail[(size_t)(src + a.taps - 1) * C + ch];
    };
    if (a.taps <= 4) {
      float xs[DC_CHUNK + 3];  // the three inputs in front and the chunk's own
      if (local0 >= 3) {       // all of them this step's rows: asked for at once (rows behind the last token: that one's again)
#pragma unroll
        for (int u = 0; u < DC_CHUNK + 3; ++u) xs[u] = row_of(row0 + min(u - 3, n - 1));
      } else {  // (places before the taps' reach are not read)
#pragma unroll
        for (int u = 0; u < 3; ++u) xs[u] = u - 3 + a.taps - 1 >= 0 ? input(local0 + u - 3) : 0.f;
#pragma unroll
        for (int u = 3; u < DC_CHUNK + 3; ++u) xs[u] = row_of(row0 + min(u - 3, n - 1));
      }
#pragma unroll
      for (int t = 0; t < DC_CHUNK; ++t) {
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (j >= 4 - a.taps) acc = fmaf(w[j - 4 + a.taps], xs[t + j], acc);
        dst[t * pitch] = t < n ? silu_f32(acc) : 0.f;
      }
    } else {
      for (int t = 0; t < DC_CHUNK; ++t) {
        float acc = 0.f;
        if (t < n)
          for (int j = 0; j < a.taps; ++j) acc = fmaf(w[j], input(local0 + t - (a.taps - 1) + j), acc);
        dst[t * pitch] = t < n ? silu_f32(acc) : 0.f;
      }
    }
  }
  const float rate = expf(a.a_log[h]);
#pragma unroll
  for (int u = 0; u < DECAYS; ++u) {
    const int i = u * 256 + tid;
    gs[i] = i / DKP < n && i % DKP < dk ? expf(-rate * softplus(z[u])) : 1.f;
  }
  if (tid < DC_CHUNK) beta[tid] = tid < n ? sigmoid_f32(to_f32<T>(proj[(size_t)(row0 + tid) * a.ld + a.col_b + h])) : 0.f;
  __syncthreads();
  {  // unit vectors, the queries also times dk^-1/2: a wavefront four tokens
    const int lane = tid & (TK_WAVE - 1), wave = tid / TK_WAVE;
    const float qmul = 1.0f / sqrtf((float)dk);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      float* row = (u < 4 ? qs : ks) + (wave * 4 + (u & 3)) * dkp;
      float ss = 0.f;
#pragma unroll
      for (int i = lane; i < DKP; i += TK_WAVE) ss = fmaf(row[i], row[i], ss);  // (zeros behind dk)
      float mul = 1.0f / sqrtf(wave_sum(ss) + 1e-6f);
      if (u < 4) mul *= qmul;
#pragma unroll
      for (int i = lane; i < DKP; i += TK_WAVE) row[i] *= mul;
    }
  }
  __syncthreads();
  {  // M and P: 16 lanes a token s, a sixteenth of the channels each, the decays multiplied up from s on
    const int s = tid >> 4, cg = tid & 15;
    float M[DC_CHUNK], P[DC_CHUNK];
#pragma unroll
    for (int t = 0; t < DC_CHUNK; ++t) M[t] = P[t] = 0.f;
    int end = DKP;
    asm volatile("" : "+s"(end));  // (a loop also where it is one turn: its reads, all asked for at once, would fill the registers)
#pragma unroll 1
    for (int c = 4 * cg; c < end; c += 64) {
      const v4f k = *(const v4f*)(ks + s * dkp + c);
      v4f e = k;
#pragma unroll
      for (int t = 0; t < DC_CHUNK; ++t) {
        const v4f g = *(const v4f*)(gs + t * dkp + c), kt = *(const v4f*)(ks + t * dkp + c), qt = *(const v4f*)(qs + t * dkp + c);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          e[j] = t > s ? e[j] * g[j] : k[j];
          M[t] = fmaf(kt[j], e[j], M[t]);
          P[t] = fmaf(qt[j], e[j], P[t]);
        }
      }
    }
#pragma unroll
    for (int t = 0; t < DC_CHUNK; ++t) {
      const float m = row_sum16(M[t]), p = row_sum16(P[t]);
      if (cg == 0) {
        Ms[t * DC_LD + s] = t > s ? m : 0.f;
        Ps[t * DC_LD + s] = t >= s ? p : 0.f;
      }
    }
  }
  __syncthreads();
  if (tid < DC_CHUNK) {  // column tid of T, row by row, times beta
    float col[DC_CHUNK];
#pragma unroll
    for (int t = 0; t < DC_CHUNK; ++t) {
      float sum = 0.f;
#pragma unroll
      for (int s = 0; s < t; ++s) sum = fmaf(Ms[t * DC_LD + s], col[s], sum);
      col[t] = (t == tid ? 1.f : 0.f) - beta[t] * sum;
    }
#pragma unroll
    for (int t = 0; t < DC_CHUNK; ++t) Ts[t * DC_LD + tid] = col[t] * beta[tid];
  }
  __syncthreads();
  float* out = a.rec + ((size_t)chunk * a.H + h) * dc_words(dkp, dvp);
  // sum over s <= t of row t of T beta (of P) times x[s]
  auto row_times = [&](const float* m, int t, const float (&x)[DC_CHUNK]) {
    float sum = 0.f;
#pragma unroll
    for (int s4 = 0; s4 < DC_CHUNK / 4; ++s4) {
      if (4 * s4 > t) break;
      const v4f f = *(const v4f*)(m + t * DC_LD + 4 * s4);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (4 * s4 + j <= t) sum = fmaf(f[j], x[4 * s4 + j], sum);
    }
    return sum;
  };
  for (int i = tid; i < dkp + dvp; i += 256) {
    if (i < dkp) {
      const int c = i;
      float ke[DC_CHUNK], w[DC_CHUNK];
      float p = 1.f;
#pragma unroll
      for (int t = 0; t < DC_CHUNK; ++t) {
        p *= gs[t * dkp + c];
        ke[t] = ks[t * dkp + c] * p;
      }
      out[dc_d_at(dkp) + c] = p;
      float* at = out + (size_t)((c >> 4) * 64 + ((c >> 2) & 3) * 16) * 4 + (c & 3);  // token t 4 t further
      p = 1.f;
#pragma unroll
      for (int t = 0; t < DC_CHUNK; ++t) {
        w[t] = row_times(Ts, t, ke);
        at[4 * t] = w[t];
        p *= gs[t * dkp + c];
        at[dc_q_at(dkp) + 4 * t] = fmaf(qs[t * dkp + c], p, -row_times(Ps, t, w));
      }
      p = 1.f;
      v4f kh[4];
#pragma unroll
      for (int s = DC_CHUNK - 1; s >= 0; --s) {
        kh[s >> 2][s & 3] = ks[s * dkp + c] * p;
        p *= gs[s * dkp + c];
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) *(v4f*)(out + dc_k_at(dkp) + (size_t)((c >> 4) * 64 + q * 16 + (c & 15)) * 4) = kh[q];
    } else {
      const int c = i - dkp;
      float x[DC_CHUNK], v[DC_CHUNK];
      v4f vp[4], op[4];
#pragma unroll
      for (int t = 0; t < DC_CHUNK; ++t) x[t] = vs[t * dvp + c];
#pragma unroll
      for (int t = 0; t < DC_CHUNK; ++t) {
        v[t] = row_times(Ts, t, x);
        vp[t >> 2][t & 3] = v[t];
        op[t >> 2][t & 3] = row_times(Ps, t, v);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const size_t at = (size_t)((c >> 4) * 64 + q * 16 + (c & 15)) * 4;
        *(v4f*)(out + dc_v_at(dkp) + at) = vp[q];
        *(v4f*)(out + dc_o_at(dkp, dvp) + at) = op[q];
      }
    }
  }
}

// RB: blocks of 16 rows of S a wavefront holds (dkp = 64 RB).  Bound by a chunk's chain of products, sum and update (0.9 us): W S, which it
// goes on from, comes first, Q S waits behind the barrier.  The sets of operands are taken in whole turns and the remainder by itself: left
// out of the middle of a turn, the loop waits for all that is on its way and copies it.
template <int RB>
__global__ __launch_bounds__(256) void delta_chunk_walk_kernel(DeltaChunkArgs a) {
  __shared__ __align__(16) v4f part[2][2][4][TK_WAVE];  // [chunk's parity][W S, Q S][wavefront][lane]
  constexpr int SETS = RB <= 2 ? 4 : (RB == 3 ? 3 : 2);  // chunks whose operands are there or on their way, as many as registers hold
  const int h = blockIdx.x, r = blockIdx.y, nb = blockIdx.z, tid = threadIdx.x;
  const int lane = tid & (TK_WAVE - 1), wave = tid / TK_WAVE;
  const int lr = lane & 15, q = lane >> 4;
  const int dkp = a.dkp, dvp = a.dvp;
  const int first = a.q_start[r], last = a.q_start[r + 1];
  if (first >= last) return;
  const int c0 = a.chunk_first[r], chunks = a.chunk_first[r + 1] - c0;  // none: a request that the recurrence takes
  if (chunks <= 0) return;
  const size_t words = dc_words(dkp, dvp), step = (size_t)a.H * words;
  const int col = nb * 16 + lr;
  float* s_col = a.state + (size_t)a.slots[r] * a.state_stride + ((size_t)h * a.dv + (col < a.dv ? col : 0)) * a.dk;
  v4f S[RB];
#pragma unroll
  for (int b = 0; b < RB; ++b)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int row = 16 * (wave * RB + b) + 4 * q + j;
      S[b][j] = col < a.dv && row < a.dk ? s_col[row] : 0.f;
    }
  struct Operands {
    v4f w[RB], qx[RB], k[RB], d[RB], v;
    float o;
  };
  const float* base = a.rec + (size_t)c0 * step + (size_t)h * words;
  auto ask = [&](int c, Operands& x) {
    const float* p = base + (size_t)c * step;
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      const size_t at = (size_t)((wave * RB + b) * 64 + lane) * 4;
      x.w[b] = *(const v4f*)(p + at);
      x.qx[b] = *(const v4f*)(p + dc_q_at(dkp) + at);
      x.k[b] = *(const v4f*)(p + dc_k_at(dkp) + at);
      x.d[b] = *(const v4f*)(p + dc_d_at(dkp) + 16 * (wave * RB + b) + 4 * q);
    }
    x.v = *(const v4f*)(p + dc_v_at(dkp) + (size_t)(nb * 64 + lane) * 4);
    x.o = p[dc_o_at(dkp, dvp) + (size_t)nb * 256 + tid];
    __builtin_amdgcn_sched_barrier(0);  // (asked for here, a chunk ahead of their use)
  };
  // the output this thread adds up: float tid of the products' [lane][4]
  const int token = 4 * (tid >> 6) + (tid & 3), ocol = nb * 16 + ((tid >> 2) & 15);
  float o_before = 0.f;
  auto deliver = [&](int c) {  // the outputs of chunk c, whose Q S the wavefronts left behind its barrier
    const float* f = (const float*)part[c & 1][1];
    const float sum = o_before + ((f[tid] + f[256 + tid]) + (f[512 + tid] + f[768 + tid]));
    const int t = first + c * DC_CHUNK + token;
    if (t < last && ocol < a.dv) a.o[(size_t)t * a.H * a.dv + (size_t)h * a.dv + ocol] = sum;
  };
  auto walk = [&](int c, const Operands& x) {
    v4f ws = (v4f){0.f, 0.f, 0.f, 0.f}, qs = ws;
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) ws = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w[b][e], S[b][e], ws, 0, 0, 0);
    v4f(*p)[4][TK_WAVE] = part[c & 1];
    p[0][wave][lane] = ws;
    __syncthreads();
    const v4f w0 = p[0][0][lane], w1 = p[0][1][lane], w2 = p[0][2][lane], w3 = p[0][3][lane];
    __builtin_amdgcn_sched_barrier(0);  // (Q S while the quarters of W S come)
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) qs = __builtin_amdgcn_mfma_f32_16x16x4f32(x.qx[b][e], S[b][e], qs, 0, 0, 0);
    if (c > 0) deliver(c - 1);
    o_before = x.o;
    const v4f u = x.v - ((w0 + w1) + (w2 + w3));
#pragma unroll
    for (int b = 0; b < RB; ++b) S[b] = S[b] * x.d[b];
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int b = 0; b < RB; ++b) S[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[b][e], u[e], S[b], 0, 0, 0);
    p[1][wave][lane] = qs;
  };
  Operands x[SETS];
#pragma unroll
  for (int i = 0; i < SETS - 1; ++i) ask(min(i, chunks - 1), x[i]);
  // (whole turns of the sets, and what is left behind them: with a way out of the middle of a turn the compiler moves what was asked for
  // between registers at its end, and waits for all of it there)
  int c = 0;
#pragma unroll 1
  for (; c + SETS <= chunks; c += SETS) {
#pragma unroll
    for (int i = 0; i < SETS; ++i) {
      ask(min(c + i + SETS - 1, chunks - 1), x[(i + SETS - 1) % SETS]);  // (behind the last chunk that one again)
      walk(c + i, x[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < SETS - 1; ++i)
    if (c + i < chunks) walk(c + i, x[i]);
  __syncthreads();
  deliver(chunks - 1);
  if (col < a.dv) {
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int row = 16 * (wave * RB + b) + 4 * q + j;
        if (row < a.dk) s_col[row] = S[b][j];
      }
  }
}

template <typename T, int DKP>
static bool launch_factors_of(const DeltaChunkArgs& a, int n_chunks, size_t lds, hipStream_t stream) {
  auto kernel = delta_chunk_factors_kernel<T, DKP>;
  if (lds > 64 * 1024 && hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) return false;
  hipLaunchKernelGGL(kernel, dim3(n_chunks, a.H), dim3(256), lds, stream, a);
  return true;
}
template <typename T>
static bool launch_factors(const DeltaChunkArgs& a, int n_chunks, size_t lds, hipStream_t stream) {
  switch (a.dkp / 64) {
    case 1: return launch_factors_of<T, 64>(a, n_chunks, lds, stream);
    case 2: return launch_factors_of<T, 128>(a, n_chunks, lds, stream);
    case 3: return launch_factors_of<T, 192>(a, n_chunks, lds, stream);
    default: return launch_factors_of<T, 256>(a, n_chunks, lds, stream);
  }
}

TK_API int tk_delta_chunk_tokens() { return DC_CHUNK; }
TK_API int tk_delta_chunk_words(int dk, int dv) {
  return dk > 0 && dk <= DC_MAX_DK && dv > 0 && dv <= DC_MAX_DV ? (int)dc_words((dk + 63) / 64 * 64, (dv + 15) / 16 * 16) : 0;
}

// proj, a_pre, conv_w, a_log, dt_bias, state: as tk_delta_prepare takes them; chunk_req, chunk_row0 [n_chunks], chunk_first
// [n_requests + 1]: the step's rows in chunks of 16 in the requests' order (none for a request that is left out); rec: [n_chunks][H][tk_delta_chunk_words]; o: [tokens][H * dv].
// The convolutions' tails stay as they are (tk_delta_tail moves them on afterwards).
TK_API int tk_delta_chunks(int dt, const void* proj, int ld, int col_b, const float* a_pre, int ld_a, const float* conv_w, int taps,
                           const float* a_log, const float* dt_bias, float* state, size_t state_stride, size_t tail_off,
                           const int* q_start, const int* slots, const int* chunk_req, const int* chunk_row0, const int* chunk_first,
                           float* rec, float* o, int n_chunks, int n_requests, int H, int G, int dk, int dv, hipStream_t stream) {
  TK_REQUIRE(n_chunks >= 0 && n_requests >= 0 && H > 0 && G > 0 && H % G == 0 && tk_delta_chunk_words(dk, dv) > 0,
             "delta_chunks: bad sizes heads=%d kv heads=%d dk=%d dv=%d", H, G, dk, dv);
  TK_REQUIRE(taps >= 1 && taps <= DR_MAX_TAPS, "delta_chunks: %d taps (1..%d)", taps, DR_MAX_TAPS);
  const int C = 2 * G * dk + H * dv;
  TK_REQUIRE(ld >= C && col_b >= 0 && col_b + H <= ld && ld_a >= H * dk, "delta_chunks: row strides %d, %d too short", ld, ld_a);
  TK_REQUIRE((size_t)H * dv * dk <= tail_off && tail_off + (size_t)(taps - 1) * C <= state_stride, "delta_chunks: the state row is too short");
  TK_REQUIRE(H < 65536 && n_requests < 65536, "delta_chunks: too many heads or requests");
  if (n_chunks == 0 || n_requests == 0) return 0;
  DeltaChunkArgs a = {proj, ld, col_b, a_pre, ld_a, conv_w, taps, a_log, dt_bias, state, state_stride, tail_off, q_start, slots,
                      chunk_req, chunk_row0, chunk_first, rec, o, H, G, dk, dv, (dk + 63) / 64 * 64, (dv + 15) / 16 * 16};
  const size_t lds = sizeof(float) * ((size_t)DC_CHUNK * (3 * a.dkp + a.dvp) + 3 * DC_CHUNK * DC_LD + DC_CHUNK);
  const bool ok = dt == TK_F32 ? launch_factors<float>(a, n_chunks, lds, stream) : launch_factors<bf16_t>(a, n_chunks, lds, stream);
  TK_REQUIRE(ok, "delta_chunks: %zu bytes of local memory could not be reserved", lds);
  const dim3 grid(H, n_requests, a.dvp / 16);
  switch (a.dkp / 64) {
    case 1: hipLaunchKernelGGL(delta_chunk_walk_kernel<1>, grid, dim3(256), 0, stream, a); break;
    case 2: hipLaunchKernelGGL(delta_chunk_walk_kernel<2>, grid, dim3(256), 0, stream, a); break;
    case 3: hipLaunchKernelGGL(delta_chunk_walk_kernel<3>, grid, dim3(256), 0, stream, a); break;
    default: hipLaunchKernelGGL(delta_chunk_walk_kernel<4>, grid, dim3(256), 0, stream, a); break;
  }
  TK_CHECK_LAUNCH("delta_chunks");
  return 0;
}
