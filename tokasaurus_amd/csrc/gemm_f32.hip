// 32-bit matrix products on the matrix cores' 32-bit multiply-adds (v_mfma_f32_16x16x4_f32):
//     C[M,N] = A[M,K] * W[N,K]^T (+ bias[N]) (+ residual[M,N])
// for row-major operands whose rows start at multiples of 16 bytes (K and the stride of A
// multiples of 4; gemm_generic.hip has the kernels for any others).  Products and sums are
// 32-bit throughout: the instruction multiplies and adds 32-bit numbers, unsplit (but for products so many that their time counts, which
// gemm_f32_pieces_kernel makes of exact parts of the numbers, with smaller errors).
//
// A wavefront owns TM x TN blocks of 16 tokens x 16 weight rows.  In a block of 16 elements of K lane l holds elements
// 4 * (l / 16) .. + 3 of weight row l % 16 and of token l % 16; instruction s of the block then multiplies element s of
// every lane, so it sums the elements 4 q + s, q < 4, which is a permutation of K that both operands share.  Weights as
// the first operand: acc[j] of lane (r, q) = C[token r][weight row 4 q + j], a 16-byte store.
//
// Two kinds of kernels:
//   gemm_f32_few_kernel (up to 16 tokens, bound by reading W once): a workgroup's wavefronts cut K between them and add up
//     in the order of K; operands straight from memory to registers, two sets of them, so that one set's loads are in
//     flight while the other is multiplied.  Sixteen sums a result (one an instruction of a set) keep every chain of
//     additions at 32 to 64 elements: with one chain a wavefront the error is three times as large, at no gain.
//   gemm_f32_stream_kernel and, for a K that is no multiple of 32, gemm_f32_kernel (more tokens, bound by the matrix cores): four wavefronts share a tile's rows through local memory.
//     A compute unit's caches bring about 18 bytes a cycle: wavefronts that each load the operands of 32 x 32 results for
//     themselves need 32 and reach half of the matrix cores' rate (2 048 x 16 384 x 2 048: 76 TFLOP/s, straight from
//     memory or through local memory of their own); a shared tile of 64 x 64 needs 16, of 128 x 128 8.  Where the tiles are
//     too few to fill the chip K is cut among workgroups, whose sums a second kernel adds in the order of K.
// Measured against the plain kernels that this replaces (us; floors at 5.05 TB/s and 153 TFLOP/s): 4 tokens 2 048 x 2 048 6.9
// (floor 3.3), 2 048 x 8 192 17.5 (13), 16 384 x 2 048 29.5 (27); before 36 for the first two in the mean, and 33.  301
// tokens 2 048 x 2 048 38 (17), 2 048 x 8 192 116 (66), 3 072 x 2 048 53 (25), 16 384 x 2 048 207 (132); before 746 for
// the first two in the mean, 301 and 643 (gemm_f32_stream_kernel has the figures for K of a multiple of 32).  Errors against 64-bit
// sums: up to 32 tokens those of the plain kernel (1.2e-7 of the norm at 2 048 elements), beyond at most the plain kernel's.
#include "common.h"
#include <type_traits>

typedef float f4 __attribute__((ext_vector_type(4)));

struct GemmF32Args {
  const float* A;
  int lda;
  const float* W;
  float* C;
  int ldc;
  const float* residual;
  int ldr;
  const float* bias;
  int M, N, K;
  float* part;  // [cuts][M][N] sums of K's parts, or null: one part, finished here
};

// bias and residual, and the store of four neighbouring outputs of a token (of those whose bit in `only` is set)
__device__ __forceinline__ void gf_store(const GemmF32Args& a, f4 v, int token, int n, int only = 15) {
  float* c = a.C + (size_t)token * a.ldc + n;
  float o[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    o[j] = v[j];
    if (n + j < a.N) {
      if (a.bias) o[j] += a.bias[n + j];
      if (a.residual) o[j] += a.residual[(size_t)token * a.ldr + n + j];
    }
  }
  if (only == 15 && n + 3 < a.N && ((uintptr_t)c & 15) == 0) {
    *(f4*)c = (f4){o[0], o[1], o[2], o[3]};
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (n + j < a.N && (only >> j & 1)) c[j] = o[j];
  }
}

#define GF_HALVES_ROWS 2048  // weight rows up to which the few-row kernel takes 8 a workgroup: one for each of 256 compute units
#define GF_UNROLL 4  // blocks of 16 elements a set of loads

// HALVES (up to 8 tokens, K a multiple of 32): a workgroup has 8 weight rows, and the unused half of the matrix core's rows and of its
// columns takes the next 16 elements of K (the blocks of results off the diagonal are not used), so that a weight of few rows gives
// every compute unit a workgroup and a load takes whole lines of 128 bytes.  4 tokens, us by rows of 16 / of 8, weights from memory: 2,048 x
// 2,048 8.6 / 6.9, 2,048 x 8,192 26.4 / 17.5, 3,072 x 2,048 8.8 / 9.6, 16,384 x 2,048 26.8 / 31.2 (these of 8 with the other half's elements
// a half of K on, 1 to 8 tokens at 2,048 x 4,096 9.8 to 12.4, now 8.4 to 10.3).  Each chain of sums is half as long: error 1.2e-7 / 1.0e-7 of
// the norm over 2,048 elements, 1.6e-7 / 1.3e-7 over 8,192.
// A wavefront's walk begins at a set that the workgroup's number gives, those of one die at different ones: begun at the first by
// all, rows of 32 and 64 KB keep to few of the memory's channels (us together / apart: 2,048 x 8,192 19.4 / 15.0 at 1 token, 19.4 / 15.4 at 4,
// 2,048 x 16,384 29.9 / 24.0 and 30.2 / 26.5, 2,048 x 11,008 21.4 / 19.9 and 22.0 / 20.6, else within 2 %).  One order for all rows up to 8, whatever
// their number: a step of 3 rows is recorded with 4.
//
// What a step of few rows would launch a kernel for behind the product (4 rows of the 1B shape: rotation and append 4.9 us, activation 4.6,
// each little more than a launch and a trip to memory) is done where the results pass anyway:
// EPI = FEW_GLU: W is [gate | up], 8 rows of each a workgroup, so that a gate and its up lie 32 lanes apart: silu(gate) * up.
// EPI = FEW_ROPE: W is [q | k | v] by heads, a workgroup's rows are 8 elements of a head and the 8 half a head on, which the
//   rotation pairs: q turned to its rows, k turned and v as it is to their pages.
// (The norm in front of a product does not pay here: its weight is a third load beside those of A and W, in every workgroup; gate and
// up with the norm folded in 31.9 us for 26.2 and the norm's own 4.5, the head 209 for 182.)
enum { FEW_STORE = 0, FEW_GLU = 1, FEW_ROPE = 2 };
struct FewExtra {
  // FEW_ROPE: positions and requests of the rows, the requests' pages, cosines and sines [positions][d / 2] (null: no rotation)
  const int *positions, *token_req, *block_table;
  int table_stride;
  const float *cos, *sin;
  float *kcache, *vcache;
  int nq, nkv, d, P;
};

template <bool HALVES, int EPI>
__global__ __launch_bounds__(512) void gemm_f32_few_kernel(GemmF32Args a, FewExtra more, int KS, int share, int spare) {
  static_assert(!HALVES || EPI == FEW_STORE, "");
  extern __shared__ __align__(16) f4 sums[];  // [wavefronts - 1][64]
  // every argument that a first load needs, in one trip
  asm volatile("" ::"s"(a.A), "s"(a.W), "s"(a.lda), "s"(a.M), "s"(a.N), "s"(a.K), "s"(KS), "s"(share), "s"(spare));
  // (the wavefront's number as one value for all its lanes, so that its loop counts in scalar registers)
  const int lane = threadIdx.x & 63, kw = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, q = lane >> 4;
  constexpr int ROWS = HALVES ? 8 : 16;
  const int n0 = blockIdx.x * ROWS, own = HALVES ? r & 7 : r;
  const int from = HALVES ? (r >> 3) * 16 : 0;
  constexpr int STEP = HALVES ? 32 : 16;  // elements of K a block and its partner are on
  const int blocks = HALVES ? a.K >> 5 : (a.K + 15) >> 4;
  // (the last wavefronts take one block more, so that a block that K cuts lies behind whole sets: 4 tokens, 2,048 x
  // 2,056 9.2 / 8.1 us, 1 token 8.6 / 7.5)
  const int b0 = kw * share + max(kw - (KS - spare), 0), b1 = b0 + share + (kw >= KS - spare ? 1 : 0);
  // (FEW_GLU, FEW_ROPE: a.N outputs in pairs, of which a workgroup has 8)
  int w_row = min(n0 + own, a.N - 1), first = 0, head = 0;
  if (EPI == FEW_GLU) {
    first = blockIdx.x * 8;
    w_row = min(first + (r & 7), a.N / 2 - 1) + (r >> 3) * (a.N / 2);
  }
  if (EPI == FEW_ROPE) {
    const int each = more.d >> 4;
    head = blockIdx.x / each;
    first = (blockIdx.x - head * each) * 8;
    w_row = head * more.d + first + (r & 7) + (r >> 3) * (more.d >> 1);
  }
  const float* wp = a.W + (size_t)w_row * a.K + from + 4 * q;
  const float* ap = a.A + (size_t)min(own, a.M - 1) * a.lda + from + 4 * q;
  f4 acc[GF_UNROLL][4];
#pragma unroll
  for (int u = 0; u < GF_UNROLL; ++u)
#pragma unroll
    for (int s = 0; s < 4; ++s) acc[u][s] = (f4){0.f, 0.f, 0.f, 0.f};
  f4 w[2][GF_UNROLL], x[2][GF_UNROLL];
  // (nothing moves across the end of a set's loads: the compiler would else sink each load to its first use and wait there)
#define GF_LOAD(set, b)                                                                             \
  do {                                                                                              \
    _Pragma("unroll") for (int u = 0; u < GF_UNROLL; ++u) {                                         \
      w[set][u] = *(const f4*)(wp + (size_t)(place(b) + u) * STEP);                                 \
      x[set][u] = *(const f4*)(ap + (size_t)(place(b) + u) * STEP);                                 \
    }                                                                                               \
    __builtin_amdgcn_sched_barrier(0);                                                              \
  } while (0)
#define GF_MULTIPLY(set)                                                                            \
  _Pragma("unroll") for (int u = 0; u < GF_UNROLL; ++u) _Pragma("unroll") for (int s = 0; s < 4; ++s) \
      acc[u][s] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[set][u][s], x[set][u][s], acc[u][s], 0, 0, 0)
  const int exact = HALVES || (a.K & 15) == 0 ? b1 : min(b1, blocks - 1);  // blocks up to here lie inside K whole
  const int sets = max(exact - b0, 0) / GF_UNROLL;
  const int turn = HALVES && sets > 0 ? (int)((blockIdx.x >> 3) % (unsigned)sets) * GF_UNROLL : 0;
  auto place = [&](int at) { return !HALVES ? at : (at + turn < b0 + sets * GF_UNROLL ? at + turn : at + turn - sets * GF_UNROLL); };
  int b = b0;
  if (sets > 0) {
    GF_LOAD(0, b);
    int s = 0;
#pragma unroll 1
    for (; s + 2 < sets; s += 2, b += 2 * GF_UNROLL) {
      GF_LOAD(1, b + GF_UNROLL);
      GF_MULTIPLY(0);
      GF_LOAD(0, b + 2 * GF_UNROLL);
      GF_MULTIPLY(1);
    }
    if (s + 1 < sets) {
      GF_LOAD(1, b + GF_UNROLL);
      GF_MULTIPLY(0);
      GF_MULTIPLY(1);
      b += 2 * GF_UNROLL;
    } else {
      GF_MULTIPLY(0);
      b += GF_UNROLL;
    }
  }
#undef GF_LOAD
#undef GF_MULTIPLY
#pragma unroll 1
  for (; b < b1; ++b) {  // what is left, the last block perhaps cut by K: zeros behind it
    const bool in = HALVES || b * 16 + 4 * q < a.K;
    const long off = in ? (long)b * STEP : -4L * q;
    f4 wv = *(const f4*)(wp + off), xv = *(const f4*)(ap + off);
    if (!in) wv = xv = (f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s) acc[0][s] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[s], xv[s], acc[0][s], 0, 0, 0);
  }
  f4 part[GF_UNROLL];
#pragma unroll
  for (int u = 0; u < GF_UNROLL; ++u) part[u] = (acc[u][0] + acc[u][1]) + (acc[u][2] + acc[u][3]);
  f4 sum = (part[0] + part[1]) + (part[2] + part[3]);
  if (KS > 1) {
    if (kw > 0) sums[(kw - 1) * 64 + lane] = sum;
    __syncthreads();
    if (kw > 0) return;
#pragma unroll 4
    for (int k = 0; k < KS - 1; ++k) sum += sums[k * 64 + lane];
  }
  if (HALVES) {  // the partners' sums of token r lie in the lanes of token r + 8 and of rows 8 more
#pragma unroll
    for (int j = 0; j < 4; ++j) sum[j] += __shfl(sum[j], (lane + 40) & 63, 64);
  }
  if (EPI == FEW_STORE) {
    if (r < min(a.M, ROWS) && 4 * q < ROWS && n0 + 4 * q < a.N) gf_store(a, sum, r, n0 + 4 * q);
    return;
  }
  f4 other;  // lanes of the first 8 rows: their partners
  if (a.bias) {
    const int n = EPI == FEW_GLU ? (q >> 1) * (a.N / 2) + first + 4 * (q & 1) : head * more.d + (q >> 1) * (more.d >> 1) + first + 4 * (q & 1);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (EPI == FEW_ROPE || first + 4 * (q & 1) + j < a.N / 2) sum[j] += a.bias[n + j];
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) other[j] = __shfl_xor(sum[j], 32, 64);
  if (r >= a.M) return;
  if (EPI == FEW_GLU) {
    const int n = first + 4 * q;
    if (q >= 2) return;
    float* c = a.C + (size_t)r * a.ldc + n;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (n + j < a.N / 2) c[j] = sum[j] / (1.0f + expf(-sum[j])) * other[j];
    return;
  }
  const int pos = more.positions[r], pair = first + 4 * (q & 1), e = pair + (q >> 1) * (more.d >> 1);
  f4 o = sum;
  if (head < more.nq + more.nkv && more.cos) {
    const f4 cs = *(const f4*)(more.cos + (size_t)pos * (more.d >> 1) + pair), sn = *(const f4*)(more.sin + (size_t)pos * (more.d >> 1) + pair);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float u = q < 2 ? sum[j] : other[j], v = q < 2 ? other[j] : sum[j];
      rotate_pair(u, v, cs[j], sn[j], u, v);
      o[j] = q < 2 ? u : v;
    }
  }
  if (head < more.nq) {
    *(f4*)(a.C + (size_t)r * a.ldc + head * more.d + e) = o;
    return;
  }
  const size_t page = more.block_table[(size_t)more.token_req[r] * more.table_stride + pos / more.P];
  const int p = pos % more.P;
  if (head < more.nq + more.nkv) {
    *(f4*)(more.kcache + (page * more.nkv + head - more.nq) * key_page_elems(more.P, more.d) + key_offset(more.P, p, e)) = o;
  } else {
    float* v = more.vcache + (page * more.nkv + head - more.nq - more.nkv) * more.P * more.d;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[value_offset(more.d, p, e + j)] = o[j];
  }
}

// The chains of a tile's sums added, and the results stored, or the part of K among the other parts' sums.  MASKED: of this lane's 4 TN TM
// results only those whose bit (t, u, j) in `only` is set.
template <int TM, int TN, int CHAINS, bool MASKED = false>
__device__ __forceinline__ void gf_finish(const GemmF32Args& a, f4 (&acc)[CHAINS][TN][TM], int m0, int n0, int wave, int r, int q, uint64_t only = 0) {
#pragma unroll
  for (int half = CHAINS / 2; half > 0; half /= 2)
#pragma unroll
    for (int c = 0; c < half; ++c)
#pragma unroll
      for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int u = 0; u < TM; ++u) acc[c][t][u] += acc[c + half][t][u];
#pragma unroll
  for (int u = 0; u < TM; ++u) {
    const int token = m0 + (wave >> 1) * 16 * TM + 16 * u + r;
    if (token >= a.M) continue;
#pragma unroll
    for (int t = 0; t < TN; ++t) {
      const int n = n0 + (wave & 1) * 16 * TN + 16 * t + 4 * q;
      if (n >= a.N) continue;
      const int some = MASKED ? (int)(only >> (4 * (t * TM + u))) & 15 : 15;
      if (MASKED && some == 0) continue;
      if (a.part) {  // (N is a multiple of 4 then)
        float* part = a.part + ((size_t)blockIdx.y * a.M + token) * a.N + n;
        if (!MASKED) {
          *(f4*)part = acc[0][t][u];
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (some >> j & 1) part[j] = acc[0][t][u][j];
        }
      } else {
        gf_store(a, acc[0][t][u], token, n, some);
      }
    }
  }
}

#define GS_ROW 36  // floats a row of 32 takes in local memory: 16 lanes that read 16 rows at one place meet 64 different banks

// A workgroup: a tile of 32 TM tokens x 32 TN weight rows, its four wavefronts a quarter each, over the steps of 32 elements
// of K that its cut (blockIdx.y) has.  A load brings 8 rows' 128 bytes.  Two tiles' rows in local memory: while one is read
// the next step's, which have been in flight for a step, are written to the other, and the step after that is asked for.
// CHAINS sums a result, added at the end: 8 for the smallest tile, which then is as exact as the few-row kernel (registers
// are free there), else 1.
template <int TM, int TN, int CHAINS>
__global__ __launch_bounds__(256) void gemm_f32_kernel(GemmF32Args a) {
  extern __shared__ __align__(16) float tile[];  // [2][32 * (TN + TM)][GS_ROW], weight rows first
  constexpr int ROWS = 32 * (TN + TM), LOADS = ROWS / 32;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4;
  // Workgroups that share weight rows run on one die (the hardware deals workgroups to the eight dies in turn), so that
  // those rows pass through one L2: the number is [groups of 8 column tiles][row tiles][column tile within the 8].
  const int mt = (a.M + 32 * TM - 1) / (32 * TM);
  const int g = blockIdx.x / 8;
  const int n0 = ((g / mt) * 8 + blockIdx.x % 8) * 32 * TN, m0 = (g % mt) * 32 * TM;
  if (n0 >= a.N) return;  // the same for the whole workgroup
  const int steps = (a.K + 31) >> 5;
  const int s0 = (int)((long)steps * blockIdx.y / gridDim.y), s1 = (int)((long)steps * (blockIdx.y + 1) / gridDim.y);
  const int lr = tid >> 3, lc = (tid & 7) * 4;  // load i brings rows 32 i + lr, 16 bytes a lane
  const float* src[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i)
    src[i] = i < TN ? a.W + (size_t)min(n0 + 32 * i + lr, a.N - 1) * a.K + lc
                    : a.A + (size_t)min(m0 + 32 * (i - TN) + lr, a.M - 1) * a.lda + lc;
  f4 acc[CHAINS][TN][TM];
#pragma unroll
  for (int c = 0; c < CHAINS; ++c)
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
      for (int u = 0; u < TM; ++u) acc[c][t][u] = (f4){0.f, 0.f, 0.f, 0.f};
  f4 next[LOADS];
  auto load = [&](int s) {
    if (s * 32 + 32 <= a.K) {
#pragma unroll
      for (int i = 0; i < LOADS; ++i) next[i] = *(const f4*)(src[i] + (size_t)s * 32);
    } else {  // K ends inside the step: zeros behind it
      const bool in = s * 32 + lc < a.K;
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        next[i] = *(const f4*)(src[i] + (in ? (long)s * 32 : -(long)lc));
        if (!in) next[i] = (f4){0.f, 0.f, 0.f, 0.f};
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // (the compiler would else sink the loads to where they are stored)
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) *(f4*)(tile + ((size_t)buf * ROWS + 32 * i + lr) * GS_ROW + lc) = next[i];
  };
  const float* wrow = tile + ((wave & 1) * 16 * TN + r) * GS_ROW + 4 * q;
  const float* xrow = tile + (32 * TN + (wave >> 1) * 16 * TM + r) * GS_ROW + 4 * q;
  load(s0);
  store(0);
  load(min(s0 + 1, s1 - 1));
  __syncthreads();
#pragma unroll 1
  for (int s = s0; s < s1; ++s) {
    const int buf = (s - s0) & 1;
    f4 w[2][TN], x[2][TM];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
#pragma unroll
      for (int t = 0; t < TN; ++t) w[b][t] = *(const f4*)(wrow + (buf * ROWS + 16 * t) * GS_ROW + 16 * b);
#pragma unroll
      for (int t = 0; t < TM; ++t) x[b][t] = *(const f4*)(xrow + (buf * ROWS + 16 * t) * GS_ROW + 16 * b);
    }
    store(buf ^ 1);
    load(min(s + 2, s1 - 1));  // (the last two steps load one again that nobody reads)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int t = 0; t < TN; ++t)
#pragma unroll
          for (int u = 0; u < TM; ++u) {
            const int c = (4 * b + e) % CHAINS;
            acc[c][t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[b][t][e], x[b][u][e], acc[c][t][u], 0, 0, 0);
          }
    __syncthreads();
  }
  gf_finish<TM, TN, CHAINS>(a, acc, m0, n0, wave, r, q);
}

// The same for a K of a multiple of 32, with the same bits: rows of A and W go straight from memory to local memory, STAGES - 1 steps
// ahead, with no registers between, the 16-byte piece c of a row at place c ^ gs_swizzle(row), which 16 lanes that read 16
// rows at one place find in 64 different banks.  Through registers a compute unit gets about 18 bytes a cycle, and a tile of 64 x 64 needs
// 16 at the matrix cores' full rate.  us through registers / straight, weights from memory: 301 tokens 16,384 x 2,048 192 / 177, 2,048 x
// 8,192 105 / 97, 3,072 x 2,048 48.3 / 44.6; 100 tokens 90 / 81, 50 / 46, 24.1 / 22.5; 17 tokens 44.6 / 40.0, 27.8 / 24.8, 13.9 / 12.4; 2,048 tokens
// 1,117 / 1,018 (135 TFLOP/s), 604 / 559, 229 / 213.
__device__ __forceinline__ int gs_swizzle(int row) { return (row ^ (row >> 3 & 1)) & 7; }

template <int TM, int TN, int CHAINS, int STAGES>
__global__ __launch_bounds__(256) void gemm_f32_stream_kernel(GemmF32Args a) {
  extern __shared__ __align__(16) float tile[];  // [STAGES][32 * (TN + TM)][32], weight rows first
  constexpr int ROWS = 32 * (TN + TM), LOADS = ROWS / 32;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int mt = (a.M + 32 * TM - 1) / (32 * TM);  // (workgroups on the dies as in gemm_f32_kernel)
  const int g = blockIdx.x / 8;
  const int n0 = ((g / mt) * 8 + blockIdx.x % 8) * 32 * TN, m0 = (g % mt) * 32 * TM;
  if (n0 >= a.N) return;  // the same for the whole workgroup
  const int all = a.K >> 5;
  const int s0 = (int)((long)all * blockIdx.y / gridDim.y), steps = (int)((long)all * (blockIdx.y + 1) / gridDim.y) - s0;
  const int lr = 8 * wave + (lane >> 3);  // load i brings row 32 i + lr
  const int lc = ((lane & 7) ^ gs_swizzle(lr)) * 4;
  const float* src[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i)
    src[i] = (i < TN ? a.W + (size_t)min(n0 + 32 * i + lr, a.N - 1) * a.K : a.A + (size_t)min(m0 + 32 * (i - TN) + lr, a.M - 1) * a.lda) + lc + (size_t)s0 * 32;
  const unsigned lds = (unsigned)(uintptr_t)(__attribute__((address_space(3))) float*)tile;
  auto ask = [&](int step, int place) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      load_to_lds((const bf16_t*)(src[i] + (size_t)step * 32), lds + (unsigned)((place * ROWS + 32 * i + 8 * wave) * 32 * (int)sizeof(float)));
  };
  for (int s = 0; s < STAGES - 1 && s < steps; ++s) ask(s, s);
  f4 acc[CHAINS][TN][TM];
#pragma unroll
  for (int c = 0; c < CHAINS; ++c)
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
      for (int u = 0; u < TM; ++u) acc[c][t][u] = (f4){0.f, 0.f, 0.f, 0.f};
  const int piece[2] = {(q ^ gs_swizzle(r)) * 4, ((4 + q) ^ gs_swizzle(r)) * 4};
  const float* wrow = tile + ((wave & 1) * 16 * TN + r) * 32;
  const float* xrow = tile + (32 * TN + (wave >> 1) * 16 * TM + r) * 32;
  int here = 0, next = STAGES - 1;
#pragma unroll 1
  for (int s = 0; s < steps; ++s) {
    // the step is there when only the loads of the STAGES - 2 behind it are left; behind the barrier every wavefront's are,
    // and every wavefront is through with the step before, whose place is filled again
    if (s + STAGES - 2 < steps) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((STAGES - 2) * LOADS) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (s + STAGES - 1 < steps) ask(s + STAGES - 1, next);
    f4 w[2][TN], x[2][TM];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
#pragma unroll
      for (int t = 0; t < TN; ++t) w[b][t] = *(const f4*)(wrow + (here * ROWS + 16 * t) * 32 + piece[b]);
#pragma unroll
      for (int t = 0; t < TM; ++t) x[b][t] = *(const f4*)(xrow + (here * ROWS + 16 * t) * 32 + piece[b]);
    }
    here = here + 1 == STAGES ? 0 : here + 1;
    next = next + 1 == STAGES ? 0 : next + 1;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int t = 0; t < TN; ++t)
#pragma unroll
          for (int u = 0; u < TM; ++u) {
            const int c = (4 * b + e) % CHAINS;
            acc[c][t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[b][t][e], x[b][u][e], acc[c][t][u], 0, 0, 0);
          }
  }
  gf_finish<TM, TN, CHAINS>(a, acc, m0, n0, wave, r, q);
}

// Many products over a K of a multiple of 32: the numbers as exact sums of three bfloat16 numbers (their 24 bits, 8 at a time, by truncation)
// on the matrix cores' bfloat16 multiply-adds, whose products are exact and whose sums are 32-bit.  Of the nine products of pieces all count but that
// of the two smallest, under 2^-30 of the whole (without the next two, (1, 2) and (2, 1), up to 2^-21 would be left out, always towards zero: a
// product by itself would be off by 6.5e-8 root mean square and 4.5e-7 at most, where a rounding is 2.5e-8 and 6.0e-8).  The largest are summed by
// themselves, one rounding for 32 elements where the 32-bit instruction rounds after every fourth, the others beside them: errors against 64 bits
// are not larger than the unsplit products', from one term a row to dense rows (below).
// Eight instructions of 16 x 16 x 32 take 136 cycles where eight of 16 x 16 x 4 take 272; the pieces, made by every wavefront for itself, cost nearly as
// much as the products, side by side with them where two workgroups share a compute unit.
// Pieces reach down to 2^-133, and an infinite number has pieces that are no numbers: results that are not finite, or below GP_LEAST (zero too:
// numbers of less than 2^-133 have no pieces at all), or of a row of A or W with an operand of GP_MOST and more, are made again, unsplit, by the
// workgroup that has them.  Else the bits below 2^-133 that are lost are at most 2^-102 of each of the K products, K 2^-52 of a result.  Which
// way a result is made depends on its own two rows alone, not on what else is in its tile (so a row of zeros costs its tiles their time
// twice, and changes no other row).
// Two wavefronts make the pieces of the same rows: each looks at half a step's numbers, which the other has last (16 instructions of some 370 a
// step; 301 rows 16,384 x 2,048 151.9 us without, 152.1 with, 2,048 rows 697 and 700).
// us unsplit / split, weights from memory:
//   33 rows   16,384 x 2,048 50.1 / 46.2, 2,048 x 8,192 32.5 / 29.6, 128,256 x 2,048 512 / 288
//   200       16,384 x 2,048 146 / 121, 2,048 x 8,192 79.2 / 65.1, 2,048 x 2,048 28.5 / 25.4
//   301       16,384 x 2,048 177 / 168, 2,048 x 8,192 96.6 / 89.8, 2,048 x 2,048 32.7 / 30.2, 3,072 x 2,048 44.6 / 39.2
//   2,048     16,384 x 2,048 1,020 / 840, 2,048 x 8,192 565 / 423, 2,048 x 2,048 145 / 127
// Errors, root of the squares' sums over that of the results, unsplit / split: 70 rows 7,300 x 1,024 2.9e-7 / 9.8e-8, of numbers in [1, 2) 1.27e-7 / 4.5e-8,
// of 2, 8 and 32 terms a row 3.5e-8 / 3.5e-8, 5.2e-8 / 5.2e-8 and 6.8e-8 / 5.0e-8; 2,048 rows 2,048 x 2,048 8.1e-7 / 2.7e-7, in [1, 2) 6.8e-7 / 2.5e-7, of 1, 2,
// 8 and 32 terms 2.53e-8 / 2.53e-8, 3.1e-8 / 2.6e-8, 5.4e-8 / 2.8e-8 and 1.0e-7 / 4.3e-8.
typedef __attribute__((ext_vector_type(8))) __bf16 gf_bf16x8_t;

// (most: the greatest number of `lo` so far)
__device__ __forceinline__ void gf_pieces(f4 lo, f4 hi, gf_bf16x8_t (&piece)[3], float& most) {
  // (one instruction for two numbers; of the compiler's maximum each would first be made a quiet number)
  asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(most) : "v"(lo[0]), "v"(lo[1]));
  asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(most) : "v"(lo[2]), "v"(lo[3]));
  float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
  for (int n = 0; n < 3; ++n) {
    uint32_t packed[4];
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      const uint32_t ua = __float_as_uint(v[i]), ub = __float_as_uint(v[i + 1]);
      packed[i / 2] = __builtin_amdgcn_perm(ub, ua, 0x07060302);  // the upper halves, the first below
      if (n < 2) {
        v[i] -= __uint_as_float(ua & 0xffff0000u);
        v[i + 1] -= __uint_as_float(ub & 0xffff0000u);
      }
    }
    __builtin_memcpy(&piece[n], packed, sizeof(piece[n]));
  }
}

#define GP_LEAST 0x1p-50f
#define GP_MOST 0x1p30f
#define GP_STAGES 2  // steps in local memory: two workgroups of the largest tile share a compute unit
template <int TM, int TN>
__global__ __launch_bounds__(256, 2) void gemm_f32_pieces_kernel(GemmF32Args a) {
  extern __shared__ __align__(16) float tile[];  // [GP_STAGES][32 * (TN + TM)][32], weight rows first, pieces in places as above
  constexpr int ROWS = 32 * (TN + TM), LOADS = ROWS / 32, STAGES = GP_STAGES;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int mt = (a.M + 32 * TM - 1) / (32 * TM);  // (workgroups on the dies as in gemm_f32_kernel)
  const int g = blockIdx.x / 8;
  const int n0 = ((g / mt) * 8 + blockIdx.x % 8) * 32 * TN, m0 = (g % mt) * 32 * TM;
  if (n0 >= a.N) return;  // the same for the whole workgroup
  const int all = a.K >> 5;
  const int s0 = (int)((long)all * blockIdx.y / gridDim.y), steps = (int)((long)all * (blockIdx.y + 1) / gridDim.y) - s0;
  const int lr = 8 * wave + (lane >> 3);  // load i brings row 32 i + lr
  const int lc = ((lane & 7) ^ gs_swizzle(lr)) * 4;
  const float* src[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i)
    src[i] = (i < TN ? a.W + (size_t)min(n0 + 32 * i + lr, a.N - 1) * a.K : a.A + (size_t)min(m0 + 32 * (i - TN) + lr, a.M - 1) * a.lda) + lc + (size_t)s0 * 32;
  const unsigned lds = (unsigned)(uintptr_t)(__attribute__((address_space(3))) float*)tile;
  auto ask = [&](int step, int place) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      load_to_lds((const bf16_t*)(src[i] + (size_t)step * 32), lds + (unsigned)((place * ROWS + 32 * i + 8 * wave) * 32 * (int)sizeof(float)));
  };
  f4 acc[1][TN][TM], small[TN][TM];
  const int last = 4 * ((wave ^ (wave >> 1)) & 1);  // the halves of a step change places between wavefronts that share rows
  const int piece[2] = {((last + q) ^ gs_swizzle(r)) * 4, ((4 - last + q) ^ gs_swizzle(r)) * 4};
  const float* wrow = tile + ((wave & 1) * 16 * TN + r) * 32;
  const float* xrow = tile + (32 * TN + (wave >> 1) * 16 * TM + r) * 32;
  float most = 0.f;
  auto walk = [&](auto unsplit) {
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
      for (int u = 0; u < TM; ++u) acc[0][t][u] = small[t][u] = (f4){0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < STAGES - 1 && s < steps; ++s) ask(s, s);
    int here = 0, next = STAGES - 1;
#pragma unroll 1
    for (int s = 0; s < steps; ++s) {
      if (s + STAGES - 2 < steps) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((STAGES - 2) * LOADS) : "memory");
      else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if (s + STAGES - 1 < steps) ask(s + STAGES - 1, next);
      const float *wr = wrow + here * ROWS * 32, *xr = xrow + here * ROWS * 32;
      if constexpr (decltype(unsplit)::value) {
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int u = 0; u < TM; ++u) {
            const f4 x = *(const f4*)(xr + 16 * u * 32 + piece[b]);
#pragma unroll
            for (int t = 0; t < TN; ++t) {
              const f4 w = *(const f4*)(wr + 16 * t * 32 + piece[b]);
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[0][t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[e], x[e], acc[0][t][u], 0, 0, 0);
            }
          }
      } else {
        gf_bf16x8_t w[TN][3];
#pragma unroll
        for (int t = 0; t < TN; ++t) gf_pieces(*(const f4*)(wr + 16 * t * 32 + piece[0]), *(const f4*)(wr + 16 * t * 32 + piece[1]), w[t], most);
#pragma unroll
        for (int u = 0; u < TM; ++u) {
          gf_bf16x8_t x[3];
          gf_pieces(*(const f4*)(xr + 16 * u * 32 + piece[0]), *(const f4*)(xr + 16 * u * 32 + piece[1]), x, most);
#define GP_PRODUCTS(SUM, I, J) \
  _Pragma("unroll") for (int t = 0; t < TN; ++t) SUM = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[t][I], x[J], SUM, 0, 0, 0)
          GP_PRODUCTS(small[t][u], 2, 1);
          GP_PRODUCTS(small[t][u], 1, 2);
          GP_PRODUCTS(small[t][u], 2, 0);
          GP_PRODUCTS(small[t][u], 0, 2);
          GP_PRODUCTS(small[t][u], 1, 1);
          GP_PRODUCTS(small[t][u], 1, 0);
          GP_PRODUCTS(small[t][u], 0, 1);
          GP_PRODUCTS(acc[0][t][u], 0, 0);
#undef GP_PRODUCTS
        }
      }
      here = here + 1 == STAGES ? 0 : here + 1;
      next = next + 1 == STAGES ? 0 : next + 1;
    }
  };
  walk(std::integral_constant<bool, false>{});
  // which results go unsplit: a bit each
  uint64_t again = 0;
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int u = 0; u < TM; ++u) {
      acc[0][t][u] += small[t][u];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float size = fabsf(acc[0][t][u][j]);
        again |= (uint64_t)!(size >= GP_LEAST && size < INFINITY) << (4 * (t * TM + u) + j);
      }
    }
  const bool large = !(most < GP_MOST);
  if (!__syncthreads_or(large || again != 0)) {
    gf_finish<TM, TN, 1>(a, acc, m0, n0, wave, r, q);
    return;
  }
  if (__syncthreads_or(large)) {
    // the rows with such operands, a thread a row (none is read behind its cut of K)
    if (tid < ROWS) {
      const float* row = tid < 32 * TN ? a.W + (size_t)min(n0 + tid, a.N - 1) * a.K : a.A + (size_t)min(m0 + tid - 32 * TN, a.M - 1) * a.lda;
      float top = 0.f;
      for (int k = s0 * 32; k < (s0 + steps) * 32; k += 4) {
        const f4 v = *(const f4*)(row + k);
        top = fmaxf(fmaxf(fmaxf(top, fabsf(v[0])), fmaxf(fabsf(v[1]), fabsf(v[2]))), fabsf(v[3]));
      }
      tile[tid] = top;
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
      for (int u = 0; u < TM; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float top = fmaxf(tile[(wave & 1) * 16 * TN + 16 * t + 4 * q + j], tile[32 * TN + (wave >> 1) * 16 * TM + 16 * u + r]);
          again |= (uint64_t)!(top < GP_MOST) << (4 * (t * TM + u) + j);
        }
    __syncthreads();
  }
  gf_finish<TM, TN, 1, true>(a, acc, m0, n0, wave, r, q, ~again);
  walk(std::integral_constant<bool, true>{});
  gf_finish<TM, TN, 1, true>(a, acc, m0, n0, wave, r, q, again);
}

// The sums of K's parts added in the order of K: a thread four neighbouring outputs.
__global__ __launch_bounds__(256) void gemm_f32_sum_kernel(GemmF32Args a, int cuts) {
  const int n = (blockIdx.x * blockDim.x + threadIdx.x) * 4, token = blockIdx.y;
  if (n >= a.N) return;
  const float* p = a.part + (size_t)token * a.N + n;
  f4 v = *(const f4*)p;
#pragma unroll 8
  for (int c = 1; c < cuts; ++c) v += *(const f4*)(p + (size_t)c * a.M * a.N);
  gf_store(a, v, token, n);
}

// Whether the kernels take the operands: rows at multiples of 16 bytes.
TK_API int tk_gemm_f32_takes(const void* A, int lda, const void* W, int K) {
  return ((((uintptr_t)A | (uintptr_t)W) & 15) == 0 && (lda & 3) == 0 && (K & 3) == 0) ? 1 : 0;
}

// workgroups of tiles of 32 tm tokens x 32 tn weight rows (their number over the columns is filled up to eights, see the kernel)
static long gf_tiles(int M, int N, int tm, int tn) {
  return (((long)N + 32 * tn - 1) / (32 * tn) + 7) / 8 * 8 * (((long)M + 32 * tm - 1) / (32 * tm));
}

// Whether gemm_f32_sum_kernel takes parts of these results: four columns a thread, a row of workgroups a token.
static bool gf_cuts_add(int M, int N) { return (N & 3) == 0 && M < 65536; }

// Whether products go by bfloat16 pieces: the rows of a tile (64 or 128, 128 weight rows), 0 if not; and into how many parts they cut K, the same
// for both ends of a call.  They pay from 7 * 2^27 multiply-adds on (rows counted in tiles of 64), where the steps' work outweighs a longer beginning:
// 200 rows 2,816 x 1,024 25.3 / 25.4 us, 160 rows 2,048 x 2,048 25.8 / 27.7, 128 rows 3,072 x 2,048 26.6 / 27.0, 64 rows 19.7 / 21.5 (with six of
// the eight products); 400 rows 8,192 x 256 26.5 / 20.8 and 4,096 x 512 29.6 / 25.7, 200 rows 2,048 x 2,048 28.5 / 25.4.
// Tile and parts are those of the least time by the steps of 32 elements of K that a compute unit takes one after the other (in proportion to
// a step's time with one workgroup on it and with two, which fit: 1.25 and 1.9 us for 64 rows, 1.95 and 3.4 for 128) and the parts' way through memory.
// What it takes was the best of 1 to 4 parts and its own, or within 1 % of it, at twenty sizes of 64 to 4,096 rows.
static int gf_pieces_tile(int M, int N, int K, int* cuts) {
  const long most = K / 256 < 32 ? K / 256 : 32, steps = K / 32;
  if (M <= 32 || K % 32 != 0 || most < 1 || ((long)M + 63) / 64 * 64 * N * K < 7L << 27) return 0;
  double best = 0;
  int tile = 0;
  for (int tm = 2; tm <= 4; tm += 2)
    for (int c = 1; c <= (gf_cuts_add(M, N) ? most : 1); ++c) {
      const long groups = gf_tiles(M, N, tm, 4) * c, rest = groups % 512;
      const double one = tm == 2 ? 1.05 : 1.6, two = tm == 2 ? 1.58 : 2.75;
      const double us = (groups / 512 * two + (rest == 0 ? 0 : (rest <= 256 ? one : two))) * ((steps + c - 1) / c) + (c > 1 ? 2 + c * (4e-6 / 3) * M * N : 0);
      if (tile == 0 || us < best) best = us, tile = 32 * tm, *cuts = c;
    }
  return tile;
}

// How many parts K is cut into among workgroups (the caller brings M * N floats for each where there is more than one):
// so many that the tiles times the parts are about five workgroups a compute unit, of 256 elements of K at least.  In us at
// 1 / 2 / 4 / 8 / 16 parts: 301 tokens 2 048 x 8 192 (160 tiles) 188 / 170 / 124 / 108 / 111; 600 tokens (320 tiles) 329 / 240 /
// 199 / 199 / 207; 301 tokens 3 072 x 2 048 (240 tiles) 49 / 50 / 48 / 51 / 59; 16 384 x 2 048 (1 280 tiles) 203 / 202 / 216.
TK_API int tk_gemm_f32_cuts(int M, int N, int K) {
  int split_cuts;
  if (gf_pieces_tile(M, N, K, &split_cuts)) return split_cuts;
  if (M <= 16 || !gf_cuts_add(M, N)) return 1;
  long cuts = 1280 / gf_tiles(M, N, M <= 32 ? 1 : 2, 2);
  const long most = K / 256;
  if (cuts > most || M <= 32) cuts = most;  // (few tokens: chains of 32 elements in every part)
  if (cuts > 32) cuts = 32;
  return cuts < 1 ? 1 : (int)cuts;
}

template <int TM, int TN, int CHAINS>
static bool gf_launch(const GemmF32Args& a, int cuts, hipStream_t stream) {
  const long grid = gf_tiles(a.M, a.N, TM, TN);
  if (grid > 0x7fffffffL) return false;
  // steps in local memory: 2 of the largest tile, so that two workgroups share a compute unit (3: 1,117 us for 2,048 tokens and 16,384 x 2,048
  // as before, 2: 1,018), else 3 (2: 301 tokens 189 / 177, 102 / 97 us)
  constexpr int STAGES = TM * TN == 16 ? 2 : 3;
  const bool stream_in = a.K % 32 == 0;
  const size_t lds = stream_in ? (size_t)STAGES * 32 * (TM + TN) * 32 * sizeof(float) : (size_t)2 * 32 * (TM + TN) * GS_ROW * sizeof(float);
  auto kernel = stream_in ? gemm_f32_stream_kernel<TM, TN, CHAINS, STAGES> : gemm_f32_kernel<TM, TN, CHAINS>;
  if (lds > 64 * 1024 && hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) return false;
  hipLaunchKernelGGL(kernel, dim3((unsigned)grid, cuts), dim3(256), lds, stream, a);
  return true;
}

template <int TM>
static bool gf_launch_pieces(const GemmF32Args& a, int cuts, hipStream_t stream) {
  const long grid = gf_tiles(a.M, a.N, TM, 4);
  if (grid > 0x7fffffffL) return false;
  const size_t lds = (size_t)GP_STAGES * 32 * (TM + 4) * 32 * sizeof(float);  // (64 KB at most)
  hipLaunchKernelGGL((gemm_f32_pieces_kernel<TM, 4>), dim3((unsigned)grid, cuts), dim3(256), lds, stream, a);
  return true;
}

template <int EPI>
static void gf_launch_few(const GemmF32Args& a, const FewExtra& x, hipStream_t stream) {
  // (2, 4, 8 wavefronts at 4 tokens, 2 048 x 2 048: 9.0, 8.2, 9.0 us, 2 048 x 8 192: 34, 25, 26, 16 384 x 2 048: 33, 30, 30)
  const int KS = a.K < 64 ? 1 : (a.K < 4096 ? 4 : 8);
  const size_t lds = (KS - 1) * 64 * sizeof(f4);
  if constexpr (EPI == FEW_STORE) {
    // rows of 8 where rows of 16 leave compute units without a workgroup
    if (a.M <= 8 && a.K % 32 == 0 && a.K >= 256 && a.N <= GF_HALVES_ROWS) {
      const int blocks = a.K / 32;
      hipLaunchKernelGGL((gemm_f32_few_kernel<true, FEW_STORE>), dim3((a.N + 7) / 8), dim3(64 * KS), lds, stream, a, x, KS, blocks / KS, blocks % KS);
      return;
    }
  }
  const int blocks = (a.K + 15) / 16;
  // (pairs of rows: 8 a workgroup, of a head or of gate and up)
  const int groups = EPI == FEW_STORE ? (a.N + 15) / 16 : (EPI == FEW_GLU ? (a.N / 2 + 7) / 8 : a.N / 16);
  hipLaunchKernelGGL((gemm_f32_few_kernel<false, EPI>), dim3(groups), dim3(64 * KS), lds, stream, a, x, KS, blocks / KS, blocks % KS);
}

TK_API int tk_gemm_f32(const void* A, int lda, const void* W, void* C, int ldc, const void* residual, int ldr,
                       const void* bias, int M, int N, int K, int cuts, void* part, hipStream_t stream) {
  TK_REQUIRE(M >= 0 && N > 0 && K > 0 && lda >= K && ldc >= N, "gemm_f32: bad sizes M=%d N=%d K=%d lda=%d ldc=%d", M, N, K, lda, ldc);
  TK_REQUIRE(!residual || ldr >= N, "gemm_f32: residual stride %d < N %d", ldr, N);
  TK_REQUIRE(tk_gemm_f32_takes(A, lda, W, K), "gemm_f32: rows of A and W must start at multiples of 16 bytes");
  TK_REQUIRE(cuts >= 1 && cuts <= (K + 31) / 32 && cuts < 65536 && (cuts == 1 || (part && gf_cuts_add(M, N) && M > 16)),
             "gemm_f32: K=%d in %d parts", K, cuts);
  if (M == 0) return 0;
  GemmF32Args a = {(const float*)A, lda, (const float*)W, (float*)C, ldc, (const float*)residual, ldr, (const float*)bias, M, N, K,
                   cuts > 1 ? (float*)part : nullptr};
  if (M <= 16) {
    gf_launch_few<FEW_STORE>(a, FewExtra{}, stream);
    TK_CHECK_LAUNCH("gemm_f32");
    return 0;
  }
  // tiles of 128 x 128 read the operands half as often, where they still fill the chip twice over; up to 32 tokens leave half
  // of a 64-token tile empty
  bool ok;
  int unused;
  const int pieces = gf_pieces_tile(M, N, K, &unused);
  if (pieces == 64) ok = gf_launch_pieces<2>(a, cuts, stream);
  else if (pieces) ok = gf_launch_pieces<4>(a, cuts, stream);
  else if (M <= 32) ok = gf_launch<1, 2, 8>(a, cuts, stream);
  else if (gf_tiles(M, N, 4, 4) >= 512) ok = gf_launch<4, 4, 1>(a, cuts, stream);
  else ok = gf_launch<2, 2, 1>(a, cuts, stream);
  TK_REQUIRE(ok, "gemm_f32: M=%d N=%d take too many workgroups, or their local memory could not be reserved", M, N);
  if (cuts > 1) hipLaunchKernelGGL(gemm_f32_sum_kernel, dim3((N / 4 + 255) / 256, M), dim3(256), 0, stream, a, cuts);
  TK_CHECK_LAUNCH("gemm_f32");
  return 0;
}

// Few rows (up to 16) with what stands behind the product.  glu: W is [gate | up] and C takes silu(gate) * up, [M, N / 2].  Else W is
// [q | k | v] by heads of d elements, C takes the turned queries [M, nq * d], keys and values go to the pages; cos and sin may be
// null: no rotation.
TK_API int tk_gemm_f32_few(const void* A, int lda, const void* W, void* C, int ldc, const void* bias, int M, int N, int K, int glu,
                           const int* positions, const int* token_req, const int* block_table, int table_stride, const float* cos,
                           const float* sin, float* kcache, float* vcache, int nq, int nkv, int d, int P, hipStream_t stream) {
  TK_REQUIRE(M > 0 && M <= 16 && N > 0 && K > 0 && lda >= K, "gemm_f32_few: bad sizes M=%d N=%d K=%d lda=%d", M, N, K, lda);
  TK_REQUIRE(tk_gemm_f32_takes(A, lda, W, K), "gemm_f32_few: rows of A and W must start at multiples of 16 bytes");
  TK_REQUIRE(!glu || (N % 2 == 0 && ldc >= N / 2), "gemm_f32_few: gate and up of %d rows, result rows of %d", N, ldc);
  TK_REQUIRE(glu || (positions && token_req && block_table && kcache && vcache && nq > 0 && nkv > 0 && d > 0 && d % 16 == 0 && P > 0 &&
                     N == (nq + 2 * nkv) * d && ldc >= nq * d && ldc % 4 == 0 && !cos == !sin &&
                     (((uintptr_t)C | (uintptr_t)cos | (uintptr_t)sin | (uintptr_t)kcache) & 15) == 0),
             "gemm_f32_few: rotation and append of %d + 2 x %d heads of %d from %d outputs", nq, nkv, d, N);
  const GemmF32Args a = {(const float*)A, lda, (const float*)W, (float*)C, ldc, nullptr, 0, (const float*)bias, M, N, K, nullptr};
  const FewExtra x = {positions, token_req, block_table, table_stride, cos, sin, kcache, vcache, nq, nkv, d, P};
  if (glu) gf_launch_few<FEW_GLU>(a, x, stream);
  else gf_launch_few<FEW_ROPE>(a, x, stream);
  TK_CHECK_LAUNCH("gemm_f32_few");
  return 0;
}
