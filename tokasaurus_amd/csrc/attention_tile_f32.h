// Paged attention in 32-bit arithmetic on the matrix cores (v_mfma_f32_16x16x4_f32): scores,
// softmax weights and the weighted values are 32-bit numbers and 32-bit sums, whatever the
// storage type of queries, keys and values (from bfloat16 storage some of the products run on the bfloat16 matrix cores,
// exactly: ScoresFromStorage, at_pieces).  For the 32-bit path, and for mixers that ask for exactly that: a sliding
// window, key and value heads of different sizes, a scale of the model's choosing and a
// learned sink per query head in the softmax's denominator; or, with `score_bias` (one number a
// query head), no softmax at all: a visible key's weight is sigmoid(score + score_bias[head]), not
// normalised over the keys (the sums of wavefronts and chunks are then added as they are).  With `section` > 0 positions are
// cut into sections at multiples of it, counted from a request's start, and a query sees only keys of its own section.
//
// A wavefront owns a tile of 16 "columns": tt = 16 / gg neighbouring tokens of one request
// times gg neighbouring query heads of one kv head (gg = 1 for prompt portions; up to 16 for
// single decoded tokens, so that the heads that share keys share their loads).  It walks the
// keys in steps of 16, at absolute multiples of 16, from the first step that its earliest
// column sees to the last that its latest column sees:
//   S^T = K Q^T       keys as the first operand: a lane then holds, for its column (lane % 16),
//                     the scores of keys 4 * (lane / 16) + i, i < 4
//   O^T += V^T P^T    which is exactly its second operand here (the order of the sum over the
//                     16 keys is a free choice: slot lane / 16 of product i is key 4 * (lane / 16) + i)
// The sum over a head's elements is permuted the same way: a lane loads whole 8-element pieces
// of its key (the page layout's unit) and of its query, piece lane / 16 + 4 m.
//   K pages: [page][kv head][dk / 8][P][8]    V pages: [page][kv head][P / 4][dv][4]
// With bfloat16 storage and a tile a wavefront (prompts) a step is 32 keys and the weighted values go through the bfloat16
// matrix cores in three exact pieces (at_pieces), and references move seldom (AT_SLACK).  Bound by the softmax's vector instructions: some
// 250 a step, of which references that move with every maximum took 45, exp2f with its care for results below 2^-126 40, and tanhf
// 200.  us, with these / now, 32 heads of 64 over 8 kv heads: 2,048 tokens 93.0 / 75.4, with a window of 1,024 and a soft cap 93.1 / 73.1, 8,192
// 964 / 841, 562 and 938 with a window and sinks 63.5 / 49.4, 300 with a cap 29.0 / 19.9; 32 heads of 128, 2,048 tokens 153 / 122, with a cap 195 / 132; 16 of
// 80, 4 x 1,024 105 / 80; of 256, one block a step, with a cap 559 / 511.  Results that differ from the rounded 64-bit ones: 2.84e-4 / 2.74e-4
// at 2,048 tokens of 64, with the cap 2.99e-4 / 2.94e-4, keys eight times as large 3.49e-4 / 3.46e-4.
// Needs dk % 8 == 0, dv % 16 == 0, P % 16 == 0 (a step of 16 keys lies inside one page).
#pragma once

#include "common.h"

typedef float v4f __attribute__((ext_vector_type(4)));
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;

// Scores from bfloat16 storage: the product of two bfloat16 numbers is exact in 32-bit, so the matrix cores'
// bfloat16 product with 32-bit sums (v_mfma_f32_16x16x32_bf16) gives 32-bit scores of the stored queries and keys
// like the 32-bit product of the converted operands, at an eighth of the instructions and without the conversions.
// Its operands are what a lane holds anyway: 8 neighbouring elements of key lane % 16 (of the column's query) from
// element 8 * (lane / 16) of every 32 on.  The weights are 32-bit numbers: weighted values are 32-bit products, or where a step
// is two blocks of keys (at_halves) products of the weights' three exact pieces.
template <typename T>
struct ScoresFromStorage { static constexpr bool value = false; };
template <>
struct ScoresFromStorage<bf16_t> { static constexpr bool value = true; };
template <typename R>
__device__ __forceinline__ bf16x8_t as_bf16x8(const R& raw) {
  bf16x8_t v;
  __builtin_memcpy(&v, &raw, sizeof(v));
  return v;
}

#define AT_WAVES 4
#define AT_MAX_KM 8   // dk <= 256
#define AT_MAX_VT 16  // dv <= 256

// 8 (4) neighbouring elements of the storage type, moved as one: what a lane loads of a key (of the values)
template <typename T>
struct __align__(16) Raw8 { T v[8]; };
template <typename T>
struct __align__(sizeof(T) * 4) Raw4 { T v[4]; };

// What may follow the weighted sum of the values before it is stored, for mixers whose values were turned by their own
// positions and whose heads have a gate: pair m of a head's result is turned back by -position * vfreq[m] (pairs
// (m, m + dv/2) with `pair_half`, which the launch takes only where dv is 16 times the kernel's VT, and (2m, 2m + 1)
// without), then the head is multiplied by sigmoid(gate[token][head]).  Null pointers: nothing of the kind.
template <typename T>
struct AfterSum {
  const float* vfreq;
  int pair_half;
  const T* gate;
  int gate_stride;
};
__device__ __forceinline__ void turn_back(float& u, float& v, float pos, float freq) {
  float sn, cs;
  sincosf(__fmul_rn(pos, freq), &sn, &cs);
  rotate_pair(u, v, cs, -sn, u, v);
}
template <typename T>
__device__ __forceinline__ float gate_of(const AfterSum<T>& after, int tok, int head) {
  return after.gate ? 1.0f / (1.0f + expf(-to_f32<T>(after.gate[(size_t)tok * after.gate_stride + head]))) : 1.f;
}

// What may happen to a score between the scaling and the softmax, for mixers that ask for it: a soft cap
// (score <- cap * tanh(score / cap), cap > 0) and then a learned bias by distance, rel[bucket][head] with
// bucket = bucket_of[min(query position - key position, far)] (a table that the host made).
struct ScoreShape {
  float softcap;
  const int* bucket_of;
  int far;
  const float* rel;
};
// `in_caps`: scale / softcap, so that the product of the stored numbers is rounded once on its way to the tanh (a
// product and a division a score before, of which the division is ten instructions).
// tanh of all of a lane's scores together: up to AT_TANH_NEAR, which scores below five eighths of the cap are, x + x^3 q(x^2) with q of the least
// greatest error in (tanh(x) / x - 1) / x^2, 1.5e-10 of the result in front of the roundings, in 9 instructions where tanhf takes some 30 and
// branches; tanhf of a greater one, which a wavefront that has none of them does not compute.  Relative errors from 64 bits, root mean square
// (largest), tanhf / this: up to an eighth 2.46e-8 (6.14e-8) / 2.44e-8 (5.97e-8), to a quarter 2.47e-8 (6.44e-8) / 2.45e-8 (6.02e-8), to a half 2.53e-8
// (6.43e-8) / 2.51e-8 (6.31e-8), to the end 2.84e-8 (7.46e-8) / 2.82e-8 (7.16e-8).
#define AT_TANH_NEAR 0.625f
__device__ __forceinline__ float near_tanh(float x) {
  const float z = x * x;
  float q = 0.002147537f;
  q = fmaf(q, z, -0.008182674f);
  q = fmaf(q, z, 0.021702968f);
  q = fmaf(q, z, -0.053947203f);
  q = fmaf(q, z, 0.1333321f);
  q = fmaf(q, z, -0.3333333f);
  return fmaf(x * z, q, x);
}
template <int N>
__device__ __forceinline__ void capped_scores(float (&sc)[N], float softcap) {
  float most = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i) most = fmaxf(most, fabsf(sc[i]));
  if (__any(most > AT_TANH_NEAR)) {
    // (every score by its own size: the greatest may be of another row, or of a key that no row sees, whose page holds anything)
#pragma unroll
    for (int i = 0; i < N; ++i) {
      sc[i] = softcap * (fabsf(sc[i]) > AT_TANH_NEAR ? tanhf(sc[i]) : near_tanh(sc[i]));
      asm volatile("" : "+v"(sc[i]));  // (one after the other: side by side they take registers from the walk)
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < N; ++i) sc[i] = softcap * near_tanh(sc[i]);
}

// Blocks of 16 keys that a wavefront takes a step: two where the weighted values go through the bfloat16 matrix cores
// (at_pieces) and the registers hold two blocks' keys and values twice.
template <typename T, int KM, int VT, bool SPLIT>
__device__ constexpr int at_halves() { return ScoresFromStorage<T>::value && !SPLIT && KM <= 4 && VT <= 8 ? 2 : 1; }

// A 32-bit weight as the sum of three bfloat16 numbers, exactly (its 24 bits, 8 at a time): a bfloat16 value times each
// is exact in 32-bit, so three products of v_mfma_f32_16x16x32_bf16 add what eight of v_mfma_f32_16x16x4_f32 add, in a
// quarter of their time.  piece[n] holds what a lane's operand needs: the pieces of its 8 keys' weights.
// An infinite value would meet pieces that are zero (NaN where the 32-bit product is infinite): a wavefront that ends
// with a sum that is not finite walks its keys again with 32-bit products.
__device__ __forceinline__ void at_pieces(const float (&p)[8], bf16x8_t (&piece)[3]) {
  uint32_t packed[3][4];
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    float a = p[i], b = p[i + 1];
#pragma unroll
    for (int n = 0; n < 3; ++n) {
      const uint32_t ua = __float_as_uint(a), ub = __float_as_uint(b);
      packed[n][i / 2] = __builtin_amdgcn_perm(ub, ua, 0x07060302);  // the upper halves, a's below
      a -= __uint_as_float(ua & 0xffff0000u);
      b -= __uint_as_float(ub & 0xffff0000u);
    }
  }
#pragma unroll
  for (int n = 0; n < 3; ++n) __builtin_memcpy(&piece[n], packed[n], sizeof(piece[n]));
}

// What a score may be above its column's reference, and the reference as the exponents take it (0 while no key was seen).
#define AT_LOG2E 1.44269504088896341f
#define AT_SLACK 5.5f
__device__ __forceinline__ float at_reference(float m) {
  float r = m == -INFINITY ? 0.f : m * AT_LOG2E;
  asm("" : "+v"(r));  // (rounded wherever it is used: in a difference the compiler would leave the rounding out, 2e-6 of a weight at scores of 30)
  return r;
}

// The result of matrix products moved to ordinary registers at this place, in front of any branch.  The compiler waits for a
// product that is read in its own stretch of code; a read of an accumulation register behind a branch it has placed one to
// three instructions behind the product, which then was lost (with a branch around the products of a value head's last block,
// heads of 112 and 240 missed one key in four of their last but one).
__device__ __forceinline__ void at_settle(v4f& x) { asm volatile("" : "+v"(x)); }

// Which (tile, block of heads) a workgroup takes.  Causal tiles late in a prompt see many keys, early ones few, and
// workgroups land on the compute units in turn: with tiles in launch order a unit gets the same place of the prompt
// again and again (2,048 tokens and 8 blocks of heads: every 256th workgroup is the same tile).
// So the late tiles go first, and every other round of 256 workgroups runs the other way; blocks of heads vary fastest, so that those of one number meet in one
// chiplet's cache (workgroups go round the 8 chiplets) where their count is 8.
__device__ __forceinline__ void at_place(int& tile, int& hy) {
  const int nx = gridDim.x, ny = gridDim.y, all = nx * ny;
  int id = blockIdx.x + nx * blockIdx.y;
  const int base = id & ~255;
  if ((base & 256) && base + 256 <= all) id = base + ((31 - ((id & 255) >> 3)) << 3) + (id & 7);
  tile = nx - 1 - id / ny;
  hy = id % ny;
}

// SPLIT: the NW wavefronts of a workgroup share one tile and take its key steps in turn
// (wavefront w the steps w, w + NW, ..); they add up through LDS, always in wavefront order.
// For steps of few tiles (single decoded tokens), whose walks would else be one long chain each.
//
// PART (with SPLIT): the keys are also cut into chunks of `chunk` keys at absolute multiples of it, a workgroup a
// (tile, head block, chunk): blockIdx.z names the chunk.  A workgroup leaves its maxima, sums and weighted values
// unnormalised in `part`; attention_tile_merge_kernel adds the chunks in ascending order.  For single decoded
// tokens after long contexts, where a tile's walk would else keep one workgroup busy and the chip idle.
//
// (Four wavefronts a SIMD for heads up to 64 elements, two up to 128: one hides the loads and the exponentials of another.)
template <typename T, int KM, int VT, bool SPLIT, int NW, bool PART = false>
__global__ __launch_bounds__(NW * TK_WAVE, SPLIT ? 1 : (KM <= 2 && VT <= 4 ? 4 : (KM <= 4 && VT <= 8 ? 2 : 1))) void attention_tile_f32_kernel(
    const T* __restrict__ q, int q_stride, T* __restrict__ out, int out_stride, const T* __restrict__ kcache,
    const T* __restrict__ vcache, const int* __restrict__ block_table, int table_stride,
    const int* __restrict__ q_start, const int* __restrict__ kv_len, const int* __restrict__ tile_req,
    const int* __restrict__ tile_row0, int nq, int nkv, int dk, int dv, int P, int window, int section, float scale,
    const float* __restrict__ sink, const float* __restrict__ score_bias, int gg, AfterSum<T> after, ScoreShape shape,
    int chunk = 0, float* __restrict__ part = nullptr) {
  extern __shared__ float merge[];  // SPLIT: [waves][16] maxima, [waves][16] sums, [waves - 1][VT][4][64] weighted values
  const int lane = threadIdx.x & (TK_WAVE - 1), wave = threadIdx.x / TK_WAVE;
  const int group = nq / nkv;
  const int blocks_per_kv = group / gg;  // head blocks of gg heads
  int tile = blockIdx.x, hy = blockIdx.y;
  if constexpr (!SPLIT) at_place(tile, hy);
  const int hb = SPLIT ? hy : hy * NW + wave;
  if (hb >= nkv * blocks_per_kv) return;
  const int kvh = hb / blocks_per_kv;
  const int head0 = kvh * group + (hb % blocks_per_kv) * gg;
  const int r = tile_req[tile];
  const int row0 = tile_row0[tile];
  const int tt = 16 / gg;
  const int col = lane & 15, c = lane >> 4;
  // this lane's column: a token and a query head
  const int tok = row0 + col / gg;
  const int head = head0 + col % gg;
  const int q_end = q_start[r + 1];
  const int kv = kv_len[r];
  const bool live = tok < q_end;
  const int n_tok = min(tt, q_end - row0);
  const int pos0 = kv - (q_end - row0);         // position of the tile's first token
  const int pos = pos0 + col / gg;              // of this column's token
  const int last_all = pos0 + n_tok - 1;  // the last key any column of the tile sees
  // (PART) this workgroup's chunk: with a window or sections the launch holds only as many chunks as those touch, and
  // blockIdx.z counts from the chunk of the first key that the tile sees (absolute multiples of `chunk` all the same)
  const int first_seen = section > 0 ? pos0 / section * section : (window > 0 ? max(0, pos0 - window + 1) : 0);
  const int lo_col = section > 0 ? pos / section * section : 0;            // the first key of this column's section
  const int lo_last = section > 0 ? last_all / section * section : 0;      // of the last column's
  const int zc = PART ? first_seen / chunk + (int)blockIdx.z : 0;
  const int last = PART ? min(last_all, (zc + 1) * chunk - 1) : last_all;  // the last this workgroup walks
  const int lo_tile = max(first_seen, PART ? zc * chunk : 0);
  const int* table = block_table + (size_t)r * table_stride;
  const int pieces = dk / 8;
  const size_t key_page = key_page_elems(P, dk);

  // the column's query, piece c + 4 m (as stored, for scores from storage; else as 32-bit numbers)
  constexpr bool STORED = ScoresFromStorage<T>::value;
  float qv[STORED ? 1 : KM][8];
  Raw8<T> qraw[STORED ? KM : 1];
#pragma unroll
  for (int m = 0; m < KM; ++m) {
    const int piece = c + 4 * m;
    const bool in = live && piece < pieces;
    const T* src = q + (size_t)(in ? tok : 0) * q_stride + (size_t)head * dk + (in ? piece : 0) * 8;
    if constexpr (STORED) {
#pragma unroll
      for (int e = 0; e < 8; ++e) qraw[m].v[e] = in ? src[e] : from_f32<T>(0.f);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) qv[m][e] = in ? to_f32<T>(src[e]) : 0.f;
    }
  }

  v4f o[VT];
  const bool sig = score_bias != nullptr;
  const float in_caps = shape.softcap > 0.f ? scale / shape.softcap : 0.f;
  const float pb = sig && live ? score_bias[head] : 0.f;
  // (sigmoid weights have no maximum to follow: it stays 0, so every merge below multiplies by exp(0))
  float m_run, l_run;  // l_run: this lane's share of the column's sum

  // where this lane's pieces of a key and its values lie inside a page, for the page's first key: both offsets
  // grow linearly with the key's place in the page (8 elements a key, dv a key)
  int koff[KM], voff[VT];
#pragma unroll
  for (int m = 0; m < KM; ++m) koff[m] = (int)key_offset(P, col, (c + 4 * m < pieces ? c + 4 * m : 0) * 8);
#pragma unroll
  for (int t = 0; t < VT; ++t) voff[t] = (int)value_offset(dv, 4 * c, 16 * t < dv ? 16 * t + col : 0);
  constexpr int H = at_halves<T, KM, VT, SPLIT>();  // blocks of 16 keys a step
  // a step that every column of the tile sees whole needs no masks (the same for all lanes)
  auto seen_whole = [&](int k0) {
    return k0 + 16 * H - 1 <= pos0 && (window <= 0 || last_all - k0 < window) && k0 >= lo_last && n_tok * gg == 16;
  };
  auto sees = [&](int kp) { return live && kp <= pos && kp >= lo_col && (window <= 0 || pos - kp < window); };
  bool odd = false;  // the wavefront has met a value that is not finite in a step with masks
  const int step = SPLIT ? 16 * NW : 16 * H;
  const int k_first = (lo_tile / (16 * H)) * (16 * H) + (SPLIT ? 16 * wave : 0);
  // The pages of this wavefront's blocks of keys, 64 blocks at a time: lane j asks for the page of block `base + j`, and
  // a step reads its pages' numbers from those lanes.  So no load of keys or values waits for a load of a page number.
  int pv = 0;
#define AT_PAGES(BASE)                                                  \
  do {                                                                  \
    const int kj = k_first + ((BASE) + lane) * (step / H);              \
    pv = kj <= last ? max(table[kj / P], 0) : 0;                        \
  } while (0)
  // `wide`: the weighted values as 32-bit products (see at_pieces)
  auto walk = [&](auto wide) {
#pragma unroll
  for (int t = 0; t < VT; ++t) o[t] = (v4f){0.f, 0.f, 0.f, 0.f};
  m_run = sig ? 0.f : -INFINITY;
  l_run = 0.f;
  int k0 = k_first;
  AT_PAGES(0);
  // this lane's pieces of key k0 + 16 h + col and its values (element 16 t + col of keys k0 + 16 h + 4 c + i); the keys
  // are asked for a step ahead, and (SPLIT, where nothing else hides the wait) the values too
  Raw8<T> kr[H][KM];
  Raw4<T> vr[H][VT];
  auto load_keys = [&](Raw8<T>(&dst)[H][KM], int at, int block) {
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const int page = __builtin_amdgcn_readlane(pv, (block + h) & 63);
      const T* kbase = kcache + ((size_t)page * nkv + kvh) * key_page + ((at + 16 * h) % P) * 8;
#pragma unroll
      for (int m = 0; m < KM; ++m) dst[h][m] = *(const Raw8<T>*)(kbase + koff[m]);
    }
  };
  auto load_values = [&](Raw4<T>(&dst)[H][VT], int at, int block) {
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const int page = __builtin_amdgcn_readlane(pv, (block + h) & 63);
      const T* vbase = vcache + ((size_t)page * nkv + kvh) * P * dv + ((at + 16 * h) % P) * dv;
#pragma unroll
      for (int t = 0; t < VT; ++t) dst[h][t] = *(const Raw4<T>*)(vbase + voff[t]);
    }
  };
  if (k0 <= last) {
    load_keys(kr, k0, 0);
    if constexpr (SPLIT) load_values(vr, k0, 0);
  }
  int j = 0;
#pragma unroll 1
  for (; k0 <= last; k0 += step, j += H) {
    if constexpr (!SPLIT) load_values(vr, k0, j);
    Raw8<T> kn[H][KM];
    Raw4<T> vn[H][VT];
    const int k1 = k0 + step;
    if (k1 <= last) {
      if (((j + H) & 63) == 0) AT_PAGES(j + H);
      load_keys(kn, k1, j + H);
      if constexpr (SPLIT) load_values(vn, k1, j + H);
    }
    // S^T = K Q^T (a piece beyond the head's size meets zeros of the query)
    v4f s[H];
#pragma unroll
    for (int h = 0; h < H; ++h) {
      s[h] = (v4f){0.f, 0.f, 0.f, 0.f};
      if constexpr (STORED) {
#pragma unroll
        for (int m = 0; m < KM; ++m)
          s[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(kr[h][m]), as_bf16x8(qraw[m]), s[h], 0, 0, 0);
      } else {
#pragma unroll
        for (int m = 0; m < KM; ++m)
#pragma unroll
          for (int e = 0; e < 8; ++e)
            s[h] = __builtin_amdgcn_mfma_f32_16x16x4f32(to_f32<T>(kr[h][m].v[e]), qv[m][e], s[h], 0, 0, 0);
      }
    }
#pragma unroll
    for (int h = 0; h < H; ++h) at_settle(s[h]);
    // this lane now holds, for its column, keys k0 + 16 h + 4 c + i: number 4 h + i below
    float sc[4 * H];
#pragma unroll
    for (int i = 0; i < 4 * H; ++i) sc[i] = s[i / 4][i % 4] * (shape.softcap > 0.f ? in_caps : scale);
    if (shape.softcap > 0.f) capped_scores(sc, shape.softcap);
    if (shape.rel) {
#pragma unroll
      for (int i = 0; i < 4 * H; ++i) {
        const int dist = pos - (k0 + 16 * (i / 4) + 4 * c + i % 4);
        sc[i] += shape.rel[(size_t)shape.bucket_of[min(max(dist, 0), shape.far)] * nq + head];
      }
    }
    float tmax = -INFINITY;
    if (seen_whole(k0)) {
#pragma unroll
      for (int i = 0; i < 4 * H; ++i) tmax = fmaxf(tmax, sc[i]);
    } else {
#pragma unroll
      for (int i = 0; i < 4 * H; ++i) {
        const int kp = k0 + 16 * (i / 4) + 4 * c + i % 4;
        sc[i] = sees(kp) ? sc[i] : -INFINITY;
        tmax = fmaxf(tmax, sc[i]);
        // a key that no column sees may be anything (a page's places behind the request's last token, a page given back):
        // its weight is zero, and so must its values be, or a NaN there would reach the sums
        if (kp > last_all || kp < first_seen) {
#pragma unroll
          for (int t = 0; t < VT; ++t) vr[i / 4][t].v[i % 4] = from_f32<T>(0.f);
        }
      }
      // the same for a value that is not finite where some columns see its key and others do not; those that do get it below
      // (the heads of one token see the same keys)
      if (decltype(wide)::value && n_tok > 1) {
        float zero = 0.f;  // or NaN
#pragma unroll
        for (int t = 0; t < VT; ++t)
#pragma unroll
          for (int i = 0; i < 4 * H; ++i) zero = fmaf(to_f32<T>(vr[i / 4][t].v[i % 4]), 0.f, zero);
        if (__builtin_expect(__any(zero != 0.f), 0)) {
          odd = true;
#pragma unroll
          for (int t = 0; t < VT; ++t)
#pragma unroll
            for (int i = 0; i < 4 * H; ++i) {
              T& v = vr[i / 4][t].v[i % 4];
              v = fabsf(to_f32<T>(v)) < INFINITY ? v : from_f32<T>(0.f);
            }
        }
      }
    }
    float p[4 * H];
    float alpha = 1.f;
    if (sig) {
      // 1 / (1 + exp(-(score + bias))); a masked score gives 1 / (1 + inf) = 0
#pragma unroll
      for (int i = 0; i < 4 * H; ++i) p[i] = 1.0f / (1.0f + exp2f(-(sc[i] + pb) * 1.44269504088896341f));
    } else if constexpr (!decltype(wide)::value) {
      // Any reference near the greatest score will do, so it moves only when a score is AT_SLACK above it (terms up to 256, whose roundings are
      // relative as ever), and the four lanes of a column need to agree on nothing in between.  exp2 of (score - reference) log2(e), the reference's
      // product rounded alike for all of a column: the hardware's own exponential (a masked score gives exp2(-inf) = 0)
      if (__any(tmax > m_run + AT_SLACK)) {
        tmax = fmaxf(tmax, __shfl_xor(tmax, 16, TK_WAVE));
        tmax = fmaxf(tmax, __shfl_xor(tmax, 32, TK_WAVE));
        const float m_new = tmax > m_run + AT_SLACK ? tmax : m_run;
        const float back = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(at_reference(m_run) - at_reference(m_new));
        l_run *= back;
#pragma unroll
        for (int t = 0; t < VT; ++t) o[t] = o[t] * back;
        m_run = m_new;
      }
      const float reference = at_reference(m_run);
#pragma unroll
      for (int i = 0; i < 4 * H; ++i) p[i] = __builtin_amdgcn_exp2f(fmaf(sc[i], AT_LOG2E, -reference));
      l_run += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
    } else {
      tmax = fmaxf(tmax, __shfl_xor(tmax, 16, TK_WAVE));
      tmax = fmaxf(tmax, __shfl_xor(tmax, 32, TK_WAVE));
      const float m_new = fmaxf(m_run, tmax);
      if (m_new == -INFINITY) {
#pragma unroll
        for (int i = 0; i < 4 * H; ++i) p[i] = sc[i] == -INFINITY ? 0.f : sc[i];  // (no key seen, or scores that are all NaN)
      } else {
        // exp2 of the difference times log2(e): the hardware's own exponential (a masked score gives exp2(-inf) = 0)
        alpha = exp2f((m_run - m_new) * 1.44269504088896341f);
#pragma unroll
        for (int i = 0; i < 4 * H; ++i) p[i] = exp2f((sc[i] - m_new) * 1.44269504088896341f);
      }
      m_run = m_new;
      l_run = l_run * alpha + ((p[0] + p[1]) + (p[2] + p[3]));
      if constexpr (H == 2) l_run += (p[4] + p[5]) + (p[6] + p[7]);
    }
    // O^T += V^T P^T
    // (for all VT blocks, also those behind dv, whose lanes hold some of the head's first values and are never stored)
    if constexpr (decltype(wide)::value) {
#pragma unroll
      for (int t = 0; t < VT; ++t) o[t] = o[t] * alpha;
    }
    if constexpr (decltype(wide)::value) {
#pragma unroll
      for (int t = 0; t < VT; ++t)
#pragma unroll
        for (int i = 0; i < 4 * H; ++i)
          o[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(to_f32<T>(vr[i / 4][t].v[i % 4]), p[i], o[t], 0, 0, 0);
    } else if constexpr (H == 2) {
      bf16x8_t piece[3];
      at_pieces(p, piece);
#pragma unroll
      for (int n = 2; n >= 0; --n)
#pragma unroll
        for (int t = 0; t < VT; ++t) {
          Raw8<T> v8;
          __builtin_memcpy(&v8.v[0], &vr[0][t], sizeof(vr[0][t]));
          __builtin_memcpy(&v8.v[4], &vr[1][t], sizeof(vr[1][t]));
          o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(v8), piece[n], o[t], 0, 0, 0);
        }
    }
#pragma unroll
    for (int t = 0; t < VT; ++t) at_settle(o[t]);
#pragma unroll
    for (int h = 0; h < H; ++h) {
#pragma unroll
      for (int m = 0; m < KM; ++m) kr[h][m] = kn[h][m];
      if constexpr (SPLIT) {
#pragma unroll
        for (int t = 0; t < VT; ++t) vr[h][t] = vn[h][t];
      }
    }
  }
  };
  walk(std::integral_constant<bool, H == 1>{});
  bool late = H == 2;  // whether the terms' reference is at_reference's, which may be behind the greatest score
  if constexpr (H == 2) {
    // again, with the greatest score as reference and 32-bit products, where that cannot be: an infinite value, values whose sum is finite only with
    // weights of one and less, a score whose reference is beyond 32 bits
    bool finite = fabsf(at_reference(m_run)) < INFINITY;
#pragma unroll
    for (int t = 0; t < VT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) finite = finite && fabsf(o[t][i]) < INFINITY;
    if (!__all(finite)) {
      walk(std::integral_constant<bool, true>{});
      late = false;
    }
  }
#undef AT_PAGES
  if (__builtin_expect(odd, 0)) {
    // the values left out of the steps with masks, each for the columns that see its key: their sums are not finite
    int places = P, size = dv;
    asm volatile("" : "+s"(places), "+s"(size));  // (nothing of this is made ready in front of the walk, whose registers are full)
#pragma unroll 1
    for (int k0 = k_first; k0 <= last; k0 += step) {
      if (seen_whole(k0)) continue;
#pragma unroll 1
      for (int kp = max(k0, first_seen); kp < k0 + 16 * H && kp <= last; ++kp) {
        const T* vbase = vcache + ((size_t)max(table[kp / places], 0) * nkv + kvh) * places * size;
#pragma unroll
        for (int t = 0; t < VT; ++t)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float v = 16 * t < size ? to_f32<T>(vbase[value_offset(size, kp % places, 16 * t + 4 * c + e)]) : 0.f;
            if (sees(kp) && !(fabsf(v) < INFINITY)) o[t][e] += v;
          }
      }
    }
  }
  // the column's sum, from the four lanes that share it (always in this order)
  float l = l_run;
  l += __shfl_xor(l, 16, TK_WAVE);
  l += __shfl_xor(l, 32, TK_WAVE);
  if constexpr (SPLIT) {
    float* sm = merge;
    float* sl = merge + NW * 16;
    float* so = merge + 2 * NW * 16;
    if (c == 0) {
      sm[wave * 16 + col] = m_run;
      sl[wave * 16 + col] = l;
    }
    // (the first wavefront adds the others' sums to its own, which never leave its registers)
    if (wave > 0) {
#pragma unroll
      for (int t = 0; t < VT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) so[(((wave - 1) * VT + t) * 4 + i) * TK_WAVE + lane] = o[t][i];
    }
    __syncthreads();
    if (wave != 0) return;
    float m_all = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) m_all = fmaxf(m_all, sm[w * 16 + col]);
    l = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float mw = sm[w * 16 + col];
      const float f = (mw == -INFINITY) ? 0.f : expf(mw - m_all);
      l = fmaf(sl[w * 16 + col], f, l);
      if (w == 0) {
#pragma unroll
        for (int t = 0; t < VT; ++t) o[t] = o[t] * f;
      } else {
#pragma unroll
        for (int t = 0; t < VT; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) o[t][i] = fmaf(so[(((w - 1) * VT + t) * 4 + i) * TK_WAVE + lane], f, o[t][i]);
      }
    }
    m_run = m_all;
  }
  if constexpr (PART) {
    // [tile][head block][chunk]: 16 maxima, 16 sums, [VT][4][64] weighted values as the lanes hold them
    const size_t unit = 32 + (size_t)VT * 4 * TK_WAVE;
    float* dst = part + (((size_t)tile * gridDim.y + blockIdx.y) * gridDim.z + blockIdx.z) * unit;
    if (c == 0) {
      dst[col] = m_run;
      dst[16 + col] = l;
    }
#pragma unroll
    for (int t = 0; t < VT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) dst[32 + (t * 4 + i) * TK_WAVE + lane] = o[t][i];
    return;
  }
  float keep = 1.f;
  if (sink && live && !sig) {
    // the sink joins the softmax like one more score: the maximum may rise to it
    const float sk = sink[head], m_all = fmaxf(m_run, sk);
    if (late && m_run > -INFINITY) {  // (from the reference that the terms have)
      const float above = fmaf(sk, AT_LOG2E, -at_reference(m_run));
      keep = above > 0.f ? exp2f(-above) : 1.f;
      l = l * keep + (above > 0.f ? 1.f : exp2f(above));
    } else {
      keep = (m_run == -INFINITY) ? 0.f : expf(m_run - m_all);
      l = l * keep + expf(sk - m_all);
    }
  }
  if (!live) return;
  const float inv = sig ? 1.f : keep / l;
#pragma unroll
  for (int t = 0; t < VT; ++t) o[t] = o[t] * inv;
  if (after.vfreq) {
    const float fp = (float)pos;
    if (after.pair_half) {  // dv == 16 VT: element 16 t + 4 c + i meets the one of block t + VT / 2
#pragma unroll
      for (int t = 0; t < VT / 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float u = o[t][i], v = o[t + VT / 2][i];
          turn_back(u, v, fp, after.vfreq[16 * t + 4 * c + i]);
          o[t][i] = u;
          o[t + VT / 2][i] = v;
        }
    } else {
#pragma unroll
      for (int t = 0; t < VT; ++t)
        if (16 * t < dv) {
#pragma unroll
          for (int i = 0; i < 4; i += 2) {
            float u = o[t][i], v = o[t][i + 1];
            turn_back(u, v, fp, after.vfreq[(16 * t + 4 * c + i) / 2]);
            o[t][i] = u;
            o[t][i + 1] = v;
          }
        }
    }
  }
  const float g = gate_of(after, tok, head);
  T* dst = out + (size_t)tok * out_stride + (size_t)head * dv;
#pragma unroll
  for (int t = 0; t < VT; ++t) {
    if (16 * t < dv) {
#pragma unroll
      for (int i = 0; i < 4; ++i) dst[16 * t + 4 * c + i] = from_f32<T>(o[t][i] * g);
    }
  }
}

// A workgroup a (tile, head block), a wavefront a block of 16 value elements: the chunks' partial results added in
// ascending order, then the sink and the division, with the lanes' places as in the kernel above.
template <typename T, int VT>
__global__ __launch_bounds__(VT * TK_WAVE) void attention_tile_merge_kernel(
    const float* __restrict__ part, int chunks, T* __restrict__ out, int out_stride, const int* __restrict__ q_start,
    const int* __restrict__ tile_req, const int* __restrict__ tile_row0, int nq, int nkv, int dv,
    const float* __restrict__ sink, int gg, int plain_sums, const int* __restrict__ kv_len, AfterSum<T> after) {
  __shared__ float ex[VT * TK_WAVE * 4];  // the wavefronts' results, where the halves of a head are turned back
  const int lane = threadIdx.x & (TK_WAVE - 1), t = threadIdx.x / TK_WAVE;
  if (16 * t >= dv) return;  // (never with halves to turn back: dv is 16 VT then, and every wavefront reaches the barrier)
  const int group = nq / nkv, blocks_per_kv = group / gg;
  const int hb = blockIdx.y, tile = blockIdx.x;
  const int head0 = (hb / blocks_per_kv) * group + (hb % blocks_per_kv) * gg;
  const int col = lane & 15, c = lane >> 4;
  const int tok = tile_row0[tile] + col / gg, head = head0 + col % gg;
  const bool live = tok < q_start[tile_req[tile] + 1];
  const size_t unit = 32 + (size_t)VT * 4 * TK_WAVE;
  const float* src = part + ((size_t)tile * gridDim.y + hb) * chunks * unit;
  float m_all = -INFINITY;
#pragma unroll 8
  for (int z = 0; z < chunks; ++z) m_all = fmaxf(m_all, src[z * unit + col]);
  float l = 0.f;
  v4f o = (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int z = 0; z < chunks; ++z) {
    const float mz = src[z * unit + col];
    const float lz = src[z * unit + 16 + col];
    v4f oz;
#pragma unroll
    for (int i = 0; i < 4; ++i) oz[i] = src[z * unit + 32 + (t * 4 + i) * TK_WAVE + lane];
    // a chunk none of whose keys this column sees (maximum -inf, sums zero) adds nothing
    const float f = (mz == -INFINITY) ? 0.f : expf(mz - m_all);
    l = fmaf(lz, f, l);
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = fmaf(oz[i], f, o[i]);
  }
  float keep = 1.f;
  if (sink && live && !plain_sums) {
    const float sk = sink[head], m2 = fmaxf(m_all, sk);
    keep = (m_all == -INFINITY) ? 0.f : expf(m_all - m2);
    l = l * keep + expf(sk - m2);
  }
  const float inv = !live ? 0.f : (plain_sums ? 1.f : keep / l);  // (sigmoid weights: every chunk's maximum is 0 and its sums count as they are)
  float r[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = live ? o[i] * inv : 0.f;
  if (after.vfreq) {
    const int req = tile_req[tile];
    const float fp = live ? (float)(kv_len[req] - (q_start[req + 1] - tok)) : 0.f;
    if (after.pair_half) {
#pragma unroll
      for (int i = 0; i < 4; ++i) ex[(t * TK_WAVE + lane) * 4 + i] = r[i];
      __syncthreads();
      const bool low = t < VT / 2;
      const int other = low ? t + VT / 2 : t - VT / 2;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float u = low ? r[i] : ex[(other * TK_WAVE + lane) * 4 + i];
        float v = low ? ex[(other * TK_WAVE + lane) * 4 + i] : r[i];
        turn_back(u, v, fp, after.vfreq[16 * (low ? t : other) + 4 * c + i]);
        r[i] = low ? u : v;
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; i += 2) turn_back(r[i], r[i + 1], fp, after.vfreq[(16 * t + 4 * c + i) / 2]);
    }
  }
  if (!live) return;
  const float g = gate_of(after, tok, head);
  T* dst = out + (size_t)tok * out_stride + (size_t)head * dv;
#pragma unroll
  for (int i = 0; i < 4; ++i) dst[16 * t + 4 * c + i] = from_f32<T>(r[i] * g);
}

// Blocks of 16 value elements that the kernel is built for (VT) and a head of dv elements takes: its own number up to 8, so
// that no head in use pays for blocks that it does not have, then 12 or 16.
static int at_value_blocks(int dv) {
  const int vt = dv / 16;
  return vt <= 2 ? 2 : (vt <= 8 ? vt : (vt <= 12 ? 12 : 16));
}

// A launch's arguments, as tk_attention_tile_f32 takes them.
struct AttentionTileCall {
  dim3 grid;
  bool split;
  hipStream_t stream;
  const void* q;
  int q_stride;
  void* out;
  int out_stride;
  const void *kcache, *vcache;
  const int* block_table;
  int table_stride;
  const int *q_start, *kv_len, *tile_req, *tile_row0;
  int nq, nkv, dk, dv, P, window, section;
  float scale;
  const float *sink, *score_bias;
  int gg, chunk;
  float* part;
  const float* vfreq;
  int v_pair_half;
  const void* gate;
  int gate_stride;
  ScoreShape shape;
};

template <typename T, int KM, int VT>
static void at_launch(const AttentionTileCall& a) {
  // halves of a head meet inside a lane only where the head fills the kernel's blocks of 16 (the entry point has checked)
  const AfterSum<T> after = {a.vfreq, a.v_pair_half, (const T*)a.gate, a.gate_stride};
  const AfterSum<T> none = {nullptr, 0, nullptr, 0};
#define AT_COMMON                                                                                                               \
  (const T*)a.q, a.q_stride, (T*)a.out, a.out_stride, (const T*)a.kcache, (const T*)a.vcache, a.block_table, a.table_stride, a.q_start, \
      a.kv_len, a.tile_req, a.tile_row0, a.nq, a.nkv, a.dk, a.dv, a.P, a.window, a.section, a.scale, a.sink, a.score_bias, a.gg
  // split: eight wavefronts a tile where their sums fit the local memory, else four
  constexpr int NW = VT <= 4 ? 8 : 4;
  const size_t smem = sizeof(float) * (NW * 32 + (size_t)(NW - 1) * VT * 4 * TK_WAVE);
  if (a.split && a.chunk > 0) {
    hipLaunchKernelGGL((attention_tile_f32_kernel<T, KM, VT, true, NW, true>), a.grid, dim3(NW * TK_WAVE), smem, a.stream,
                       AT_COMMON, none, a.shape, a.chunk, a.part);
    hipLaunchKernelGGL((attention_tile_merge_kernel<T, VT>), dim3(a.grid.x, a.grid.y), dim3(VT * TK_WAVE), 0, a.stream, a.part,
                       (int)a.grid.z, (T*)a.out, a.out_stride, a.q_start, a.tile_req, a.tile_row0, a.nq, a.nkv, a.dv, a.sink, a.gg,
                       a.score_bias ? 1 : 0, a.kv_len, after);
  } else if (a.split) {
    hipLaunchKernelGGL((attention_tile_f32_kernel<T, KM, VT, true, NW>), a.grid, dim3(NW * TK_WAVE), smem, a.stream, AT_COMMON,
                       after, a.shape);
  } else {
    hipLaunchKernelGGL((attention_tile_f32_kernel<T, KM, VT, false, AT_WAVES>), a.grid, dim3(AT_WAVES * TK_WAVE), 0, a.stream,
                       AT_COMMON, after, a.shape);
  }
#undef AT_COMMON
}

template <typename T, int KM>
static void at_launch_blocks(const AttentionTileCall& a) {
  switch (at_value_blocks(a.dv)) {
    case 2: at_launch<T, KM, 2>(a); break;
    case 3: at_launch<T, KM, 3>(a); break;
    case 4: at_launch<T, KM, 4>(a); break;
    case 5: at_launch<T, KM, 5>(a); break;
    case 6: at_launch<T, KM, 6>(a); break;
    case 7: at_launch<T, KM, 7>(a); break;
    case 8: at_launch<T, KM, 8>(a); break;
    case 12: at_launch<T, KM, 12>(a); break;
    default: at_launch<T, KM, 16>(a); break;
  }
}

template <typename T>
static void at_launch_sizes(const AttentionTileCall& a) {
  const int km = (a.dk + 31) / 32;
  if (km <= 1) at_launch_blocks<T, 1>(a);
  else if (km <= 2) at_launch_blocks<T, 2>(a);
  else if (km <= 4) at_launch_blocks<T, 4>(a);
  else at_launch_blocks<T, 8>(a);
}

// The storage types' kernels, a source each (the many sizes take the compiler its time).
void attention_tile_launch_f32(const AttentionTileCall& a);   // attention_tile_f32.hip
void attention_tile_launch_bf16(const AttentionTileCall& a);  // attention_tile_bf16.hip
