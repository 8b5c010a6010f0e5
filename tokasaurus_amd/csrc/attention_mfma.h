// Device code of the matrix-core attention, shared by the attention kernel and by kernels
// that run attention as one of their phases.  See attention_mfma.hip for the method.
#pragma once

#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

template <bool SHARED>
__device__ __forceinline__ bf16x8_t load_bf16x8(const bf16_t* p) {
  if constexpr (SHARED) {
    union { uint64_t u[2]; bf16x8_t v; } x;
    x.u[0] = shared_load64(p);
    x.u[1] = shared_load64(p + 4);
    return x.v;
  } else {
    return *(const bf16x8_t*)p;
  }
}
template <bool SHARED>
__device__ __forceinline__ void store_f32x4(float* p, f32x4_t v) {
  if constexpr (SHARED) {
    union { uint64_t u[2]; f32x4_t v; } x;
    x.v = v;
    shared_store64(p, x.u[0]);
    shared_store64(p + 2, x.u[1]);
  } else {
    *(f32x4_t*)p = v;
  }
}
template <bool SHARED>
__device__ __forceinline__ void store_f32x2(float* p, float a, float b) {
  if constexpr (SHARED) {
    union { uint64_t u; float f[2]; } x;
    x.f[0] = a;
    x.f[1] = b;
    shared_store64(p, x.u);
  } else {
    p[0] = a;
    p[1] = b;
  }
}

struct AttnArgs {
  const bf16_t* q;
  int q_stride;
  bf16_t* out;
  int out_stride;
  const bf16_t* kcache;
  const bf16_t* vcache;
  const int* block_table;
  int table_stride;
  const int* q_start;   // [requests + 1]
  const int* kv_len;    // [requests]
  const int* tile_req;  // [tiles]
  const int* tile_row0; // [tiles] first row of the wavefront's first row tile
  const int* tile_row1; // [tiles] first row of its second row tile, -1 for none; null: the 16 rows after the first
  int n_tiles;
  int nq, nkv, group, P, p_shift, window;
  float scale_log2;  // scale * log2(e) > 0
  int split;         // keys per split, a multiple of 32
  int even;          // whether the wavefronts of a workgroup share the keys that are there evenly
  int max_splits;    // splits a tile may have (size of the scratch)
  float* part_o;     // [tiles][nkv][max_splits][16 * RT][D]
  float* part_ml;    // [tiles][nkv][max_splits][16 * RT][2]
  // [tiles][nkv] arrivals of a tile's splits, all zero between launches (null: the splits are
  // added by a kernel of their own): the workgroup whose arrival completes a tile adds its splits
  // and sets the count back to zero
  unsigned* tickets;
};

// A load that another workgroup's write-through store of the same launch is visible to.
__device__ __forceinline__ float shared_load_f32(const float* p) {
  return __uint_as_float(__hip_atomic_load((const uint32_t*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// What a (wavefront's) tile covers.  Per row tile: rows row0 .. row0 + 15 (row0 < 0: none),
// keys [lo, hi] that some row sees and [full_lo, full_hi] that every row sees.
struct TileRange {
  int req, qs, qlen, kvl, n_rows, lo, hi, s_first, s_last;
  int row0[2], rt_lo[2], rt_hi[2], full_lo[2], full_hi[2];
};

__device__ __forceinline__ TileRange tile_range(const AttnArgs& a, int tile, int row_tiles) {
  TileRange t;
  // a null tile list stands for one token a request, each a tile of its own
  t.req = a.tile_req ? a.tile_req[tile] : tile;
  t.qs = a.tile_req ? a.q_start[t.req] : t.req;
  t.qlen = a.tile_req ? a.q_start[t.req + 1] - t.qs : 1;
  t.kvl = a.kv_len[t.req];
  t.n_rows = t.qlen * a.group;
  t.row0[0] = a.tile_req ? a.tile_row0[tile] : 0;
  t.row0[1] = -1;
  if (row_tiles == 2) {
    t.row0[1] = a.tile_row1 ? a.tile_row1[tile] : t.row0[0] + 16;
    if (t.row0[1] >= t.n_rows || t.row0[0] < 0) t.row0[1] = -1;  // row0 < 0: a tile that only fills a group
  }
  t.lo = 0x7fffffff;
  t.hi = -1;
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    t.rt_lo[rt] = t.full_lo[rt] = 0x7fffffff;
    t.rt_hi[rt] = t.full_hi[rt] = -1;
    if (t.row0[rt] < 0) continue;
    // (a request of one token, decoded: no divisions in front of its first loads)
    const int first_tok = t.qlen == 1 ? 0 : t.row0[rt] / a.group;
    const int last_tok = t.qlen == 1 ? 0 : min(t.row0[rt] + 15, t.n_rows - 1) / a.group;
    const int pos_first = t.kvl - t.qlen + first_tok, pos_last = t.kvl - t.qlen + last_tok;
    t.rt_hi[rt] = pos_last;
    t.rt_lo[rt] = a.window > 0 ? max(0, pos_first - a.window + 1) : 0;
    t.full_hi[rt] = pos_first;
    t.full_lo[rt] = a.window > 0 ? max(0, pos_last - a.window + 1) : 0;
    t.lo = min(t.lo, t.rt_lo[rt]);
    t.hi = max(t.hi, t.rt_hi[rt]);
  }
  t.s_first = a.max_splits == 1 || t.lo == 0 ? 0 : t.lo / a.split;
  t.s_last = a.max_splits == 1 ? 0 : t.hi / a.split;
  return t;
}

// first <= x <= last as one unsigned comparison (an empty range, last < first, holds nothing)
struct Range {
  int first;
  unsigned span;
  __device__ __forceinline__ bool holds(int x) const { return (unsigned)(x - first) <= span; }
};
__device__ __forceinline__ Range range_of(int first, int last) {
  return last >= first ? Range{first, (unsigned)(last - first)} : Range{0x7fffffff, 0u};
}

// The maximum over the four lanes (r, 0..3) that share a row: lanes 16 and 32 apart,
// with the gfx950 swaps of 16-lane rows and of wavefront halves.
__device__ __forceinline__ float max_over_quarters(float x) {
  const unsigned u = __float_as_uint(x);
  const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const float y = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const unsigned v = __float_as_uint(y);
  const auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// The loads of one step of 32 keys.  Keys: lane (r, q) reads 8 values of key
// kb + 16 blk + r for every 32-wide step over the head size.  Values: lane (r, q)
// reads, for d = 16 dt + r, the 4 keys kb + 16 blk + 4q .. + 3.  Every address lies
// in a page of the tile's key range [lo, hi], so a load past the end reads valid
// memory (whose contents the masks keep out of the result).
template <int DT>
struct StepRegs {
  bf16x8_t kv[2][(DT + 1) / 2];
  union { bf16x4_t half[2]; uint32_t u[4]; bf16x8_t whole; } vv[DT];  // the two 16-key blocks side by side
};

// BIG: pages of 16 keys or more, so the 16 keys of a block lie in one page, which a
// scalar load looks up; the lane's part of the address is the same in every step.
// The pages of the two 16-key blocks of the step at `kb` (BIG only): looked up a step before
// the loads that need them are issued, so that no load waits for a table entry.
struct StepPages {
  int page[2];
};

__device__ __forceinline__ StepPages step_pages(const AttnArgs& a, const int* table, int kb, int lo, int hi) {
  const int sh = a.p_shift;
  StepPages p;
  p.page[0] = table[min(max(kb >> sh, lo >> sh), hi >> sh)];
  p.page[1] = table[min(max((kb + 16) >> sh, lo >> sh), hi >> sh)];
  return p;
}

template <int DT, bool BIG>
__device__ __forceinline__ void load_step(StepRegs<DT>& s, const AttnArgs& a, const int* table, const StepPages& pages,
                                          int kvh, int kb, int lo, int hi, int r, int q) {
  constexpr int D = DT * 16;
  constexpr int KS = (DT + 1) / 2;
  const int P = a.P, sh = a.p_shift;
  // the lane's own part of a key and of a value address inside any page of this kv head
  const unsigned lane_k = (unsigned)(kvh * P * D + r * 8);
  const unsigned lane_v = (unsigned)(kvh * P * D + (q * D + r) * 4);
#pragma unroll
  for (int blk = 0; blk < 2; ++blk) {
    const bf16_t* kp;
    const bf16_t* vp;
    if constexpr (BIG) {
      const int key0 = kb + blk * 16;
      // one 32 x 32 -> 64-bit product a page: the kv head's offset is in the lane's part already
      const size_t base = (size_t)(unsigned)pages.page[blk] * (unsigned)(a.nkv * P * D);
      const int in_page = key0 & (P - 1);
      kp = a.kcache + base + (unsigned)(in_page * 8) + lane_k;
      vp = a.vcache + base + (unsigned)((in_page >> 2) * (D * 4)) + lane_v;
    } else {
      const int kk = min(max(kb + blk * 16 + r, lo), hi);
      const int page = table[kk >> sh];
      kp = a.kcache + ((size_t)page * a.nkv + kvh) * ((size_t)P * D) + (size_t)(kk & (P - 1)) * 8;
      int kc = kb + blk * 16 + q * 4;
      if (kc > hi) kc = hi & ~3;
      if (kc + 3 < lo) kc = lo & ~3;
      const int vpage = table[kc >> sh];
      vp = a.vcache + ((size_t)vpage * a.nkv + kvh) * ((size_t)P * D) + (size_t)((kc & (P - 1)) >> 2) * (D * 4) + r * 4;
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int d0 = ks * 32 + q * 8;  // piece d0 / 8 of the key
      if (d0 < D) {
        s.kv[blk][ks] = *(const bf16x8_t*)(kp + (size_t)(d0 >> 3) * P * 8);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) s.kv[blk][ks][e] = (__bf16)0.f;
      }
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) s.vv[dt].half[blk] = *(const bf16x4_t*)(vp + dt * 64);
  }
}

// One row of a split tile from the partial results of its `nsp` splits, added in split order by
// one wavefront (lane i takes the statistics of split i, i + 64, ..; every lane then sums one
// or more of the row's D outputs over the splits, with the weights handed from lane to lane).
// Called inside the attention kernel by the workgroup that arrived last at the tile: the other
// splits' results were written through the caches by other workgroups of this launch.
__device__ __forceinline__ void merge_row_shared(const AttnArgs& a, const TileRange& t, const int tile, const int kvh,
                                                 const int row, const int rows_per_tile, const int nsp, const int D,
                                                 const int lane) {
  const int base = row < 16 ? t.row0[0] : t.row0[1];
  const int flat = base + (row & 15);
  if (base < 0 || flat >= t.n_rows) return;
  const size_t item0 = ((size_t)tile * a.nkv + kvh) * a.max_splits;
  const float* ml = a.part_ml + (item0 * rows_per_tile + row) * 2;
  const size_t ml_step = (size_t)rows_per_tile * 2;
  const float* po = a.part_o + (item0 * rows_per_tile + row) * D;
  const size_t po_step = (size_t)rows_per_tile * D;
  const int tok = flat / a.group, g = flat - tok * a.group;
  bf16_t* op = a.out + (size_t)(t.qs + tok) * a.out_stride + (size_t)(kvh * a.group + g) * D;
  if (nsp <= 64) {
    // every load of the row is asked for before the first is waited for: one trip to memory
    float ms_own = -INFINITY, ls_own = 0.f;
    if (lane < nsp) {
      ms_own = shared_load_f32(ml + lane * ml_step);
      ls_own = shared_load_f32(ml + lane * ml_step + 1);
    }
    constexpr int AHEAD = 16;
    float ahead[AHEAD];
    const int d_first = min(lane, D - 1);
#pragma unroll
    for (int sp = 0; sp < AHEAD; ++sp) ahead[sp] = sp < nsp ? shared_load_f32(po + sp * po_step + d_first) : 0.f;
    const float m = wave_max(ms_own);
    const float w = ms_own == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ms_own - m);
    const float inv = 1.0f / wave_sum(w * ls_own);
    for (int d0 = 0; d0 < D; d0 += 64) {  // every lane stays in the loop: the weights come from all of them
      const int d = min(d0 + lane, D - 1);
      float o = 0.f;
#pragma unroll
      for (int sp = 0; sp < AHEAD; ++sp) {
        const float ws = __shfl(w, sp, 64);
        const float v = d0 == 0 ? ahead[sp] : (sp < nsp ? shared_load_f32(po + sp * po_step + d) : 0.f);
        if (sp < nsp) o += ws * v;
      }
#pragma unroll 8
      for (int sp = AHEAD; sp < nsp; ++sp) o += __shfl(w, sp, 64) * shared_load_f32(po + sp * po_step + d);
      if (d0 + lane < D) op[d] = __float2bfloat16(o * inv);
    }
    return;
  }
  float m = -INFINITY;
  for (int sp = lane; sp < nsp; sp += 64) m = fmaxf(m, shared_load_f32(ml + sp * ml_step));
  m = wave_max(m);
  float l = 0.f;
  for (int sp = lane; sp < nsp; sp += 64) {
    const float ms = shared_load_f32(ml + sp * ml_step);
    l += (ms == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ms - m)) * shared_load_f32(ml + sp * ml_step + 1);
  }
  const float inv = 1.0f / wave_sum(l);
  for (int d = lane; d < D; d += 64) {
    float o = 0.f;
#pragma unroll 8
    for (int sp = 0; sp < nsp; ++sp) {
      const float ms = shared_load_f32(ml + sp * ml_step);
      const float w = ms == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ms - m);
      o += w * shared_load_f32(po + sp * po_step + d);
    }
    op[d] = __float2bfloat16(o * inv);
  }
}

// Wavefronts a workgroup may have: the fewer, the more registers each has for loads in flight.
__host__ __device__ constexpr int max_waves(int dt, int rt) { return rt == 2 ? 4 : (dt <= 4 ? 16 : 8); }

// One (tile, kv head, split) item of the attention: the body of the kernel, for the NW
// wavefronts of a workgroup together (all of them must call it: it synchronises them when
// NW > 1).  wg_part is LDS of NW * 16 * RT * (D + 4) floats (unused when NW is 1).
// SHARED (a.tickets must be there): the workgroups of the launch hand the partial results of
// split tiles to each other.  They are written with stores that write through the caches; a
// workgroup then counts itself in at the tile's ticket, and the one whose arrival makes the
// tile's splits complete adds them, in split order whoever it is, and writes the rows: no
// second kernel.  A tile with one split writes its rows itself as ever.
// PF steps of loads are in flight: a lone wavefront on a long tile waits on memory otherwise.
// GROUPED (long prompts: two row tiles, pages of 16 keys or more, whole keys, no splits): the
// GROUP_WAVES wavefronts of the workgroup have a tile each (`tile` is the wavefront's own, two
// neighbouring row tiles), and all the tiles belong to one request: the host fills a request's
// tiles up to a multiple of GROUP_WAVES with empty ones (row0 < 0).  The wavefronts walk the
// keys that any of them sees together: every step's keys and values are loaded once, a quarter
// by each wavefront, and pass through LDS (two buffers, one barrier a step) in the lane order
// of the operands; the pages of a step are looked up a step before its loads are issued.  No
// ring of loads is held in registers, so twice the wavefronts fit a SIMD, and a wavefront issues
// a quarter of the loads and of their addresses.  With KSPLIT > 1 the workgroup has KSPLIT such
// sets of wavefronts on the same tiles; set c takes the steps c, c + KSPLIT, .. through buffers of
// its own, and the sets' results are added through LDS at the end, in the order of the sets.
// wg_part: 64 bytes for the tiles' key ranges, then for each set 2 buffers of (2 KS + DT) KB.
#define GROUP_WAVES 4
template <int DT, int RT, bool BIG, bool SHARED, bool GROUPED = false, int KSPLIT = 1>
__device__ __forceinline__ void attention_item(const AttnArgs& a, const int tile, const int kvh, const int split_index,
                                               float* wg_part, const int NW) {
  static_assert(!GROUPED || (RT == 2 && BIG && !SHARED), "grouped tiles: prompts on pages of 16 keys or more");
  static_assert(KSPLIT == 1 || GROUPED, "steps are dealt out among the wavefronts of grouped tiles only");
  constexpr int D = DT * 16;
  constexpr int KS = (DT + 1) / 2;  // 32-wide steps over the head size
  constexpr int PF = RT == 1 ? 2 : 3;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, q = lane >> 4;
  const TileRange t = tile_range(a, tile, RT);
  const int s = GROUPED ? 0 : t.s_first + split_index;
  if (!GROUPED && s > t.s_last) return;
  const int nsp = GROUPED ? 1 : t.s_last - t.s_first + 1;
  // this wavefront's part of the split: `sub` keys, a multiple of 32.  Fixed parts of the split, or (`even`) of the keys that are there:
  // of a request (or a prompt's tile) that ends, or whose window begins, inside the split every wavefront then takes as many as the others.  Fixed
  // parts give a workgroup as many wavefronts as it has keys to read, so that requests of all lengths end at one time, and are the
  // rule; the host asks for even ones where they were ahead.
  const int k_first = max((t.lo >> 5) << 5, s * a.split), k_last = min(t.hi + 1, (s + 1) * a.split);
  const bool even = a.even != 0;
  const int sub = even ? (((k_last - k_first + NW - 1) / NW + 31) >> 5) << 5 : a.split / NW;
  const int part = (even ? k_first : s * a.split) + wave * sub;
  const int k_begin = max(k_first, part), k_end = min(k_last, part + sub);
  const int* table = a.block_table + (size_t)t.req * a.table_stride;

  // the steps (by their first key) in which a row tile has a row that sees a key, in which all
  // of its rows see all 32 keys, and in which all 32 keys lie in the tile's range
  Range active[RT], unmasked[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    active[rt] = range_of(t.rt_lo[rt] - 31, t.rt_hi[rt]);
    unmasked[rt] = range_of(t.full_lo[rt], t.full_hi[rt] - 31);
  }
  const Range inside = range_of(t.lo, t.hi - 31);

  // this lane's row in each of the RT tiles
  // (the first key a row sees and the row's number are worked out again where they are needed,
  // at the masked steps and at the end: two registers less a row tile in the loop)
  int pos_r[RT];
  bf16x8_t qv[RT][KS];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int flat = t.row0[rt] >= 0 ? t.row0[rt] + r : t.n_rows;
    const bool valid = flat < t.n_rows;
    const int fl = valid ? flat : t.n_rows - 1;
    const int tok = t.qlen == 1 ? 0 : fl / a.group, g = fl - tok * a.group;
    const int pos = t.kvl - t.qlen + tok;
    pos_r[rt] = valid ? pos : -1;
    const bf16_t* qp = a.q + (size_t)(t.qs + tok) * a.q_stride + (size_t)(kvh * a.group + g) * D;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int d0 = ks * 32 + q * 8;
      if (d0 < D) {
        qv[rt][ks] = *(const bf16x8_t*)(qp + d0);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) qv[rt][ks][e] = (__bf16)0.f;
      }
    }
  }

  // Running maximum of the row's products and sum of this lane's keys.  The maximum itself is the terms' reference, in every step: so the greatest
  // weight is exactly 1 in bfloat16 too.  A reference that may be behind it moves seldom (us a layer of 8 kv heads: 32 heads of 64, 2,048 tokens
  // 47.1 / 42.0, 8,192 370 / 343), but rounds the greatest weight, 2^-8 of a result that is that key's values.  (The same reference with lanes that agree
  // only in steps where one has a greater product gives these bits and is slower, 51.7 and 406.)
  float m_run[RT], l_run[RT];
  f32x4_t acc[RT][DT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    m_run[rt] = -INFINITY;
    l_run[rt] = 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc[rt][dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  auto compute_step = [&](StepRegs<DT>& cur, const int kb) {
    if (!inside.holds(kb)) {
      // values of keys outside the tile's range may be anything (a freed page): make them
      // zero by masking their 16 bits
      uint32_t keep[4];
#pragma unroll
      for (int blk = 0; blk < 2; ++blk)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int key = kb + blk * 16 + q * 4 + 2 * h;
          const uint32_t lo16 = (key >= t.lo && key <= t.hi) ? 0x0000ffffu : 0u;
          const uint32_t hi16 = (key + 1 >= t.lo && key + 1 <= t.hi) ? 0xffff0000u : 0u;
          keep[blk * 2 + h] = lo16 | hi16;
        }
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) cur.vv[dt].u[i] &= keep[i];
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      if (!active[rt].holds(kb)) continue;  // none of the tile's rows sees these keys
      f32x4_t st[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        st[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cur.kv[0][ks], qv[rt][ks], st[0], 0, 0, 0);
        st[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cur.kv[1][ks], qv[rt][ks], st[1], 0, 0, 0);
      }
      // scores stay as the products are (scale_log2 > 0 keeps their order); the scale goes
      // into the exponent's multiply-add
      float sc[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) sc[e] = st[e >> 2][e & 3];
      if (!unmasked[rt].holds(kb)) {
        const int lo_row = a.window > 0 ? max(0, pos_r[rt] - a.window + 1) : 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int key = kb + (e >> 2) * 16 + q * 4 + (e & 3);
          if (!(key >= lo_row && key <= pos_r[rt])) sc[e] = -INFINITY;
        }
      }
      float mx = fmaxf(fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3])), fmaxf(fmaxf(sc[4], sc[5]), fmaxf(sc[6], sc[7])));
      mx = max_over_quarters(mx);
      const float m_new = fmaxf(m_run[rt], mx);
      const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
      const float mc = m_use * a.scale_log2;
      if (__any(m_new > m_run[rt])) {
        // some row's maximum moved: weigh what was summed so far
        const float alpha = __builtin_amdgcn_exp2f(fmaf(m_run[rt], a.scale_log2, -mc));  // 0 while nothing was seen
        l_run[rt] *= alpha;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) acc[rt][dt] *= alpha;
        m_run[rt] = m_new;
      }
      float p[8];
      bf16x8_t pb;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        p[e] = __builtin_amdgcn_exp2f(fmaf(sc[e], a.scale_log2, -mc));
        pb[e] = (__bf16)p[e];
      }
      l_run[rt] += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        acc[rt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cur.vv[dt].whole, pb, acc[rt][dt], 0, 0, 0);
    }
  };

  if constexpr (GROUPED) {
    constexpr int NK = 2 * KS, NV = 2 * DT;  // fragments of a step: keys 1 KB each, values 512 bytes each
    constexpr int NKR = (NK + GROUP_WAVES - 1) / GROUP_WAVES, NVR = (NV + GROUP_WAVES - 1) / GROUP_WAVES;
    // the wavefront's place among those that share the tiles' loads, and which of the KSPLIT such
    // sets it belongs to (set c takes the steps c, c + KSPLIT, ..)
    const int member = wave % GROUP_WAVES, crew = wave / GROUP_WAVES;
    int* ranges = (int*)wg_part;
    bf16x8_t* k_lds = (bf16x8_t*)(wg_part + 16) + (size_t)crew * (2 * (NK + DT) * 64);
    // values: the two 16-key blocks of a fragment side by side, as the value product's operand wants them
    bf16x8_t* v_lds = k_lds + 2 * NK * 64;  // [buffer][dt][lane]
    if (lane == 0 && crew == 0) {
      ranges[2 * member] = t.lo;
      ranges[2 * member + 1] = t.hi;
    }
    __syncthreads();
    int glo = 0x7fffffff, ghi = -1;
#pragma unroll
    for (int w = 0; w < GROUP_WAVES; ++w) {
      glo = min(glo, ranges[2 * w]);
      ghi = max(ghi, ranges[2 * w + 1]);
    }
    glo = __builtin_amdgcn_readfirstlane(glo);
    ghi = __builtin_amdgcn_readfirstlane(ghi);
    if (ghi < 0) return;  // the same for every wavefront of the workgroup
    const int g_begin = (glo >> 5) << 5, n_steps = (ghi + 1 - g_begin + 31) >> 5;
    const int P = a.P;
    const unsigned head_off = (unsigned)(kvh * P * D);
    const bool mine = t.hi >= 0;  // else an empty tile: this wavefront only carries its share of the loads

    bf16x8_t kreg[NKR];
    bf16x4_t vreg[NVR];
    // this wavefront's fragments of the step at kb, from memory into registers
    auto fetch = [&](const int kb, const StepPages& pg) {
#pragma unroll
      for (int i = 0; i < NKR; ++i) {
        const int f = i * GROUP_WAVES + member;
        if (f < NK) {
          const int blk = f / KS, ks = f - blk * KS;
          const int in_page = (kb + blk * 16) & (P - 1);
          // (chosen, not indexed: an array indexed by a number known only at run time lives in memory)
          const size_t base = (size_t)(unsigned)(blk ? pg.page[1] : pg.page[0]) * (unsigned)(a.nkv * P * D);
          const int d0 = ks * 32 + q * 8;
          if (d0 < D) {
            kreg[i] = *(const bf16x8_t*)(a.kcache + base + head_off + (unsigned)((((d0 >> 3) * P) + in_page + r) * 8));
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) kreg[i][e] = (__bf16)0.f;
          }
        }
      }
#pragma unroll
      for (int i = 0; i < NVR; ++i) {
        const int f = i * GROUP_WAVES + member;
        if (f < NV) {
          const int blk = f / DT, dt = f - blk * DT;
          const int in_page = (kb + blk * 16) & (P - 1);
          const size_t base = (size_t)(unsigned)(blk ? pg.page[1] : pg.page[0]) * (unsigned)(a.nkv * P * D);
          vreg[i] = *(const bf16x4_t*)(a.vcache + base + head_off + (unsigned)((((in_page >> 2) + q) * (D * 4)) + (dt * 16 + r) * 4));
        }
      }
    };
    // ... from the registers into buffer `buf`
    auto stash = [&](const int buf) {
#pragma unroll
      for (int i = 0; i < NKR; ++i) {
        const int f = i * GROUP_WAVES + member;
        if (f < NK) k_lds[(size_t)(buf * NK + f) * 64 + lane] = kreg[i];
      }
#pragma unroll
      for (int i = 0; i < NVR; ++i) {
        const int f = i * GROUP_WAVES + member;
        if (f < NV) {
          const int blk = f / DT, dt = f - blk * DT;
          ((bf16x4_t*)(v_lds + (size_t)(buf * DT + dt) * 64 + lane))[blk] = vreg[i];
        }
      }
    };
    // this set's j-th step and whether there is one; every wavefront of the workgroup goes round
    // the loop equally often, for the barriers' sake
    auto first_key = [&](const int j) { return g_begin + 32 * (crew + KSPLIT * j); };
    auto has = [&](const int j) { return crew + KSPLIT * j < n_steps; };
    const int rounds = (n_steps + KSPLIT - 1) / KSPLIT;
    StepPages pg = {};
    if (has(0)) {
      pg = step_pages(a, table, first_key(0), glo, ghi);
      fetch(first_key(0), pg);
    }
    if (has(1)) pg = step_pages(a, table, first_key(1), glo, ghi);
    if (has(0)) stash(0);
    if (has(1)) fetch(first_key(1), pg);
    if (has(2)) pg = step_pages(a, table, first_key(2), glo, ghi);
    __syncthreads();
    for (int j = 0; j < rounds; ++j) {
      const int kb = first_key(j), buf = j & 1;
      // the other buffer was last read before the barrier that ended the step before
      if (has(j + 1)) stash(buf ^ 1);
      if (has(j + 2)) fetch(first_key(j + 2), pg);
      if (has(j + 3)) pg = step_pages(a, table, first_key(j + 3), glo, ghi);
      if (has(j) && mine && (active[0].holds(kb) || active[1].holds(kb))) {
        StepRegs<DT> cur;
#pragma unroll
        for (int blk = 0; blk < 2; ++blk) {
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) cur.kv[blk][ks] = k_lds[(size_t)(buf * NK + blk * KS + ks) * 64 + lane];
        }
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) cur.vv[dt].whole = v_lds[(size_t)(buf * DT + dt) * 64 + lane];
        compute_step(cur, kb);
      }
      __syncthreads();
    }
  } else {
  StepRegs<DT> ring[PF];
  // With two row tiles (prompts: many steps a wavefront) the pages of a step are looked up when
  // the loads of the step before are issued; with one (decode: few steps) right before its own.
  constexpr bool AHEAD = BIG && RT == 2;
  StepPages pages = {};
  if (AHEAD && k_begin < k_end) pages = step_pages(a, table, k_begin, t.lo, t.hi);
  auto issue = [&](StepRegs<DT>& regs, int k) {
    if (BIG && !AHEAD) pages = step_pages(a, table, k, t.lo, t.hi);
    load_step<DT, BIG>(regs, a, table, pages, kvh, k, t.lo, t.hi, r, q);
    if (AHEAD && k + 32 < k_end) pages = step_pages(a, table, k + 32, t.lo, t.hi);
  };
  // Prompts' walks are whole turns of the ring, in which every load is asked for, then what is left: behind a load that may not have been
  // asked for the compiler waits for all that were (us a layer: 24 heads of 128, 1,000 tokens by pairs 27.4 / 26.3, 32 heads 1,024 30.2 / 27.8).
  // Decoded tokens' few steps are asked for together as it is (with turns of their own 64 uneven requests take 45.8 for 43.4).
  int k_next = k_begin;
  if (RT == 2 && k_end - k_begin > 32 * (2 * PF - 1)) {
#pragma unroll
    for (int i = 0; i < PF; ++i) issue(ring[i], k_begin + 32 * i);
    do {
#pragma unroll
      for (int i = 0; i < PF; ++i) {
        compute_step(ring[i], k_next + 32 * i);
        issue(ring[i], k_next + 32 * (i + PF));
      }
      k_next += 32 * PF;
    } while (k_end - k_next > 32 * (2 * PF - 1));
  } else {
#pragma unroll
    for (int i = 0; i < PF; ++i)
      if (k_begin + 32 * i < k_end) issue(ring[i], k_begin + 32 * i);
  }
  for (int kb = k_next; kb < k_end; kb += 32 * PF) {
#pragma unroll
    for (int i = 0; i < PF; ++i) {
      const int k = kb + 32 * i;
      if (k < k_end) {
        compute_step(ring[i], k);
        if (k + 32 * PF < k_end) issue(ring[i], k + 32 * PF);
      }
    }
  }
  }

  // acc[rt][dt][j] of lane (r, q) is O^T[d = 16 dt + 4q + j][row r]
  const size_t item0 = ((size_t)tile * a.nkv + kvh) * a.max_splits;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    float l = l_run[rt];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    l_run[rt] = l;
    m_run[rt] *= a.scale_log2;  // from here on in units of log 2, as the merges take it
  }
  const bool hand_over = SHARED && nsp > 1;  // the same for every wavefront of the workgroup
  if (!GROUPED && NW > 1) {
    // every wavefront leaves (max, sum, weighted values) of its rows; wavefront 0 adds them in order
    constexpr int ROW = D + 4;  // max, sum, two unused, then the values (16-byte aligned)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      float* row = wg_part + ((size_t)wave * 16 * RT + rt * 16 + r) * ROW;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) *(f32x4_t*)(row + 4 + dt * 16 + q * 4) = acc[rt][dt];
      if (q == 0) {
        row[0] = m_run[rt];
        row[1] = l_run[rt];
      }
    }
    __syncthreads();
    if (wave != 0 && !hand_over) return;
    if (wave == 0) {
      // (rows of several wavefronts are on their way together; behind the last one it is asked for again and not used)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const float* mine = wg_part + (size_t)(rt * 16 + r) * ROW;
      constexpr int NEXT = 16 * RT * ROW;  // to the next wavefront's row
      float m = -INFINITY;
      for (int w = 0; w < NW; w += 4)
        m = fmaxf(m, fmaxf(fmaxf(mine[w * NEXT], mine[min(w + 1, NW - 1) * NEXT]), fmaxf(mine[min(w + 2, NW - 1) * NEXT], mine[min(w + 3, NW - 1) * NEXT])));
      float l = 0.f;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) acc[rt][dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      auto add = [&](const float mw, const float lw, const f32x4_t (&v)[DT]) {
        const float f = (mw == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(mw - m);
        l += f * lw;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) acc[rt][dt] += f * v[dt];
      };
      for (int w = 0; w < NW; w += 2) {
        float mw[2], lw[2];
        f32x4_t v[2][DT];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const float* row = mine + min(w + i, NW - 1) * NEXT;
          mw[i] = row[0];
          lw[i] = row[1];
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) v[i][dt] = *(const f32x4_t*)(row + 4 + dt * 16 + q * 4);
        }
        add(mw[0], lw[0], v[0]);
        if (w + 1 < NW) add(mw[1], lw[1], v[1]);
      }
      m_run[rt] = m;
      l_run[rt] = l;
    }
    }
  }
  if constexpr (GROUPED && KSPLIT > 1) {
    // The sets of wavefronts that took the steps in turn each hold (max, sum, weighted values) of
    // the same rows: all but the first leave theirs in LDS (over the buffers of keys and values,
    // which the loop's last barrier has released), one row tile at a time, and the first adds them
    // in the order of the sets.
    constexpr int ROW = D + 4;
    const int member = wave % GROUP_WAVES, crew = wave / GROUP_WAVES;
    float* left = wg_part + 16;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      if (crew > 0) {
        float* row = left + ((size_t)((crew - 1) * GROUP_WAVES + member) * 16 + r) * ROW;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) *(f32x4_t*)(row + 4 + dt * 16 + q * 4) = acc[rt][dt];
        if (q == 0) {
          row[0] = m_run[rt];
          row[1] = l_run[rt];
        }
      }
      __syncthreads();
      if (crew == 0) {
        float m = m_run[rt];
#pragma unroll
        for (int c = 1; c < KSPLIT; ++c) m = fmaxf(m, left[((size_t)((c - 1) * GROUP_WAVES + member) * 16 + r) * ROW]);
        const float f0 = (m_run[rt] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(m_run[rt] - m);
        float l = f0 * l_run[rt];
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) acc[rt][dt] *= f0;
#pragma unroll
        for (int c = 1; c < KSPLIT; ++c) {
          const float* row = left + ((size_t)((c - 1) * GROUP_WAVES + member) * 16 + r) * ROW;
          const float mw = row[0];
          const float f = (mw == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(mw - m);
          l += f * row[1];
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) acc[rt][dt] += f * *(const f32x4_t*)(row + 4 + dt * 16 + q * 4);
        }
        m_run[rt] = m;
        l_run[rt] = l;
      }
      if (rt + 1 < RT) __syncthreads();  // before the next row tile's values take the place
    }
    if (crew > 0) return;
  }
  if (wave == 0 || GROUPED) {
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const float l = l_run[rt];
    const int flat = t.row0[rt] >= 0 ? t.row0[rt] + r : t.n_rows;
    if (flat >= t.n_rows) continue;
    if (nsp == 1) {
      const int tok = flat / a.group, g = flat - tok * a.group;
      bf16_t* op = a.out + (size_t)(t.qs + tok) * a.out_stride + (size_t)(kvh * a.group + g) * D;
      const float inv = 1.0f / l;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        union { bf16_t h[4]; uint2 u; } pk;
#pragma unroll
        for (int j = 0; j < 4; ++j) pk.h[j] = __float2bfloat16(acc[rt][dt][j] * inv);
        *(uint2*)(op + dt * 16 + q * 4) = pk.u;
      }
    } else {
      const size_t item = item0 + (s - t.s_first);
      float* po = a.part_o + (item * (16 * RT) + rt * 16 + r) * D;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) store_f32x4<SHARED>(po + dt * 16 + q * 4, acc[rt][dt]);
      if (q == 0) {
        float* pm = a.part_ml + (item * (16 * RT) + rt * 16 + r) * 2;
        store_f32x2<SHARED>(pm, m_run[rt], l);
      }
    }
  }
  }
  if constexpr (SHARED) {
    if (!hand_over) return;
    int last = 0;
    if (wave == 0) {
      // this wavefront's stores have been written through; then it counts the split in
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (lane == 0) {
        unsigned* ticket = a.tickets + (size_t)tile * a.nkv + kvh;
        const unsigned before = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last = before + 1 == (unsigned)nsp;
        if (last) __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
      }
      last = __builtin_amdgcn_readfirstlane(last);
      if (NW > 1 && lane == 0) ((int*)wg_part)[0] = last;  // wavefront 0 has read all it needs from here
    }
    if (NW > 1) {
      __syncthreads();
      last = ((const int*)wg_part)[0];
    }
    if (!last) return;
    for (int row = wave; row < 16 * RT; row += NW) merge_row_shared(a, t, tile, kvh, row, 16 * RT, nsp, D, lane);
  }
}
