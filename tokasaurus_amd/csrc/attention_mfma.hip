// Paged attention on the gfx950 matrix cores, bfloat16 storage, 32-bit softmax.
// One kernel serves prompt portions and single decoded tokens.
//
// Rows.  For a request and a kv head, the rows are the pairs (token of this step,
// query head of the kv head's group), numbered token * group + head, and cut into
// row tiles of 16.  A wavefront owns RT row tiles of one request and walks the keys
// they may see in steps of 32.  With the keys as the first operand of
// v_mfma_f32_16x16x32_bf16 and the queries as the second,
//     S^T[key 4q+j][row r]  is element j of lane (r = lane % 16, q = lane / 16),
// so a lane holds, for ONE row, 4 keys of each 16-key block.  These 8 numbers
// are exactly what the lane must provide as the second operand of the product
// O^T = V^T P^T, if slot 8q+j of that product's inner index stands for key 4q+j
// of the first block and slot 8q+4+j for key 4q+j of the second.  A page keeps
// its values in groups of 4 tokens ([P / 4][d][4]), so the matching first operand
// is read with two 8-byte loads per lane, and its keys in pieces of 8 elements
// ([d / 8][P][8]), so that in both kinds of load 16 neighbouring lanes read
// consecutive memory: the vector cache handles a load at the rate of the cache
// lines it touches, not of its bytes.  Nothing passes through LDS.
// P is a power of two, at least 4.
//
// Two row tiles of a wavefront need not be neighbours: under a causal mask the host
// pairs an early tile of a prompt with a late one, so that every wavefront has the
// same number of (row tile, key step) products.  A row tile is skipped in the steps
// that none of its rows sees; steps that all of its rows see whole are not masked.
//
// Splits.  The keys of a wavefront's tiles are cut at absolute multiples of `split`;
// each (tile, kv head, split) is one workgroup of NW wavefronts, which cut the split's
// keys into NW consecutive parts (multiples of 32) and add their results through
// LDS in wavefront order.  A tile with one split writes the output; otherwise
// partial (max, sum, weighted values) go to scratch and a second kernel adds them
// in split order.  With few tiles (decode) many wavefronts with two or three steps
// each keep enough loads in flight; with many tiles (prompts) NW is 1.
#include "calls.h"
#include "attention_mfma.h"

template <int DT, int RT, bool BIG, bool SHARED>
__global__ __launch_bounds__(64 * max_waves(DT, RT)) void paged_attention_mfma_kernel(AttnArgs a) {
  extern __shared__ __align__(16) float wg_part[];  // [wavefront][16 * RT rows][D + 4], when NW > 1
  // Workgroups go to the chip's eight dies in turn, each with a cache of its own.  Prompts
  // (two row tiles): kv head fastest, so a die serves few kv heads and keeps their keys and
  // values, which every tile of the request reads again, to itself.  Decoded tokens read
  // their keys once: tile fastest, as measured.
  // The splits of one tile must not all land on one die: with a multiple of 8 (tile, kv head)
  // pairs a workgroup's die would be its pair's number modulo 8 whatever its split, and one long
  // request among short ones would be read by an eighth of the chip.  So the pair that a
  // workgroup takes is turned by its split's number within its group of eight.  (Not with one
  // tile: its kv heads are spread over the dies as they are, and the splits of a head, which
  // the last of them adds, stay in one die's cache.)
  unsigned x = blockIdx.x;
  if ((gridDim.x & 7) == 0 && a.n_tiles > 1) x = (x & ~7u) | ((x + blockIdx.z) & 7u);
  const int kvh = RT == 2 ? x % a.nkv : x / a.n_tiles;
  const int tile = RT == 2 ? x / a.nkv : x % a.n_tiles;
  attention_item<DT, RT, BIG, SHARED>(a, tile, kvh, blockIdx.z, wg_part, blockDim.x >> 6);
}

// Long prompts on pages of 16 keys or more: GROUP_WAVES tiles of one request a workgroup, which
// share every load of keys and values through LDS (see attention_item, GROUPED).  KSPLIT > 1:
// KSPLIT sets of GROUP_WAVES wavefronts take the steps of the same tiles in turn and add their
// results through LDS at the end: the longest group's walk is a KSPLIT-th as long, which counts
// when the launch has too few groups for the short ones to fill the time the long ones take.
template <int DT, int KSPLIT>
__global__ __launch_bounds__(64 * GROUP_WAVES * KSPLIT) void paged_attention_group_kernel(AttnArgs a) {
  extern __shared__ __align__(16) float wg_part[];
  const int kvh = blockIdx.x % a.nkv, group = blockIdx.x / a.nkv;  // kv head fastest, as above
  // (the wavefront's number as a scalar: what a tile covers then stays in scalar registers)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  attention_item<DT, 2, true, false, true, KSPLIT>(a, group * GROUP_WAVES + wave % GROUP_WAVES, kvh, 0, wg_part,
                                                   GROUP_WAVES * KSPLIT);
}

// Adds the partial results of split tiles, always in split order.  One wavefront
// per (tile, kv head, row): lane i takes the statistics of split i (of splits i, i + 64, ..),
// then every lane sums one (or more) of the row's d outputs over the splits, with the
// weights handed from lane to lane.  Where the partial results lie depends on the launch
// alone, so the first MG_AHEAD splits are loaded before the tile's range (which says how
// many of them count) has arrived: the kernel is little more than one trip to memory.
#define MG_AHEAD 16
__global__ __launch_bounds__(256) void attention_merge_kernel(AttnArgs a, int D, int row_tiles) {
  const int tile = blockIdx.x, kvh = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.z * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int rows_per_tile = 16 * row_tiles;
  const size_t item0 = ((size_t)tile * a.nkv + kvh) * a.max_splits;
  const float* ml = a.part_ml + (item0 * rows_per_tile + row) * 2;  // split sp is sp * rows_per_tile * 2 further
  const size_t ml_step = (size_t)rows_per_tile * 2;
  const float* po = a.part_o + (item0 * rows_per_tile + row) * D;
  const size_t po_step = (size_t)rows_per_tile * D;
  // ahead of everything: what may be stale or never written is not used below
  float ahead[MG_AHEAD];
  const int d_first = min(lane, D - 1);
#pragma unroll
  for (int sp = 0; sp < MG_AHEAD; ++sp) ahead[sp] = sp < a.max_splits ? po[sp * po_step + d_first] : 0.f;
  float ms_own = -INFINITY, ls_own = 0.f;
  if (lane < a.max_splits) {
    ms_own = ml[lane * ml_step];
    ls_own = ml[lane * ml_step + 1];
  }

  const TileRange t = tile_range(a, tile, row_tiles);
  const int nsp = t.s_last - t.s_first + 1;
  if (nsp == 1) return;
  const int base = row < 16 ? t.row0[0] : t.row0[1];
  const int flat = base + (row & 15);
  if (base < 0 || flat >= t.n_rows) return;
  const int tok = flat / a.group, g = flat - tok * a.group;
  bf16_t* op = a.out + (size_t)(t.qs + tok) * a.out_stride + (size_t)(kvh * a.group + g) * D;
  if (lane >= nsp) ms_own = -INFINITY;
  float m = ms_own;
  for (int sp = lane + 64; sp < nsp; sp += 64) m = fmaxf(m, ml[sp * ml_step]);
  m = wave_max(m);
  if (nsp <= 64) {
    const float w = ms_own == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ms_own - m);
    const float inv = 1.0f / wave_sum(lane < nsp ? w * ls_own : 0.f);
    for (int d0 = 0; d0 < D; d0 += 64) {  // every lane stays in the loop: the weights come from all of them
      const int d = min(d0 + lane, D - 1);
      float o = 0.f;
#pragma unroll
      for (int sp = 0; sp < MG_AHEAD; ++sp) {
        const float ws = __shfl(w, sp, 64);
        const float v = d0 == 0 ? ahead[sp] : (sp < nsp ? po[sp * po_step + d] : 0.f);
        if (sp < nsp) o += ws * v;
      }
#pragma unroll 8
      for (int sp = MG_AHEAD; sp < nsp; ++sp) o += __shfl(w, sp, 64) * po[sp * po_step + d];
      if (d0 + lane < D) op[d] = __float2bfloat16(o * inv);
    }
    return;
  }
  float l = 0.f;
  for (int sp = lane; sp < nsp; sp += 64) {
    const float ms = ml[sp * ml_step];
    l += (ms == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ms - m)) * ml[sp * ml_step + 1];
  }
  const float inv = 1.0f / wave_sum(l);
  for (int d = lane; d < D; d += 64) {
    float o = 0.f;
#pragma unroll 8
    for (int sp = 0; sp < nsp; ++sp) {
      const float ms = ml[sp * ml_step];
      const float w = ms == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ms - m);
      o += w * po[sp * po_step + d];
    }
    op[d] = __float2bfloat16(o * inv);
  }
}

template <int DT, int RT>
static bool launch_attn(const AttnArgs& a, int grid_splits, int nw, hipStream_t stream) {
  const size_t lds = nw > 1 ? (size_t)nw * 16 * RT * (DT * 16 + 4) * sizeof(float) : 0;
  // the splits of decoded tokens' tiles (one row tile) are added by whoever arrives last, when the caller brings tickets
  const bool shared = RT == 1 && a.tickets != nullptr;
  auto kernel = a.P >= 16 ? (shared ? paged_attention_mfma_kernel<DT, RT, true, RT == 1> : paged_attention_mfma_kernel<DT, RT, true, false>)
                          : (shared ? paged_attention_mfma_kernel<DT, RT, false, RT == 1> : paged_attention_mfma_kernel<DT, RT, false, false>);
  if (lds > 64 * 1024 &&
      hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return false;
  hipLaunchKernelGGL(kernel, dim3(a.n_tiles * a.nkv, 1, grid_splits), dim3(64 * nw), lds, stream, a);
  return true;
}

// LDS of a workgroup of grouped tiles: the tiles' key ranges, then for each set of wavefronts two
// buffers of a step's keys and values; the results that the sets leave for the first one at the
// end (one row tile at a time) lie over the buffers.
static size_t group_lds_bytes(int dt, int ksplit) {
  const size_t buffers = (size_t)ksplit * 2 * (2 * ((dt + 1) / 2) * 1024 + 2 * dt * 512);
  const size_t left = (size_t)(ksplit - 1) * GROUP_WAVES * 16 * (dt * 16 + 4) * sizeof(float);
  return 64 + (buffers > left ? buffers : left);
}

template <int DT, int KSPLIT>
static bool launch_group(const AttnArgs& a, hipStream_t stream) {
  const size_t lds = group_lds_bytes(DT, KSPLIT);
  auto kernel = paged_attention_group_kernel<DT, KSPLIT>;
  if (lds > 64 * 1024 &&
      hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return false;
  hipLaunchKernelGGL(kernel, dim3(a.n_tiles / GROUP_WAVES * a.nkv), dim3(64 * GROUP_WAVES * KSPLIT), lds, stream, a);
  return true;
}

static bool launch_group_d(const AttnArgs& a, int dt, int ksplit, hipStream_t stream) {
  if (ksplit == 2) {
    switch (dt) {
      case 1: return launch_group<1, 2>(a, stream);
      case 2: return launch_group<2, 2>(a, stream);
      case 3: return launch_group<3, 2>(a, stream);
      case 4: return launch_group<4, 2>(a, stream);
      case 5: return launch_group<5, 2>(a, stream);
      case 6: return launch_group<6, 2>(a, stream);
      case 7: return launch_group<7, 2>(a, stream);
      case 8: return launch_group<8, 2>(a, stream);
      default: return false;
    }
  }
  switch (dt) {
    case 1: return launch_group<1, 1>(a, stream);
    case 2: return launch_group<2, 1>(a, stream);
    case 3: return launch_group<3, 1>(a, stream);
    case 4: return launch_group<4, 1>(a, stream);
    case 5: return launch_group<5, 1>(a, stream);
    case 6: return launch_group<6, 1>(a, stream);
    case 7: return launch_group<7, 1>(a, stream);
    case 8: return launch_group<8, 1>(a, stream);
    default: return false;
  }
}

template <int RT>
static bool launch_attn_d(const AttnArgs& a, int dt, int grid_splits, int nw, hipStream_t stream) {
  switch (dt) {
    case 1: return launch_attn<1, RT>(a, grid_splits, nw, stream);
    case 2: return launch_attn<2, RT>(a, grid_splits, nw, stream);
    case 3: return launch_attn<3, RT>(a, grid_splits, nw, stream);
    case 4: return launch_attn<4, RT>(a, grid_splits, nw, stream);
    case 5: return launch_attn<5, RT>(a, grid_splits, nw, stream);
    case 6: return launch_attn<6, RT>(a, grid_splits, nw, stream);
    case 7: return launch_attn<7, RT>(a, grid_splits, nw, stream);
    case 8: return launch_attn<8, RT>(a, grid_splits, nw, stream);
    default: return false;
  }
}

// A wavefront owns row_tiles (1 or 2) tiles of 16 rows of one request: the rows from
// tile_row0[i] and, with two, the rows from tile_row1[i] (-1: none; a null tile_row1: the
// 16 rows after the first tile).  `waves` wavefronts share a split (at most 16; 8 with a
// head size above 64; 4 with two row tiles).  `grid_splits` is an upper bound on the
// splits of any tile and `max_splits` the number the scratch has room for (grid_splits <=
// max_splits).  part_o holds tiles * nkv * max_splits * 16 * row_tiles * d floats, part_ml
// tiles * nkv * max_splits * 16 * row_tiles * 2 (both may be null when max_splits is 1).
// tickets (may be null): tiles * nkv words that are zero between launches; with them and one row
// tile a wavefront, the workgroup that completes a tile's splits adds them itself (the words are
// zero again when the launch ends); without, a second kernel adds them.
// Launches that share scratch must not overlap.
// grouped != 0 (two row tiles, P >= 16, one split of whole keys, waves 1): the caller promises
// that the tiles come in groups of 4 of one request each, filled up with empty tiles
// (tile_row0 < 0, the request's own index in tile_req): a workgroup takes a group and loads
// every key and value of the request's kv head once for its 4 tiles.  grouped 2: two sets of 4
// wavefronts take the steps of the group's keys in turn.
TK_API int tk_paged_attention_mfma(const void* q, int q_stride, void* out, int out_stride,
                                       const void* kcache, const void* vcache,
                                       const int* block_table, int table_stride,
                                       const int* q_start, const int* kv_len,
                                       const int* tile_req, const int* tile_row0, const int* tile_row1,
                                       int n_tiles, int row_tiles, int nq, int nkv, int d, int P, int window,
                                       float scale, int split, int waves, int grid_splits, int max_splits,
                                       float* part_o, float* part_ml, unsigned* tickets, int grouped, int even, hipStream_t stream) {
  TK_REQUIRE(n_tiles >= 0 && nq > 0 && nkv > 0 && nq % nkv == 0, "attention_mfma: bad sizes tiles=%d nq=%d nkv=%d", n_tiles, nq, nkv);
  TK_REQUIRE(d % 16 == 0 && d >= 16 && d <= 128, "attention_mfma: head size %d is not a multiple of 16 up to 128", d);
  TK_REQUIRE(P >= 4 && (P & (P - 1)) == 0, "attention_mfma: page size %d is not a power of two from 4", P);
  TK_REQUIRE(scale > 0.f, "attention_mfma: the scale must be positive");
  TK_REQUIRE(row_tiles == 1 || row_tiles == 2, "attention_mfma: row_tiles %d outside 1..2", row_tiles);
  TK_REQUIRE(row_tiles == 2 || !tile_row1, "attention_mfma: second row tiles given with one row tile a wavefront");
  TK_REQUIRE(split > 0 && split % 32 == 0, "attention_mfma: split %d is not a multiple of 32", split);
  TK_REQUIRE(waves >= 1 && waves <= max_waves(d / 16, row_tiles) && split % (32 * waves) == 0,
             "attention_mfma: %d wavefronts (at most %d) do not cut a split of %d keys into multiples of 32", waves,
             max_waves(d / 16, row_tiles), split);
  TK_REQUIRE((size_t)waves * 16 * row_tiles * (d + 4) * sizeof(float) <= 160 * 1024 || waves == 1,
             "attention_mfma: %d wavefronts of head size %d do not fit the local memory", waves, d);
  TK_REQUIRE(grid_splits >= 1 && grid_splits <= max_splits && grid_splits < 65536, "attention_mfma: splits %d of %d", grid_splits, max_splits);
  TK_REQUIRE(max_splits == 1 || (part_o && part_ml), "attention_mfma: split tiles need scratch");
  TK_REQUIRE(q_stride >= nq * d && out_stride >= nq * d && q_stride % 8 == 0 && out_stride % 4 == 0,
             "attention_mfma: row strides %d/%d too short or unaligned", q_stride, out_stride);
  TK_REQUIRE(((uintptr_t)q & 15) == 0 && ((uintptr_t)kcache & 15) == 0 && ((uintptr_t)vcache & 7) == 0 && ((uintptr_t)out & 7) == 0,
             "attention_mfma: operands must be 16-byte aligned");
  TK_REQUIRE(nkv < 65536, "attention_mfma: too many kv heads");
  TK_REQUIRE(!grouped || (row_tiles == 2 && P >= 16 && waves == 1 && max_splits == 1 && grid_splits == 1 &&
                          n_tiles % GROUP_WAVES == 0),
             "attention_mfma: grouped tiles need two row tiles, pages of 16 keys or more, one wavefront a tile, one split, "
             "and a multiple of %d tiles (got %d)", GROUP_WAVES, n_tiles);
  TK_REQUIRE(grouped >= 0 && grouped <= 2, "attention_mfma: %d sets of wavefronts a group (1 or 2)", grouped);
  if (n_tiles == 0) return 0;
  AttnArgs a;
  a.q = (const bf16_t*)q; a.q_stride = q_stride; a.out = (bf16_t*)out; a.out_stride = out_stride;
  a.kcache = (const bf16_t*)kcache; a.vcache = (const bf16_t*)vcache;
  a.block_table = block_table; a.table_stride = table_stride; a.q_start = q_start; a.kv_len = kv_len;
  a.tile_req = tile_req; a.tile_row0 = tile_row0; a.tile_row1 = tile_row1; a.n_tiles = n_tiles;
  a.nq = nq; a.nkv = nkv; a.group = nq / nkv; a.P = P; a.window = window;
  a.p_shift = 0;
  while ((1 << a.p_shift) < P) ++a.p_shift;
  a.scale_log2 = scale * 1.4426950408889634f;
  a.split = split; a.even = even; a.max_splits = max_splits; a.part_o = part_o; a.part_ml = part_ml;
  a.tickets = (max_splits > 1 && row_tiles == 1) ? tickets : nullptr;
  const bool ok = grouped ? launch_group_d(a, d / 16, grouped, stream)
                          : (row_tiles == 1 ? launch_attn_d<1>(a, d / 16, grid_splits, waves, stream)
                                            : launch_attn_d<2>(a, d / 16, grid_splits, waves, stream));
  TK_REQUIRE(ok, "attention_mfma: no kernel for head size %d", d);
  TK_CHECK_LAUNCH("paged_attention_mfma");
  if (max_splits > 1 && a.tickets == nullptr) {
    const int rows = 16 * row_tiles;
    hipLaunchKernelGGL(attention_merge_kernel, dim3(n_tiles, nkv, rows / 4), dim3(256), 0, stream, a, d, row_tiles);
    TK_CHECK_LAUNCH("attention_merge");
  }
  return 0;
}
