// The entry points of paged attention in 32-bit arithmetic on the matrix cores (attention_tile_f32.h), and its kernels for
// 32-bit storage.
#include "attention_tile_f32.h"

void attention_tile_launch_f32(const AttentionTileCall& a) { at_launch_sizes<float>(a); }

// Whether this kernel takes the shape (else the caller uses the plain 32-bit kernel).
TK_API int tk_attention_tile_f32_fits(int nq, int nkv, int dk, int dv, int P) {
  return (nq > 0 && nkv > 0 && nq % nkv == 0 && dk > 0 && dk % 8 == 0 && dk <= 32 * AT_MAX_KM && dv > 0 && dv % 16 == 0 &&
          dv <= 16 * AT_MAX_VT && P > 0 && P % 16 == 0) ? 1 : 0;
}

// Whether the kernel can turn back the halves of a value head of dv elements itself: the two elements of a pair lie in
// one lane where the head fills the kernel's blocks of 16 (dv is 16 times 2, 4, 8 or 16).
TK_API int tk_attention_tile_turns_halves(int dv) { return (dv == 32 || dv == 64 || dv == 128 || dv == 256) ? 1 : 0; }

// 32-bit words of `part` that a (tile, head block, chunk) takes for a value head of dv elements
TK_API int tk_attention_tile_part_words(int dv) {
  return 32 + at_value_blocks(dv) * 4 * TK_WAVE;
}

// split: the wavefronts of a workgroup share a tile's keys (see the kernel); the caller chooses it for steps of few
// tiles.  It changes the order in which a token's keys are added up, nothing else.
TK_API int tk_attention_tile_f32(int dt, const void* q, int q_stride, void* out, int out_stride, const void* kcache,
                                 const void* vcache, const int* block_table, int table_stride, const int* q_start,
                                 const int* kv_len, const int* tile_req, const int* tile_row0, int n_tiles, int nq,
                                 int nkv, int dk, int dv, int P, int window, int section, float scale, const float* sink,
                                 const float* score_bias, int gg, int split, int chunk, int chunks, float* part,
                                 const float* vfreq, int v_pair_half, const void* gate, int gate_stride, float softcap,
                                 const int* bucket_of, int far, const float* rel, hipStream_t stream) {
  TK_REQUIRE(section <= 0 || window <= 0, "attention_tile_f32: a window or sections, not both");
  TK_REQUIRE(!rel || (bucket_of && far >= 0), "attention_tile_f32: a bias by distance needs its table of buckets");
  TK_REQUIRE(!(score_bias && (rel || softcap > 0.f)), "attention_tile_f32: sigmoid weights take neither a soft cap nor a bias by distance");
  const ScoreShape shape = {softcap, bucket_of, far, rel};
  TK_REQUIRE(tk_attention_tile_f32_fits(nq, nkv, dk, dv, P), "attention_tile_f32: shape nq=%d nkv=%d dk=%d dv=%d P=%d not taken",
             nq, nkv, dk, dv, P);
  const int group = nq / nkv;
  TK_REQUIRE(gg >= 1 && gg <= 16 && (gg & (gg - 1)) == 0 && group % gg == 0, "attention_tile_f32: %d heads a tile of a group of %d", gg, group);
  TK_REQUIRE(q_stride >= nq * dk && out_stride >= nq * dv, "attention_tile_f32: row strides too short");
  if (n_tiles <= 0) return 0;
  const int head_blocks = nkv * (group / gg);
  TK_REQUIRE(!vfreq || (dv % 2 == 0 && (!v_pair_half || tk_attention_tile_turns_halves(dv))),
             "attention_tile_f32: the halves of a value head of %d do not meet inside a lane", dv);
  TK_REQUIRE(!gate || gate_stride >= nq, "attention_tile_f32: gate rows of %d hold no %d heads", gate_stride, nq);
  const bool sp = split != 0;
  const bool parts = sp && chunk > 0;
  TK_REQUIRE(!parts || (chunk % 128 == 0 && chunks > 0 && chunks < 65536 && part), "attention_tile_f32: chunks of a multiple of 128 keys, "
             "their number and a place for their results");
  const dim3 grid(n_tiles, sp ? head_blocks : (head_blocks + AT_WAVES - 1) / AT_WAVES, parts ? chunks : 1);
  TK_REQUIRE(grid.y < 65536, "attention_tile_f32: too many heads");
  const AttentionTileCall call = {grid, sp, stream, q, q_stride, out, out_stride, kcache, vcache, block_table, table_stride, q_start, kv_len,
                                  tile_req, tile_row0, nq, nkv, dk, dv, P, window, section, scale, sink, score_bias, gg, parts ? chunk : 0,
                                  part, vfreq, v_pair_half, gate, gate_stride, shape};
  if (dt == TK_F32) attention_tile_launch_f32(call);
  else attention_tile_launch_bf16(call);
  TK_CHECK_LAUNCH("attention_tile_f32");
  return 0;
}
