// A block of few hundred rows in one call of the host: norm in front made, then the stacked q, k, v product with rotation and
// append, attention, output projection with residual sum and norm, gate and up, down projection with residual sum and the next
// block's norm.  No kernel of its own: the entry points below in the order, and on the buffers, that the parts would call them.
//
// An eager step of these rows is bound by the host's calls, not by the kernels: a prompt of 101 tokens of the 1B shape is 1.2 ms
// of kernels, and its five calls a layer from Python, each with its checks and its results' memory, were 1.68 ms.  Here a launch is
// 2 to 3 us and the layers of a step share the memory for what lies between two products.  Whole steps, us, part by part / in one call:
// 1B shape 17 tokens 1,695 / 1,012, 101 1,685 / 1,242, 300 2,219 / 1,908, 500 2,247 / 2,158, 800 3,004 / 2,990; 3B shape 100 tokens 2,777 /
// 2,716, 8B shape 100 tokens 4,870 / 4,782.
#include "calls.h"

#define BLOCK_LAUNCHES 4
enum { ROUTE_LIBRARY = -1, ROUTE_STREAMED = -2 };  // else the tile of tk_gemm_tiles_bf16

struct BlockAttention {  // one launch of the attention: its tiles, and how keys are cut among workgroups
  const int* tile_req;
  const int* tile_row0;
  const int* tile_row1;
  float* part_o;
  float* part_ml;
  unsigned* tickets;
  int n_tiles, row_tiles, split, waves, max_splits, grouped, even;
};

struct BlockCalls {
  int bytes;  // of this struct, as the caller knows it
  // the step's rows and the block's sizes (inner: of gate, and of up)
  int M, hidden, nq, nkv, d, P, window, inner;
  float scale;
  // entry points of the other libraries: rotation with append, residual sum with norm, the gated activation, the library's product
  decltype(&tk_rope_append) rope_append;
  decltype(&tk_add_rmsnorm) add_rmsnorm;
  decltype(&tk_swiglu) swiglu;
  decltype(&tk_gemm_library_bf16) library;
  void* workspace;
  size_t workspace_bytes;
  // what every layer of the step reads
  const int* positions;
  const int* token_req;
  const int* q_start;
  const int* kv_len;
  const float* cos_t;
  const float* sin_t;
  // products: cuts of K (0: a whole product and a pass behind it, by the route), and whether the normed rows are rounded once
  int qkv_cuts, out_cuts, down_cuts, qkv_route, out_route, gate_route, down_route, out_once, down_once;
  int launches;
  BlockAttention attention[BLOCK_LAUNCHES];
  // memory between the products, shared by the layers
  float* part;    // cuts' sums
  void* qkv;      // [M, nq d] split, else [M, (nq + 2 nkv) d]
  void* attended;  // [M, nq d]
  void* product;  // [M, hidden], where a pass of its own follows
  void* stream;   // [M, hidden] between the halves of the block
  void* normed;
  void* gate_up;  // [M, 2 inner], the library's product
  void* act;      // [M, inner]
  // the layer
  const void* x;       // [M, hidden]
  const void* x_normed;
  const void* w_qkv;
  const void* w_out;
  const void* w_gate_up;
  const void* w_down;
  const void* mid_w;
  const void* next_w;
  void* kcache;
  void* vcache;
  const int* block_table;
  void* stream_out;
  void* normed_out;
  int table_stride, mid_w_f32, next_w_f32;
  float mid_eps, next_eps;
  int failed_in;  // whose error text tells why: 0 this library, 1 that of the passes, 2 that of the library's product
};

static int product(BlockCalls& b, const void* x, int K, const void* w, int N, int route, void* out, hipStream_t stream) {
  b.failed_in = route >= 0 ? 0 : 2;
  return route >= 0 ? tk_gemm_tiles_bf16(x, K, w, out, N, b.M, N, K, 0, route, stream)
                    : b.library(x, K, w, K, out, N, b.M, N, K, 0, b.workspace, b.workspace_bytes, stream);
}

// a projection, the residual added, and the norm that follows
static int project(BlockCalls& b, const void* x, int K, const void* w, int cuts, int route, int once, const void* residual, const void* norm_w,
                   int norm_f32, float eps, void* stream_out, void* normed, hipStream_t stream) {
  if (cuts > 0) {
    b.failed_in = 0;
    return tk_split_linear_add_rmsnorm(x, K, w, b.part, b.M, b.hidden, K, cuts, residual, norm_w, norm_f32, stream_out, normed, eps, once, stream);
  }
  const int rc = product(b, x, K, w, b.hidden, route, b.product, stream);
  if (rc) return rc;
  b.failed_in = 1;
  return b.add_rmsnorm(TK_BF16, b.product, residual, norm_w, norm_f32, stream_out, normed, b.M, b.hidden, eps, stream);
}

TK_API int tk_block_calls(BlockCalls* given, hipStream_t stream) {
  TK_REQUIRE(given && given->bytes == (int)sizeof(BlockCalls), "block_calls: the caller's struct is not this library's (%d of %d bytes)",
             given ? given->bytes : 0, (int)sizeof(BlockCalls));
  BlockCalls& b = *given;
  b.failed_in = 0;
  TK_REQUIRE(b.M > 0 && b.hidden > 0 && b.inner > 0 && b.launches >= 0 && b.launches <= BLOCK_LAUNCHES, "block_calls: bad sizes M=%d hidden=%d inner=%d, %d launches",
             b.M, b.hidden, b.inner, b.launches);
  TK_REQUIRE(b.rope_append && b.add_rmsnorm && b.swiglu && b.library, "block_calls: an entry point is missing");
  const int heads = b.nq * b.d, width = (b.nq + 2 * b.nkv) * b.d;
  int rc;
  if (b.qkv_cuts > 0) {
    rc = tk_split_linear_rope_append(b.x_normed, b.hidden, b.w_qkv, b.part, b.M, b.hidden, b.qkv_cuts, b.qkv, b.positions, b.token_req, b.block_table,
                                     b.table_stride, b.cos_t, b.sin_t, b.kcache, b.vcache, b.nq, b.nkv, b.d, b.P, stream);
  } else {
    rc = product(b, b.x_normed, b.hidden, b.w_qkv, width, b.qkv_route, b.qkv, stream);
    if (rc) return rc;
    b.failed_in = 1;
    rc = b.rope_append(TK_BF16, b.qkv, width, b.positions, b.token_req, b.block_table, b.table_stride, b.cos_t, b.sin_t, b.kcache, b.vcache, b.M,
                       b.nq, b.nkv, b.d, b.d, b.P, 1, stream);
  }
  if (rc) return rc;
  b.failed_in = 0;
  for (int i = 0; i < b.launches; ++i) {
    const BlockAttention& l = b.attention[i];
    rc = tk_paged_attention_mfma(b.qkv, b.qkv_cuts > 0 ? heads : width, b.attended, heads, b.kcache, b.vcache, b.block_table, b.table_stride, b.q_start,
                                 b.kv_len, l.tile_req, l.tile_row0, l.tile_row1, l.n_tiles, l.row_tiles, b.nq, b.nkv, b.d, b.P, b.window, b.scale,
                                 l.split, l.waves, l.max_splits, l.max_splits, l.part_o, l.part_ml, l.tickets, l.grouped, l.even, stream);
    if (rc) return rc;
  }
  rc = project(b, b.attended, heads, b.w_out, b.out_cuts, b.out_route, b.out_once, b.x, b.mid_w, b.mid_w_f32, b.mid_eps, b.stream, b.normed, stream);
  if (rc) return rc;
  if (b.gate_route == ROUTE_LIBRARY) {
    rc = product(b, b.normed, b.hidden, b.w_gate_up, 2 * b.inner, ROUTE_LIBRARY, b.gate_up, stream);
    if (rc) return rc;
    b.failed_in = 1;
    rc = b.swiglu(TK_BF16, b.gate_up, b.act, b.M, b.inner, stream);
  } else {
    b.failed_in = 0;
    rc = b.gate_route == ROUTE_STREAMED ? tk_gemm_skinny_bf16(b.normed, b.hidden, b.w_gate_up, b.act, b.inner, nullptr, 0, nullptr, b.M, b.inner, b.hidden,
                                                              2 /* gate and up */, 0, 0, 2 /* streamed */, 0, 1, stream)
                                        : tk_gemm_tiles_bf16(b.normed, b.hidden, b.w_gate_up, b.act, b.inner, b.M, b.inner, b.hidden, 1, b.gate_route, stream);
  }
  if (rc) return rc;
  return project(b, b.act, b.inner, b.w_down, b.down_cuts, b.down_route, b.down_once, b.stream, b.next_w, b.next_w_f32, b.next_eps, b.stream_out,
                 b.normed_out, stream);
}
