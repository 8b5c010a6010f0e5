"""A pre-norm block's kernels for a few hundred rows, launched by one call (csrc/block_calls.hip): what an eager step of a short
prompt waits for is the host, five calls a layer with their checks and their results' memory.

``BlockPlan`` is made once a step and shared by its layers: which products are split, tiled or the library's, the attention's
launches, and the memory for what lies between two products.  ``BlockPlan.run`` takes a layer's tensors; it refuses (None) what
the entry points read only where the general path knows a way round, and the caller goes that way.
"""

from __future__ import annotations

import ctypes
from ctypes import c_float, c_int, c_size_t, c_void_p

import torch

from tokasaurus_amd.kernels import ops
from tokasaurus_amd.kernels.library import KernelError, load

LAUNCHES = 4  # of the attention, at most
# Rows up to which a step's blocks are launched by one call.  Beyond, the kernels take several times what the host's calls do (1B shape
# at 1,024 rows 3.3 ms of kernels, 1.6 of calls).
MOST_ROWS = 1024


class _Attention(ctypes.Structure):
    _fields_ = [(n, c_void_p) for n in ("tile_req", "tile_row0", "tile_row1", "part_o", "part_ml", "tickets")] + [
        (n, c_int) for n in ("n_tiles", "row_tiles", "split", "waves", "max_splits", "grouped", "even")]


class _BlockCalls(ctypes.Structure):
    """struct BlockCalls of block_calls.hip."""

    _fields_ = (
        [(n, c_int) for n in ("bytes", "M", "hidden", "nq", "nkv", "d", "P", "window", "inner")] + [("scale", c_float)]
        + [(n, c_void_p) for n in ("rope_append", "add_rmsnorm", "swiglu", "library", "workspace")] + [("workspace_bytes", c_size_t)]
        + [(n, c_void_p) for n in ("positions", "token_req", "q_start", "kv_len", "cos_t", "sin_t")]
        + [(n, c_int) for n in ("qkv_cuts", "out_cuts", "down_cuts", "qkv_route", "out_route", "gate_route", "down_route", "out_once", "down_once",
                                "launches")]
        + [("attention", _Attention * LAUNCHES)]
        + [(n, c_void_p) for n in ("part", "qkv", "attended", "product", "stream", "normed", "gate_up", "act",
                                   "x", "x_normed", "w_qkv", "w_out", "w_gate_up", "w_down", "mid_w", "next_w", "kcache", "vcache", "block_table",
                                   "stream_out", "normed_out")]
        + [(n, c_int) for n in ("table_stride", "mid_w_f32", "next_w_f32")] + [("mid_eps", c_float), ("next_eps", c_float), ("failed_in", c_int)])


def _address(group: str, name: str) -> int:
    return ctypes.cast(getattr(load(group), name), c_void_p).value


class BlockPlan:
    """``routes``: of the q, k, v, the output, the gate and up and the down product (``Linear.many_rows_route``, ``Linear.gate_up_route``): (cuts of K or
    0, tile or -1 for the library, rounded once)."""

    def __init__(self, ctx, rows: int, hidden: int, inner: int, nq: int, nkv: int, head_dim: int, page_size: int, window: int, scale: float,
                 cos: torch.Tensor | None, sin: torch.Tensor | None, routes: dict[str, tuple], launches: list):
        m, heads, width = rows, nq * head_dim, (nq + 2 * nkv) * head_dim
        self.shape, self.page = (m, hidden), (nkv, page_size, head_dim)
        self.weights = {"w_qkv": (width, hidden), "w_out": (hidden, heads), "w_gate_up": (2 * inner, hidden), "w_down": (hidden, inner)}
        self.longest, self.requests = ctx.max_kv_len, ctx.num_requests
        b = self.calls = _BlockCalls()
        b.bytes, b.M, b.hidden, b.nq, b.nkv, b.d, b.P, b.window, b.inner, b.scale = (
            ctypes.sizeof(_BlockCalls), m, hidden, nq, nkv, head_dim, page_size, window, inner, scale)
        b.rope_append, b.add_rmsnorm, b.swiglu = (_address("core", n) for n in ("tk_rope_append", "tk_add_rmsnorm", "tk_swiglu"))
        b.library = _address("library", "tk_gemm_library_bf16")
        workspace = ops.library_workspace()
        b.workspace, b.workspace_bytes = workspace.data_ptr(), workspace.numel()
        tables = (ctx.positions, ctx.token_req, ctx.q_start, ctx.kv_len)
        b.positions, b.token_req, b.q_start, b.kv_len = (t.data_ptr() for t in tables)
        b.cos_t, b.sin_t = (cos.data_ptr(), sin.data_ptr()) if cos is not None else (None, None)
        for name in ("qkv", "out", "down"):
            cuts, route, once = routes[name]
            setattr(b, name + "_cuts", cuts)
            setattr(b, name + "_route", route)
            if name != "qkv":
                setattr(b, name + "_once", 1 if once else 0)
        b.gate_route = routes["gate"]
        b.launches = len(launches)
        # what the struct holds the addresses of (not the step itself, which holds this plan: a circle of references would keep the memory
        # until the collector comes by)
        self.kept = [*tables, cos, sin, workspace]
        for a, l in zip(b.attention, launches):
            n_tiles, splits = l.tile_req.numel(), max(1, -(-l.max_kv_len // l.split))
            a.tile_req, a.tile_row0 = l.tile_req.data_ptr(), l.tile_row0.data_ptr()
            a.tile_row1 = l.tile_row1.data_ptr() if l.tile_row1 is not None else None
            a.n_tiles, a.row_tiles, a.split, a.waves, a.max_splits, a.grouped, a.even = n_tiles, l.row_tiles, l.split, l.waves, splits, int(l.grouped), int(l.even)
            if splits > 1:
                in_kernel = l.row_tiles == 1 and ops.ATTENTION_MERGE_IN_KERNEL
                items = n_tiles * nkv * splits * 16 * l.row_tiles
                scratch = l.scratch if l.scratch is not None else ops.AttentionScratch.shared(ctx.device)
                part_o, part_ml = scratch.take(items * head_dim, items * 2, n_tiles * nkv if in_kernel else 0)
                a.part_o, a.part_ml, a.tickets = part_o.data_ptr(), part_ml.data_ptr(), scratch.tickets.data_ptr() if in_kernel else None
                self.kept += [part_o, part_ml, scratch.tickets]
            self.kept.append(l)
        # memory between the products, in pieces that start at multiples of 256 bytes
        part = max([cuts * n * 4 for (cuts, _, _), n in ((routes["qkv"], width), (routes["out"], hidden), (routes["down"], hidden))])
        sizes = {"part": part, "qkv": (heads if b.qkv_cuts else width) * 2, "attended": heads * 2,
                 "product": 0 if b.out_cuts and b.down_cuts else hidden * 2, "stream": hidden * 2, "normed": hidden * 2,
                 "gate_up": 4 * inner if b.gate_route == -1 else 0, "act": 2 * inner}
        places, at = {}, 0
        for name, a_row in sizes.items():
            places[name] = at
            at += -(-a_row * m // 256) * 256
        self.memory = torch.empty((at,), dtype=torch.uint8, device=ctx.device)
        base = self.memory.data_ptr()
        for name, place in places.items():
            setattr(b, name, base + place)
        self.aligned = (b.cos_t or 0) % 16 == 0 and (b.sin_t or 0) % 16 == 0 and base % 16 == 0

    def run(self, x: torch.Tensor, normed: torch.Tensor, weights: dict[str, torch.Tensor], mid_w: torch.Tensor, mid_eps: float, next_w: torch.Tensor,
            next_eps: float, kcache: torch.Tensor, vcache: torch.Tensor, block_table: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor] | None:
        """(the stream behind the block, its rows normed for the next one); None, and nothing done, where a tensor does not lie as the
        entry points read it."""
        b, device = self.calls, x.get_device()
        for t in (x, normed):
            if t.shape != self.shape or t.dtype != torch.bfloat16 or not t.is_contiguous() or t.get_device() != device:
                return None
        for name, w in weights.items():
            at = w.data_ptr()
            if w.shape != self.weights[name] or w.dtype != torch.bfloat16 or not w.is_contiguous() or w.get_device() != device or at % 16:
                return None
            setattr(b, name, at)
        for w in (mid_w, next_w):
            if (w.shape != self.shape[1:] or not w.is_contiguous() or w.get_device() != device
                    or not (w.dtype == torch.bfloat16 or w.dtype == torch.float32)):
                return None
        nkv, page_size, head_dim = self.page
        if not (block_table.dtype == torch.int32 and block_table.dim() == 2 and block_table.is_contiguous() and block_table.get_device() == device
                and block_table.shape[0] >= self.requests and block_table.shape[1] * page_size >= self.longest
                and kcache.get_device() == device and vcache.get_device() == device):
            return None
        ops._check_pages(kcache, vcache, nkv, page_size, head_dim, torch.bfloat16, "block_calls")
        b.x, b.x_normed, b.mid_w, b.next_w, b.kcache, b.vcache = (t.data_ptr() for t in (x, normed, mid_w, next_w, kcache, vcache))
        if (b.x | b.x_normed | b.mid_w | b.next_w | b.kcache | b.vcache) % 16 or not self.aligned:
            return None
        b.mid_w_f32, b.next_w_f32 = 1 if mid_w.dtype == torch.float32 else 0, 1 if next_w.dtype == torch.float32 else 0
        b.mid_eps, b.next_eps = mid_eps, next_eps
        b.block_table, b.table_stride = block_table.data_ptr(), block_table.stride(0)
        stream_out, normed_out = torch.empty_like(x), torch.empty_like(x)
        b.stream_out, b.normed_out = stream_out.data_ptr(), normed_out.data_ptr()
        lib = load("mfma")
        if lib.tk_block_calls(ctypes.byref(b), ops._stream()) != 0:
            raise KernelError((lib, load("core"), load("library"))[b.failed_in].tk_last_error().decode(errors="replace"))
        return stream_out, normed_out
