"""A linear map ``y = x W^T`` (``+ b`` when the checkpoint has a bias) with a fused
epilogue, the product every projection of the model goes through (``nn.Linear`` at
tokasaurus/model/llama.py:130-149,303-315,439; the reference's second architecture
gives q, k and v a bias, tokasaurus/model/qwen.py:11-25).  Several checkpoint tensors
may be stacked along the output rows into one product (q|k|v, gate|up).  The bias is added
to the 32-bit sums, before the product is rounded.

Which kernel runs is decided by the storage type and the number of rows:
  * float32: products and sums of all 24 bits (the true 32-bit path), on the matrix cores where the sizes fit them: 32-bit
    multiply-adds, or for many rows products of each number's three exact bfloat16 pieces with 32-bit sums, whose errors are not larger;
    up to 16 rows (``ops.gemm_f32_few``) with the activation, or the rotation and append, in the same kernel;
  * bfloat16, few rows (decode; how many depends on the inner size, ``ops.skinny_rows``, and ``ops.glu_rows`` for gate and
    up): the hand-written matrix-core kernels that stream the weight once and fuses the epilogue; it can also fold in the
    norm in front (``Normed`` input), leave what the norm behind it needs
    (``emit_norm``), and rotate and append q, k and v (``rope_append``);
  * bfloat16, up to 256 rows with the residual sum and norm or the rotation behind (from ``ops.split_from_rows`` on): K cut
    among workgroups, the cuts added by that pass (``ops.split_linear_add_rmsnorm``, ``ops.split_linear_rope_append``);
  * bfloat16, more rows (large decode batches, prefill): tiles of up to 256 x 256 where they are ahead
    (``ops.tiles_choice``; gate and up with the activation in the same kernel), else the library's matrix product,
    as in the reference (its projections are library calls), followed by the epilogue
    kernel; a bfloat16 weight whose inner size is no multiple of 8 takes the plain
    kernel for few rows.
"""

from __future__ import annotations

import torch

from tokasaurus_amd.kernels import ops
from tokasaurus_amd.parts.base import BIAS, MATRIX, Norm, Normed, Prepared, TensorSpec


class Placer:
    """Puts host tensors on the device once per (names, layout): tied tensors
    and shared tables end up in one buffer."""

    def __init__(self, dtype: torch.dtype, device: torch.device):
        self.dtype = dtype
        self.device = device
        self._placed: dict[tuple, torch.Tensor] = {}

    def place(self, key: tuple, make) -> torch.Tensor:
        if key not in self._placed:
            self._placed[key] = make()
        return self._placed[key]

    def bytes_placed(self) -> int:
        return sum(t.numel() * t.element_size() for t in self._placed.values())


class Linear:
    def __init__(self, in_features: int, names: list[str], out_features: list[int], bias_names: list[str | None] | None = None):
        """``bias_names``: for every stacked tensor the checkpoint name of its bias vector, or
        None for a part without one (its rows of the stacked bias are zero)."""
        assert len(names) == len(out_features)
        self.in_features = in_features
        self.names = list(names)
        self.out_features = list(out_features)
        self.total_out = sum(out_features)
        self.weight: torch.Tensor | None = None
        self.bias_names = list(bias_names) if bias_names and any(bias_names) else None
        assert self.bias_names is None or len(self.bias_names) == len(names)
        self.bias: torch.Tensor | None = None
        # rows from which the split product is taken (counted once: few calls of a step reach them)
        self.split_norm_from = ops.split_from_rows(in_features, self.total_out, ops.SPLIT_NORM_ELEMENTS)
        self.split_rope_from = ops.split_from_rows(in_features, self.total_out, ops.SPLIT_ROPE_ELEMENTS)
        # rows, or as many as they are padded to, that the weight-streaming product would take: rounded once where they are split
        self.split_once_to = ops.recorded_rows(ops.skinny_rows(in_features))

    def tensor_specs(self) -> list[TensorSpec]:
        specs = [TensorSpec(n, (o, self.in_features), MATRIX) for n, o in zip(self.names, self.out_features)]
        for b, o in zip(self.bias_names or [], self.out_features):
            if b is not None:
                specs.append(TensorSpec(b, (o,), BIAS))
        return specs

    def load(self, tensors: dict[str, torch.Tensor], placer: Placer) -> None:
        def make() -> torch.Tensor:
            parts = [tensors[n] for n in self.names]
            w = parts[0] if len(parts) == 1 else torch.cat(parts, dim=0)
            return w.to(dtype=placer.dtype).contiguous().to(placer.device)

        self.weight = placer.place(("row_major", *self.names), make)
        if self.bias_names is not None:
            def make_bias() -> torch.Tensor:
                where = next(tensors[b].device for b in self.bias_names if b is not None)
                parts = [tensors[b].to(placer.dtype) if b is not None else torch.zeros((o,), dtype=placer.dtype, device=where)
                         for b, o in zip(self.bias_names, self.out_features)]
                return torch.cat(parts).contiguous().to(placer.device)

            self.bias = placer.place(("bias", *[b or "" for b in self.bias_names], *self.names), make_bias)

    def _aligned(self) -> bool:
        # the bfloat16 matrix-core kernels read 8 inputs (16 bytes) at a time
        return self.weight.shape[1] % 8 == 0

    def _fast(self, m: int, paired: bool = False, out_f32: bool = False) -> bool:
        """Whether ``m`` rows take the weight-streaming kernels: up to a number of rows that
        depends on the inner size (``ops.skinny_rows``; gate and up: ``ops.glu_rows``); a
        32-bit result (the head) up to ``ops.SKINNY_ROWS``."""
        if self.weight.dtype != torch.bfloat16 or not 0 < m <= ops.SKINNY_MAX_ROWS or not self._aligned():
            return False
        if out_f32:
            return m <= ops.SKINNY_ROWS
        return (m <= ops.skinny_rows(self.in_features, paired)
                or (paired and m <= ops.GLU_STREAM_ROWS and m <= ops.glu_rows(self.in_features, self.total_out // 2)))

    def many_rows_route(self, m: int, split_from: int) -> "tuple[int, int, bool] | None":
        """How ``m`` rows go through this product with a pass behind it: (cuts of K, or 0 for a whole product; its tile, or -1 for the
        library's; whether the rows that the pass norms are rounded once); None where a kernel for few rows takes them, or another
        path.  ``split_from``: the rows from which that pass has the product split."""
        if self.weight.dtype != torch.bfloat16 or self.bias is not None or self.in_features % 8 or self.total_out % 8:
            return None
        if split_from <= m <= ops.SPLIT_ROWS:
            return ops.split_cuts(self.total_out, self.in_features, m), -1, m <= self.split_once_to
        if self._fast(m):
            return None
        tiles = m >= ops.PLAIN_TILES_FROM_ROWS and self.in_features <= ops.TILES_LONGEST_STRIDE
        return 0, ops.tiles_choice(m, self.total_out, self.in_features) if tiles else -1, False

    def gate_up_route(self, m: int) -> "int | None":
        """The same for gate and up with silu behind: a tile, -1 for the library's product, -2 for the streamed form."""
        inner = self.total_out // 2
        if self.weight.dtype != torch.bfloat16 or self.bias is not None or self.in_features % 8 or inner % 8:
            return None
        if self._fast(m, paired=True):
            return -2 if ops.glu_streams(m, inner, self.in_features) else None
        tiles = m >= ops.GLU_TILES_FROM_ROWS and self.in_features <= ops.TILES_LONGEST_STRIDE
        return ops.tiles_choice(m, inner, self.in_features, True) if tiles else -1

    def __call__(
        self,
        x: torch.Tensor | Normed,
        residual: torch.Tensor | None = None,
        out_f32: bool = False,
        rows: int | None = None,
        swiglu: bool = False,
        out: torch.Tensor | None = None,
        glu: "tuple[float, float] | str | None" = None,
        out_scale: float | None = None,
    ) -> torch.Tensor:
        """x [M, in] -> [M, out].  ``residual``: returns residual + product (the
        product rounded to the storage type first).  ``out_f32``: 32-bit output.
        ``swiglu``: the weight is [gate | up]; returns silu(gate) * up.
        ``rows`` limits the product to the first output rows of the stacked
        weight (a mixer that only needs its queries).  ``x`` may be a ``Normed``:
        the norm is folded into the product when it was prepared, else applied first.
        ``out`` (with ``out_f32``): a buffer [M, out] for the result, in place of new memory.
        ``glu`` (with ``swiglu``): (limit, alpha) of the gated activation with clamps, or "gelu_tanh" for gelu(gate) * up
        with the tanh form of gelu, in place of silu(gate) * up.
        ``out_scale`` (with ``out_f32``): the 32-bit result times this factor (in the few-row product's epilogue, else by a
        pass of its own)."""
        assert out_scale is None or (out_f32 and residual is None), "a factor on the result goes with 32-bit output"
        scaled = (lambda p: ops.scale_(p, out_scale)) if out_scale is not None and float(out_scale) != 1.0 else (lambda p: p)
        gated = ops.gelu_glu if glu == "gelu_tanh" else ((lambda p: ops.clamped_glu(p, glu[0], glu[1])) if glu is not None else ops.swiglu)
        assert out is None or (out_f32 and residual is None and not swiglu), "a result buffer goes with 32-bit output only"
        w, bias = self.weight, self.bias
        if rows is not None and rows != self.total_out:
            w = w[:rows]
            bias = bias[:rows] if bias is not None else None
        prenorm, eps = None, 0.0
        if isinstance(x, Normed):
            prepared = x.usable() if (self._fast(x.x.shape[0], swiglu, out_f32) and residual is None) else None
            if prepared is not None:
                prenorm, eps, x = prepared.data, x.norm.eps, prepared.data.scaled
            else:
                x = x.materialize()
        m = x.shape[0]
        if w.dtype == torch.bfloat16 and m > 0 and (m > ops.SKINNY_ROWS or self._aligned()):
            # (more rows than the weight-streaming product's may lie anywhere: where the streamed gate and up cannot read them,
            # the library's product does)
            if self._fast(m, swiglu, out_f32) and (not swiglu or ops.rows_at_16_bytes(x) or m <= ops.skinny_rows(self.in_features, paired=True)):
                return ops.gemm_skinny_bf16(x, w, residual=residual, out_f32=out_f32, swiglu=swiglu,
                                            prenorm=prenorm, norm_eps=eps, out=out, bias=bias, glu=glu if swiglu else None,
                                            out_scale=out_scale)
            # many rows: in tiles where these are ahead of the library's product (the gated form with silu in one kernel)
            direct = ops.gemm_library_direct(x, w)
            if (m >= (ops.GLU_TILES_FROM_ROWS if swiglu else ops.PLAIN_TILES_FROM_ROWS) and not out_f32 and bias is None and direct
                    and (glu is None or not swiglu)):
                shape = ops.tiles_choice(m, w.shape[0] // 2 if swiglu else w.shape[0], self.in_features, swiglu)
                if shape >= 0 and x.stride(0) <= ops.TILES_LONGEST_STRIDE:
                    prod = ops.gemm_tiles_bf16(x, w, shape, swiglu)
                    return ops.add(prod, residual.contiguous()) if residual is not None else prod
            # library matrix product (hipBLASLt), 32-bit accumulation; with a bias through the tensor
            # library, whose call adds it to the 32-bit sums in the product's own epilogue (addmm)
            if out_f32:
                if direct:
                    prod = ops.gemm_library_bf16(x, w, out_f32=True, out=out)
                else:
                    prod = (torch.mm(x, w.t(), out_dtype=torch.float32, out=out) if out is not None
                            else torch.mm(x, w.t(), out_dtype=torch.float32))
                return scaled(ops.add_bias(prod, bias) if bias is not None else prod)
            if bias is not None:
                prod = torch.addmm(bias, x, w.t())
            else:
                prod = ops.gemm_library_bf16(x, w) if direct else torch.mm(x, w.t())
            if residual is not None:
                # the product is rounded to the storage type before the residual is added, as in the
                # few-row kernel and in the pass that adds and norms (and as the reference's separate add)
                return ops.add(prod, residual.contiguous())
            return gated(prod) if swiglu else prod
        if swiglu and glu is None and residual is None and not out_f32 and w.shape[0] % 2 == 0 and ops.few_f32_takes(x, w):
            return ops.gemm_f32_few(x, w, bias)  # few 32-bit rows: the activation is part of the product's kernel
        # the 32-bit path, and few bfloat16 rows of a width the matrix-core kernel does not take
        prod = ops.gemm_generic(x, w, residual=residual, out_f32=out_f32, out=out, bias=bias)
        return gated(prod) if swiglu else scaled(prod)

    def with_residual(
        self, x: torch.Tensor, residual: torch.Tensor, emit_norm: Norm | None
    ) -> tuple[torch.Tensor, Prepared | None]:
        """residual + product and, where the kernel can, what ``emit_norm`` (the norm
        that will be applied to the result) needs so that it costs no kernel of its own."""
        m = x.shape[0]
        fusable = emit_norm is not None and getattr(emit_norm, "fusable_rms", False)
        if (fusable and self.split_norm_from <= m <= ops.SPLIT_ROWS and self.bias is None and ops.split_takes(x, self.weight)
                and residual.is_contiguous() and ops.split_norm_takes(residual, emit_norm.weight)):
            # (few rows: the next product's operand is rounded once, as where the weight-streaming product emits it)
            out, normed = ops.split_linear_add_rmsnorm(x, self.weight, residual, emit_norm.weight, emit_norm.eps, m <= self.split_once_to)
            return out, Prepared(None, emit_norm, normed)
        if fusable and self._fast(m):
            out, data = ops.gemm_skinny_bf16(x, self.weight, residual=residual, emit_weight=emit_norm.weight, bias=self.bias)
            return out, Prepared(data, emit_norm)
        if fusable and m > 0:
            # one pass adds the residual and norms the sum
            out, normed = ops.add_rmsnorm(self(x), residual.contiguous(), emit_norm.weight, emit_norm.eps)
            return out, Prepared(None, emit_norm, normed)
        return self(x, residual=residual), None

    def rope_append(self, x: torch.Tensor | Normed, rope: "ops.RopeAppend") -> torch.Tensor | None:
        """For a stacked [q | k | v] weight: the product with the rotation of q and k and the
        append of k and v to the pages in its epilogue; returns q [M, nq*d], or None when
        that kernel does not take this case (the caller then does the steps one by one)."""
        stream = x.x if isinstance(x, Normed) else x
        m = stream.shape[0]
        # (a norm that the product in front prepared is folded in below: its rows are not made for the split form)
        if (self.split_rope_from <= m <= ops.SPLIT_ROWS and self.bias is None and stream.dtype == torch.bfloat16 and rope.head_dim % 8 == 0
                and (rope.rotary_dim is None or rope.rotary_dim == rope.head_dim) and not (isinstance(x, Normed) and x.usable())):
            rows = x.materialize() if isinstance(x, Normed) else x
            q = ops.split_linear_rope_append(rows, self.weight, rope) if ops.split_takes(rows, self.weight) else None
            if q is not None:
                return q
            x = rows
        if self.weight.dtype == torch.float32:
            if not (0 < m <= ops.FEW_F32_ROWS and ops.few_f32_ropes(rope)):
                return None
            x = x.materialize() if isinstance(x, Normed) else x
            return ops.gemm_f32_few(x, self.weight, self.bias, rope) if ops.few_f32_takes(x, self.weight) else None
        most = min(ops.SKINNY_ROPE_ROWS, 2 * ops.skinny_rows(self.in_features, paired=True))
        fits = self.weight.dtype == torch.bfloat16 and 0 < m <= most and self._aligned()
        if not fits or rope.head_dim % 2 or (rope.rotary_dim is not None and rope.rotary_dim != rope.head_dim):
            return None
        prenorm, eps = None, 0.0
        if isinstance(x, Normed):
            prepared = x.usable()
            if prepared is not None:
                prenorm, eps, x = prepared.data, x.norm.eps, prepared.data.scaled
            else:
                x = x.materialize()
        return ops.gemm_skinny_bf16(x, self.weight, rope=rope, prenorm=prenorm, norm_eps=eps, bias=self.bias)
