"""Which product a linear map takes and what the products' wrappers refuse, without a GPU: tensors that say they lie on one, and
recorders in the place of the kernels."""

from __future__ import annotations

import pytest
import torch

from tokasaurus_amd.kernels import ops
from tokasaurus_amd.parts.base import Normed, Prepared
from tokasaurus_amd.parts.linear import Linear
from tokasaurus_amd.parts.norm import RMSNorm


class OnGpu(torch.Tensor):
    is_cuda = True


def on_gpu(*shape, dtype=torch.bfloat16, device="cpu"):
    return torch.empty(shape, dtype=dtype, device=device).as_subclass(OnGpu)


@pytest.fixture
def calls(monkeypatch):
    """Names of the kernels that are called; none is."""
    made = []
    monkeypatch.setattr(ops, "call", lambda name, *a: made.append(name))
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    return made


def _rope(rows, nq=4, nkv=2, d=32, page=16):
    i32 = dict(dtype=torch.int32)
    return ops.RopeAppend(on_gpu(rows, **i32), on_gpu(rows, **i32), on_gpu(1, 4, **i32), on_gpu(64, d // 2, dtype=torch.float32),
                          on_gpu(64, d // 2, dtype=torch.float32), on_gpu(*ops.key_pages_shape(4, nkv, page, d)),
                          on_gpu(*ops.value_pages_shape(4, nkv, page, d)), nq, nkv, d, page)


@pytest.mark.parametrize("where", ["host", "another device"])
def test_a_weight_that_is_not_where_the_rows_are_is_refused(calls, where):
    x, residual, norm = on_gpu(33, 192), on_gpu(33, 256), on_gpu(256)
    ops.split_linear_add_rmsnorm(x, on_gpu(256, 192), residual, norm, 1e-5)
    ops.split_linear_rope_append(x, on_gpu(256, 192), _rope(33))
    ops.gemm_tiles_bf16(x, on_gpu(256, 192), 0)
    assert calls == ["tk_split_linear_add_rmsnorm", "tk_split_linear_rope_append", "tk_gemm_tiles_bf16"]
    w = torch.empty((256, 192), dtype=torch.bfloat16) if where == "host" else on_gpu(256, 192, device="meta")
    for refused in (lambda: ops.split_linear_add_rmsnorm(x, w, residual, norm, 1e-5), lambda: ops.split_linear_rope_append(x, w, _rope(33)),
                    lambda: ops.gemm_split(x, w), lambda: ops.gemm_tiles_bf16(x, w, 0)):
        with pytest.raises(ops.KernelError):
            refused()
    assert len(calls) == 3


def linear(outputs, inner):
    lin = Linear(inner, ["w"], [outputs])
    lin.weight = on_gpu(outputs, inner)
    return lin


def norm(size):
    n = RMSNorm(size, 1e-5, "n")
    n.weight = on_gpu(size)
    return n


def test_a_prepared_norm_is_folded_into_the_product_with_the_rotation(calls):
    """Rows that the weight-streaming product in front left for this norm: no pass of a norm's own, no second rounding."""
    lin, n = linear(3072, 2048), norm(2048)
    data = ops.Prenorm(on_gpu(16, 2048), on_gpu(16, 128, dtype=torch.float32))
    rope = _rope(16, 32, 8, 64)
    assert lin.rope_append(Normed(on_gpu(16, 2048), n, Prepared(data, n)), rope) is not None
    assert calls == ["tk_gemm_skinny_bf16"]
    calls.clear()
    assert lin.rope_append(Normed(on_gpu(16, 2048), n, Prepared(None, n, on_gpu(16, 2048))), rope) is not None
    assert calls == ["tk_split_linear_rope_append"]


def test_recorded_rows_are_those_that_decode_steps_are_padded_to():
    from tokasaurus_amd.engine.runner import graph_buckets

    sizes = graph_buckets(128, 16)
    assert [ops.recorded_rows(m) for m in range(1, 129)] == [min(s for s in sizes if s >= m) for m in range(1, 129)]


@pytest.mark.parametrize("outputs,inner", [(2048, 2048), (2048, 8192), (3072, 3072), (4096, 4096), (4096, 14336), (3072, 8192)])
def test_a_decode_step_takes_the_same_products_alone_and_padded(calls, monkeypatch, outputs, inner):
    """Among the engine's own products: where a count or the size it is padded to is the library's, nothing is asked."""
    def made(m):
        calls.clear()
        linear(outputs, inner).with_residual(on_gpu(m, inner), on_gpu(m, outputs), norm(outputs))
        linear(outputs, inner).rope_append(on_gpu(m, inner), _rope(m, outputs // 64 - 16, 8, 64))
        return list(calls)

    monkeypatch.setattr(ops, "load", lambda name: type("Lib", (), {"tk_gemm_skinny_parts": lambda self, *a: 4})())
    for m in range(1, 129):
        assert made(m) == made(ops.recorded_rows(m))
    assert made(2)[0] == "tk_gemm_skinny_bf16" and made(128) == ["tk_split_linear_add_rmsnorm", "tk_split_linear_rope_append"]


@pytest.mark.parametrize("field", ["cos", "sin", "kcache", "vcache"])
def test_tables_and_pages_that_start_anywhere_are_not_refused(calls, field):
    """16 rows go to the product that reads them one by one, 33 back to the caller, who rotates them one by one."""
    lin = linear(3072, 2048)
    for rows, aligned, moved in ((16, ["tk_split_linear_rope_append"], ["tk_gemm_skinny_bf16"]), (33, ["tk_split_linear_rope_append"], [])):
        for want in (aligned, moved):
            rope = _rope(rows, 32, 8, 64)
            if want is moved:
                old = getattr(rope, field)
                setattr(rope, field, on_gpu(old.numel() + 4, dtype=old.dtype)[1 : old.numel() + 1].view(old.shape))
            calls.clear()
            assert (lin.rope_append(on_gpu(rows, 2048), rope) is None) == (not want)
            assert calls == want


@pytest.mark.parametrize("m,n,k,shape", [
    (64, 8192, 2048, -1), (65, 8192, 2048, 5), (128, 8192, 2048, 5), (129, 8192, 2048, 0), (256, 8192, 2048, 0), (257, 8192, 2048, 1), (1024, 8192, 2048, 4),
    # more than one round: only whole ones, up to two of 192 x 256
    (1280, 8192, 2048, -1), (1408, 8192, 2048, 3), (1536, 8192, 2048, 3), (1664, 8192, 2048, -1), (2048, 8192, 2048, -1), (512, 14336, 4096, 4),
    (640, 14336, 4096, -1), (1024, 14336, 4096, -1),
    # up to 128 rows: two thirds of the units
    (128, 11008, 4096, 0), (128, 10240, 2560, -1), (129, 11008, 4096, -1), (128, 4096, 2048, -1), (200, 4096, 2048, -1)])
def test_which_tile_gate_and_up_take(m, n, k, shape):
    assert ops.tiles_choice(m, n, k, True) == shape
    assert ops.tiles_choice(m, n, k - 8, True) == -1


@pytest.mark.parametrize("m,n,k,shape", [(20, 28672, 4096, -1), (128, 32768, 1024, -1), (129, 32768, 1024, 1), (1280, 3072, 8192, 0), (1800, 2048, 192, 0),
                                         (1500, 2048, 8192, -1), (2048, 4096, 14336, 2), (2048, 4096, 4096, -1), (8192, 2048, 8192, -1)])
def test_which_tile_a_plain_product_takes(m, n, k, shape):
    assert ops.tiles_choice(m, n, k) == shape


@pytest.mark.parametrize("m", [1, 128, 129, 256])
def test_cuts_fill_the_compute_units(m):
    """The fewest cuts whose workgroups fill nine tenths of the 256 units' rounds, four steps of K each; else those that fill most."""
    for n in range(64, 16384, 192):
        for k in (64, 512, 2048, 8192, 14336):
            most = max(1, min(16, k // 256))
            groups = [-(-n // 64) * (2 if m > 128 else 1) * c for c in range(1, most + 1)]
            filled = [g / (-(-g // 256) * 256) for g in groups]
            enough = [c for c, f in enumerate(filled, 1) if f >= 0.9]
            assert ops.split_cuts(n, k, m) == (enough[0] if enough else 1 + filled.index(max(filled)))


def _taken(calls, lin, x, residual, n, rope):
    calls.clear()
    lin.with_residual(x, residual, n)
    lin.rope_append(x, rope)
    return list(calls)


def test_what_the_split_products_take(calls, monkeypatch):
    """Both sides of the thresholds of a weight of 2,048 x 2,048 (48,000 and 24,000 elements of x, counted at the recorded size), and
    calls that they do not take: with a bias, of rows that start anywhere, of weights below 2^20 elements, in 32-bit."""
    monkeypatch.setattr(ops, "load", lambda name: type("Lib", (), {"tk_gemm_skinny_parts": lambda self, *a: 4})())
    monkeypatch.setattr(ops, "library_workspace", lambda: on_gpu(16))
    monkeypatch.setattr(ops, "_gpu", lambda *tensors: None)  # (what a product leaves here does not say that it lies on one)
    n, skinny, split = norm(2048), "tk_gemm_skinny_bf16", ["tk_split_linear_add_rmsnorm", "tk_split_linear_rope_append"]
    library = ["tk_gemm_library_bf16", "tk_add_rmsnorm"]
    for m, want in ((8, [skinny, skinny]), (9, [skinny, split[1]]), (16, [skinny, split[1]]), (17, split), (64, split), (256, split), (257, library)):
        assert _taken(calls, linear(2048, 2048), on_gpu(m, 2048), on_gpu(m, 2048), n, _rope(m, 16, 8, 64)) == want, m
    biased = linear(2048, 2048)
    biased.bias = on_gpu(2048)
    assert _taken(calls, biased, on_gpu(24, 2048), on_gpu(24, 2048), n, _rope(24, 16, 8, 64)) == [skinny, skinny]
    small = linear(512, 2040)
    assert _taken(calls, small, on_gpu(36, 2040), on_gpu(36, 512), norm(512), _rope(36, 4, 2, 64)) == [skinny]
    shifted = on_gpu(200, 2056)[:, 4:2052]  # (the library's product is asked through the tensor library)
    monkeypatch.setattr(torch, "mm", lambda x, w: calls.append("mm") or on_gpu(x.shape[0], w.shape[1]))
    assert _taken(calls, linear(2048, 2048), shifted, on_gpu(200, 2048), n, _rope(200, 16, 8, 64)) == ["mm", "tk_add_rmsnorm"]
    wide = on_gpu(33, 2049)[:, 1:]  # a residual whose rows do not follow each other
    assert _taken(calls, linear(2048, 2048), on_gpu(33, 2048), wide, n, _rope(33, 16, 8, 64)) == [skinny, split[1]]


def test_rows_that_lie_too_far_apart_for_tiles_are_the_librarys_in_a_blocks_call_too():
    """The longest row that a tile's offsets reach, and the next size: as the product called by itself."""
    for inner, want in ((ops.TILES_LONGEST_STRIDE, 0), (ops.TILES_LONGEST_STRIDE + 64, -1)):
        assert ops.tiles_choice(1024, 4096, inner) == 0
        lin = Linear(inner, ["w"], [4096])
        lin.weight = torch.empty((4096, inner), dtype=torch.bfloat16, device="meta")
        assert lin.many_rows_route(1024, 1 << 30) == (0, want, False)
