"""The order in which prompts' groups of tiles start."""

import pytest
import torch

from tokasaurus_amd.kernels import ops


@pytest.mark.parametrize("q_lens,kv_lens,unit,form", [([1024, 1000, 1300], [1024, 1200, 1300], 4, 2), ([2048, 2048], [2048, 2100], 4, 2)])
def test_longest_walks_start_first(monkeypatch, q_lens, kv_lens, unit, form):
    """The plan's tiles are those of every portion, each once, in the order of the keys they reach."""
    from types import SimpleNamespace

    from tokasaurus_amd.parts import attention

    monkeypatch.setattr(attention, "upload", lambda values, dtype, device: torch.tensor(values, dtype=dtype))
    start = [sum(q_lens[:i]) for i in range(len(q_lens) + 1)]
    ctx = SimpleNamespace(extras={}, num_requests=len(q_lens), host_q_start=start, host_kv_len=kv_lens, max_kv_len=max(kv_lens), device=torch.device("cpu"))
    (launch,) = attention.attention_plan(ctx, 4, 8, 64, 16).launches
    req, row0 = launch.tile_req.tolist(), launch.tile_row0.tolist()
    assert launch.row_tiles == form and (launch.grouped > 0) == (unit == 4)
    fill = ops.ATTENTION_GROUP if unit == 4 else 1
    want = ops.attention_tiles(q_lens, 4, form, fill=fill)
    assert sorted(zip(req, row0)) == sorted(zip(want[0], want[1]))
    reach = [max(kv_lens[req[j]] - q_lens[req[j]] + row0[j] // 4 for j in range(i, i + unit)) for i in range(0, len(req), unit)]
    assert reach == sorted(reach, reverse=True)
    assert all(len(set(req[i : i + unit])) == 1 for i in range(0, len(req), unit))
