"""How decoded tokens' keys are cut: whole steps of 32 keys a wavefront, no split below 128 keys, and what a mixed step cuts evenly."""

import pytest

from tokasaurus_amd.kernels import ops


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("bound", [1, 100, 128, 129, 1024, 2048, 4096, 100000])
@pytest.mark.parametrize("tiles", [1, 2, 5, 45, 512])
def test_splits_are_worth_handing_over(head_dim, bound, tiles):
    split, waves = ops.attention_split(bound, tiles, 8, head_dim)
    assert split % (32 * waves) == 0 and waves <= (16 if head_dim == 64 else 4)
    assert split >= min(bound, 128) and -(-bound // split) <= max(16, bound // 2048 + 1)
    if tiles == 1 and 1024 <= bound <= 4096:
        assert waves == 4 and -(-bound // split) in (8, 16)


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("lengths", [[1], [2000] * 45, [250 + 39 * i for i in range(45)], [8192] + [40] * 63, [100, 131072]])
def test_even_splits(head_dim, lengths):
    split, waves = ops.attention_even_split(lengths, 8, head_dim)
    whole = ops.attention_split(max(lengths), len(lengths), 8, head_dim)
    assert split % (32 * waves) == 0 and 1 <= waves <= ops.attention_max_waves(head_dim, 1)
    assert (split, waves) == whole or (512 <= split < whole[0] and waves == 4)


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("nkv", [1, 8])
@pytest.mark.parametrize("lengths", [[40] * 63 + [28000], [64] * 127 + [24000], [64] * 255 + [16000], [1] * 999 + [262143], [1] * 999 + [31000], [500] * 63 + [8000],
                                     [100] * 3 + [16000], [300] * 100 + [3000], [100, 131072]])
def test_even_splits_have_a_bounded_grid(head_dim, nkv, lengths):
    """A launch has a workgroup and partial results for every split of the longest request, times the requests: no more than a bound, or
    than the planned cut has."""
    count = lambda split: len(lengths) * nkv * -(-max(lengths) // split)  # noqa: E731
    split, _ = ops.attention_even_split(lengths, nkv, head_dim)
    planned, _ = ops.attention_split(max(lengths), len(lengths), nkv, head_dim)
    assert split <= planned and count(split) <= max(count(planned), ops.ATTENTION_EVEN_WORKGROUPS)


@pytest.mark.parametrize("head_dim", [64, 128])
def test_even_splits_where_they_are_ahead(head_dim):
    """Not where planned workgroups of rising lengths fill one round or several, nor where they are few."""
    even = lambda lengths: ops.attention_even_split(lengths, 8, head_dim) != ops.attention_split(max(lengths), len(lengths), 8, head_dim)  # noqa: E731
    for lengths in ([1000 + 466 * i for i in range(16)], [200 + 122 * i for i in range(32)], [100 + 9 * i for i in range(100)], [100] * 3 + [16000], [2000] * 60):
        assert not even(lengths)
    for lengths in ([1000] * 30 + [3000] * 2, [1500] * 20 + [6000] * 4, [90 + 17 * i for i in range(41)]):
        assert not even(lengths)
    for lengths in ([500] * 63 + [8000], [300] * 10 + [4000] * 2):
        assert even(lengths)
    for lengths in ([250 + 39 * i for i in range(45)], [1000 + 159 * i for i in range(45)], [500 + 64 * i for i in range(40)]):
        assert even(lengths) == (head_dim > 64)


@pytest.mark.parametrize("group,nkv,requests,keys,waves", [(8, 8, 1, 8192, 8), (5, 8, 4, 32768, 8), (7, 4, 1, 32768, 8), (8, 1, 16, 8192, 8), (4, 8, 1, 8192, 4), (4, 8, 16, 8192, 4),
                                                           (3, 8, 45, 2000, 4), (4, 8, 32, 4096, 8), (2, 4, 48, 8192, 8), (2, 4, 12, 32768, 8), (4, 8, 4, 16000, 8), (4, 8, 64, 8192, 8), (4, 8, 2, 131072, 8), (8, 8, 1, 1024, 4)])
def test_wavefronts_at_head_sizes_above_64(group, nkv, requests, keys, waves):
    """Eight a workgroup, but for few query heads a kv head where every workgroup has a compute unit to itself and short walks."""
    split, got = ops.attention_split(keys, requests, nkv, 128, group)
    assert got == waves and split % (32 * waves) == 0


@pytest.mark.parametrize("head_dim,tiles,nkv,waves,even", [(64, 64, 8, 8, True), (64, 32, 16, 8, True), (64, 48, 8, 8, False), (64, 61, 8, 8, True), (64, 64, 8, 4, False), (64, 64, 8, 16, False),
                                                           (128, 64, 8, 8, False)])
def test_even_parts_where_two_workgroups_of_eight_fill_a_unit(head_dim, tiles, nkv, waves, even):
    assert ops.attention_even_parts(4096, tiles, nkv, head_dim, waves) == even


@pytest.mark.parametrize("head_dim,nkv", [(32, 2), (64, 1), (64, 8), (128, 2), (128, 8)])
@pytest.mark.parametrize("bound", [1024, 1100, 2048, 4096, 8192])
def test_short_requests_are_summed_in_one_order(head_dim, nkv, bound):
    """Of a step of some requests and of the recorded step that they are padded to: those of up to 64 keys in parts of 32, or in one part."""
    def parts(n):
        split, waves = ops.attention_split(bound, n, nkv, head_dim, 4)
        even = ops.attention_even_parts(bound, n, nkv, head_dim, waves)
        assert not even or waves >= 2  # (64 keys among two and more: 32 each)
        return 32 if even else min(split // waves, 64)
    for n in range(1, 129):
        assert parts(n) == parts(ops.recorded_rows(n)), n
