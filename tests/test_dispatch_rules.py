"""Host-side rules that choose between kernels: no GPU needed."""

from tokasaurus_amd.kernels import ops


def test_rows_up_to_which_the_weight_streaming_product_is_taken():
    # the measured crossings at the 1B layer sizes: output projection about 40 rows, down
    # projection about 10, gate and up (two tiles meet in the epilogue) under 20
    assert ops.skinny_rows(2048) == 39 and ops.skinny_rows(8192) == 9 and ops.skinny_rows(2048, paired=True) == 19
    # wider models leave it earlier; tiny ones never (the kernel's own limit holds)
    assert ops.skinny_rows(4096) == 19 and ops.skinny_rows(14336) == 5 and ops.skinny_rows(4096, paired=True) == 9
    assert ops.skinny_rows(64) == ops.SKINNY_MAX_ROWS and ops.skinny_rows(10**9) == 1


def test_decode_attention_splits_fill_the_chip():
    # (keys a split, wavefronts a workgroup): about 256 workgroups, at most 16 splits, splits of whole 32-key steps a wavefront
    for tiles in (1, 2, 4, 8, 16, 64, 256):
        for bound in (1024, 8192, 131072):
            split, waves = ops.attention_split(bound, tiles, 8, 64)
            assert split % (32 * waves) == 0 and 1 <= waves <= 16
            splits = -(-bound // split)
            # few tiles: about 256 workgroups; many: splits of 8 192 keys at most (2 048 from a thousand tiles on)
            assert 1 <= splits <= 64 and (splits * tiles * 8 <= max(256, tiles * 8) * 2 or split == (8192 if tiles * 8 < 1024 else 2048))
    assert ops.attention_split(8192, 1, 8, 64) == (512, 8) and ops.attention_split(8192, 8, 8, 64) == (2048, 8)
    assert ops.attention_split(8192, 64, 8, 64) == (8192, 16)


def test_how_prompt_portions_are_cut_for_attention():
    # (wavefronts of two row tiles over all kv heads, keys of the longest request); the 1B and the 8B shape fill a wavefront
    # a token (8 kv heads of 4 query heads), the 3B shape three quarters of one
    sets = lambda prompts, tokens, d, per_token=1.0, over=None, page=16: ops.attention_group_sets(
        int(prompts * tokens * per_token), d, page, over or tokens)
    # one whole prompt, head size 64: paired tiles, from 2 048 tokens two sets, from 3 072 one
    assert [sets(1, n, 64) for n in (512, 1536, 2048, 2560, 3072, 8192)] == [0, 0, 2, 2, 1, 1]
    # several prompts: short walks keep paired tiles however many they are; longer ones take two sets
    assert [sets(b, n, 64) for b, n in ((2, 1024), (4, 512), (8, 512), (32, 256))] == [0, 0, 0, 0]
    assert [sets(b, n, 64) for b, n in ((4, 1024), (2, 1536), (2, 2048))] == [2, 2, 2]
    # portions after a long past: two sets even when few
    assert [sets(b, 256, 64, over=4096) for b in (1, 4, 8)] == [2, 2, 2] and sets(1, 2048, 64, over=8192) == 2
    assert sets(1, 1024, 64, over=2048) == 0 and sets(1, 128, 64, over=4096) == 0
    # head size 128: paired tiles run one wavefront a SIMD there, so groups are taken earlier
    assert [sets(1, n, 128) for n in (1024, 1536, 2048, 3072, 8192)] == [0, 2, 2, 1, 1]
    assert [sets(1, n, 128, per_token=0.75) for n in (1024, 2048, 3072, 4096)] == [0, 2, 2, 1]
    assert [sets(b, n, 128) for b, n in ((8, 256), (4, 512), (2, 1024), (8, 512))] == [1, 1, 2, 1]
    assert sets(2, 256, 128, over=4096) == 2 and sets(1, 1024, 128, over=2048) == 2 and sets(2, 512, 128, over=1024) == 0
    # pages of fewer than 16 keys: a 16-key block would span pages, which the grouped kernel does not take
    assert sets(1, 8192, 64, page=8) == 0 and sets(1, 8192, 128, page=4) == 0


def test_keys_of_short_portions_after_long_pasts_are_cut():
    split = ops.attention_prompt_split
    # (wavefronts, head size, keys of the longest request) -> keys a split: the walks fill 2 048 wavefronts' room
    # (1 024 at head sizes above 64), in splits of 512 keys at least and 64 splits at most
    assert split(64, 64, 32768) == 1024 and split(16, 64, 32768) == 512 and split(8, 64, 131072) == 2048
    assert split(256, 64, 4096) == 512 and split(512, 64, 8192) == 2048 and split(64, 64, 8192) == 512
    # two splits only for walks of 16 384 keys and more at head sizes up to 64; always at head sizes above
    assert split(1024, 64, 8192) == 0 and split(1024, 64, 32768) == 16384
    assert split(512, 128, 8192) == 4096 and split(1024, 128, 32768) == 0
    # whole prompts and portions after short pasts keep whole keys
    assert split(512, 64, 512) == 0 and split(256, 64, 300) == 0 and split(2048, 64, 32768) == 0 and split(8, 64, 500) == 0
    for w in (1, 8, 100, 700):
        for keys in (100, 1000, 5000, 200000):
            s = split(w, 64, keys)
            assert s == 0 or (s % 128 == 0 and 512 <= s < keys and -(-keys // s) <= 64)


def test_prompts_leave_the_split_attention_by_their_own_length():
    splits = ops.attention_tile_splits
    # 32 heads, tiles of 16 tokens: the step's own longest request decides, whatever the step is planned for
    assert not splits(512, True, 256, 256) and splits(480, True, 240, 240)
    assert splits(512, True, 256, 1024) and splits(512, True, 256, 0) and splits(512, False, 256, 256)
    assert not splits(2048, False, 64, 100_000)
    # heads wider than 128 are walked one block of keys a step
    assert splits(1023, True, 512, 512, widest=256) and not splits(1024, True, 512, 512, widest=256) and not splits(512, True, 512, 512, widest=128)
    # tokens of a section or behind a window see no more than it holds, however long the request
    assert not splits(512, True, 256, 5000, section=200) and not splits(512, True, 256, 5000, window=200)
    assert splits(512, True, 256, 5000, section=300) and splits(512, True, 256, 5000, window=300)


def test_chunks_of_split_attention_take_bounded_room_and_reach_every_key():
    words = 16 * 130
    for groups in (1, 8, 500, 2000, 70_000):
        for bound in (1024, 16384, 131072):
            for longest in (1, 255, 256, 257, 1000, bound):
                if longest > bound:
                    continue
                for reach in (0, 64, 300, 5000):
                    key_chunk, chunks = ops.attention_tile_chunks(groups, 256, bound, longest, reach, words)
                    whole, most = ops.attention_tile_chunks(groups, 256, bound, bound, reach, words)
                    # a chunk is as long as in a recorded step of this bound, whatever the step's own requests
                    assert key_chunk == whole and key_chunk % 256 == 0 and 1 <= chunks <= most
                    assert groups * most * words * 4 <= ops.ATTENTION_TILE_PART_BYTES or most == 1
                    # every tile's keys lie in its chunks: those of the tile that starts at any place of a chunk
                    seen = min(longest, reach + 15) if reach else longest
                    worst = (longest - 1) // key_chunk if not reach else min((longest - 1) // key_chunk, (key_chunk - 1 + seen - 1) // key_chunk)
                    assert chunks >= worst + 1
    # (32-bit prompts of 2,000 pairs in a step planned for 131,072 keys: one chunk where the requests are short)
    assert ops.attention_tile_chunks(2000, 256, 131072, 500, 0, words)[1] == 1


def test_which_portions_take_the_delta_rule_in_chunks():
    chunks = ops.delta_portions_in_chunks
    assert chunks([1]) == [False] and chunks([159]) == [False] and chunks([160]) == [True] and chunks([]) == []
    # single tokens and short portions keep the recurrence whatever shares their step; many portions count together
    assert chunks([300, 31, 1, 1]) == [True, False, False, False]
    assert chunks([48] * 8 + [1]) == [True] * 8 + [False] and chunks([32, 96, 31, 1]) == [False] * 4


def test_which_experts_products_run_in_tiles():
    import torch

    tiles = lambda rows, top, experts, ff=512: ops.experts_go_in_tiles(rows, top, torch.bfloat16, 1024, ff, experts)
    # from 64 pairs on, and five pairs for four experts, in steps of more than a dozen rows
    assert tiles(32, 2, 16) and not tiles(31, 2, 16) and not tiles(12, 8, 16)
    assert not tiles(32, 2, 64) and not tiles(39, 2, 64) and tiles(40, 2, 64)
    assert not tiles(39, 8, 256) and tiles(40, 8, 256)
    assert not tiles(64, 2, 16, ff=12)


def test_rows_that_gate_and_up_take_in_the_hand_written_product():
    # up to 64 where the streamed form is ahead: inner sizes up to 4,096, workgroups of 32 outputs in well filled rounds of 256
    assert [ops.glu_rows(2048, n) for n in (1000, 8192, 8224, 12288, 14336, 16416, 24576)] == [64, 64, 16, 16, 64, 16, 64]
    assert ops.glu_rows(4096, 14336) == 64 and ops.glu_rows(4096, 11008) == 16
    assert ops.glu_rows(5120, 13824) == ops.glu_rows(8192, 28672) == 16
    assert ops.glu_rows(2080, 8192) == ops.skinny_rows(2080, paired=True)


def test_32_bit_products_of_more_rows_than_a_grid_has_are_not_cut():
    # (the sums of K's parts are added by a grid with a row of workgroups a token; whole tiles of either kind take any number of rows)
    from tokasaurus_amd.kernels.library import load

    cuts = load("core").tk_gemm_f32_cuts
    for m in (65536, 65568, 65600, 67264, 71168, 76736, 131072, 1 << 20):
        for n in (16, 64, 128, 256, 1024, 1028, 4096):
            for k in (1024, 2048, 8192, 14336):
                assert cuts(m, n, k) == 1, (m, n, k)
    assert cuts(301, 2048, 8192) > 1 and cuts(301, 2050, 8192) == 1
