"""The host-side choices of the attention kernels' shapes: pure functions of
the step's sizes, checked for their invariants (what a kernel's launch
assumes) and for the measured cases their docstrings name."""

import pytest
import torch

from nnis_amd.kernels.ops import PREFILL_CLASS_LENGTH, chain_plan, decode_plan, prefill_plan_class, prefill_tile_items


@pytest.mark.parametrize("batch", [1, 2, 8, 33, 64, 256])
@pytest.mark.parametrize("kv_heads", [1, 3, 8, 32])
@pytest.mark.parametrize("longest", [1, 63, 64, 65, 600, 1100, 2048, 8191])
@pytest.mark.parametrize("width", [0, 576, 2048, 4096])
def test_decode_plan_invariants(batch, kv_heads, longest, width):
    splits, waves = decode_plan(batch, kv_heads, longest, max_waves=4, width=width)
    pages = (longest + 63) // 64
    for n in (splits, waves):
        assert n >= 1 and n & (n - 1) == 0  # powers of two
    assert waves <= 4 and waves <= max(1, pages)  # no wave without a page
    assert splits <= 8
    if pages <= 8:
        assert splits == 1  # short sequences are never cut into runs
    if splits > 1:
        assert batch * kv_heads * waves * splits <= 2048  # runs only while the chip has room for their blocks
    assert decode_plan(batch, kv_heads, longest, max_waves=1, width=width)[1] == 1


def test_decode_plan_measured_cases():
    assert decode_plan(8, 3, 2048, width=576) == (8, 4)      # a narrow model: a page or two a wave
    assert decode_plan(64, 3, 2048, width=576) == (1, 4)     # no room for runs
    assert decode_plan(16, 32, 2048, width=2048) == (1, 4)
    assert decode_plan(64, 32, 2048, width=2048) == (1, 2)   # four and more blocks a compute unit: two waves a block
    assert decode_plan(8, 3, 64, width=576) == (1, 1)


def test_prefill_plan_class_and_work_lists():
    assert [prefill_plan_class(n) for n in (1, 127, 128, 511, 512, 1023, 1024, 1279, 1280, 5000)] == [0, 0, 1, 1, 2, 2, 3, 3, 4, 4]
    for plan_class, least in enumerate(PREFILL_CLASS_LENGTH):
        assert prefill_plan_class(least) == plan_class
    # every row of every sequence lies in exactly one tile; longest tiles (by the keys they read) first
    counts, first = [37, 5, 70, 1], [0, 100, 3, 64]
    for rows in (16, 32, 64):
        seqs, row0s = prefill_tile_items(counts, first, rows)
        seen = sorted((s, r) for s, r in zip(seqs, row0s))
        assert seen == sorted((s, r) for s, n in enumerate(counts) for r in range(0, n, rows))
        ends = [first[s] + min(r + rows, counts[s]) for s, r in zip(seqs, row0s)]
        assert ends == sorted(ends, reverse=True)


def test_prefill_plan_by_class_and_size():
    from nnis_amd.engine.graph import prompt_rows as prefill_rows
    from nnis_amd.kernels import ops

    def prefill_plan(longest, rows, *sizes):
        return ops.prefill_plan(longest, prefill_rows(rows), *sizes)  # (the engine plans for a step's rows rounded up)

    assert [prefill_rows(n) for n in (1, 64, 65, 1024, 1025, 2048, 2049, 4000)] == [64, 64, 128, 1024, 1152, 2048, 2304, 4096]
    for n in (1, 64, 100, 1000, 1100, 2000, 3000):
        assert prefill_rows(prefill_rows(n)) == prefill_rows(n)  # a step replayed from a graph's rows plans as the step launched
    assert prefill_plan(100, 100, 9) == prefill_plan(100, 100, 9, 64, 9) == (1, 1)  # (short prompts: items of one column, however the key heads are given)
    assert prefill_plan(300, 300, 9) == (2, 1)
    assert prefill_plan(700, 700, 9) == (4, 2)
    assert prefill_plan(1024, 1024, 32) == (4, 2) and prefill_plan(1024, 1024, 9) == (8, 0)
    assert prefill_plan(1024, 1900, 32) == (4, 2) and prefill_plan(1024, 2000, 33, 64, 11) == (8, 0)  # items enough: the widest tiles
    assert prefill_plan(600, 4000, 36, 64, 12) == (4, 0)
    assert prefill_plan(2048, 2048, 9) == (8, 0) and prefill_plan(1300, 1300, 32) == (4, 0)
    assert prefill_plan(2048, 2048, 16) == (8, 0)  # few items of four columns: 8 waves deal an item's keys
    # items for twice the chip's waves: one wave an item (64 rows x heads an item up to 64 channels, 32 up to 128)
    assert prefill_plan(8192, 8192, 32) == (1, 0) and prefill_plan(8192, 8192, 9, 64, 3) == (8, 0)
    # half of that: one wave an item of two columns, where two divide the group
    assert prefill_plan(4096, 4096, 32) == (1, 2) and prefill_plan(2048, 2048, 64, 64, 8) == (1, 2) and prefill_plan(4096, 4096, 36, 64, 12) == (8, 0)
    assert prefill_plan(2048, 2048, 32) == (4, 0)
    assert prefill_plan(4096, 4096, 32, 128) == (1, 0) and prefill_plan(2048, 2048, 32, 128) == (8, 0) and prefill_plan(2048, 2048, 16, 128) == (8, 0)
    assert prefill_plan(600, 34000, 32) == (1, 0) and prefill_plan(1024, 1024, 32, 256) == (1, 0) and prefill_plan(1024, 1024, 32, 128) == (4, 2)
    # a group of 3 heads: items of three columns (no two-column plans), one wave an item from twice the chip's waves of them
    assert prefill_plan(8192, 8192, 24, 64, 8) == (1, 0) and prefill_plan(1216, 1216, 24, 64, 8) == (4, 0)
    assert prefill_plan(3072, 3072, 32, 64, 32) == (4, 0)


@pytest.mark.parametrize("delta, least", [(True, {1: 128, 4: 320, 16: 1280}), (False, {1: 64, 4: 128, 16: 768})])
def test_a_step_launched_and_replayed_takes_one_form_of_the_matrix_recurrences(delta, least):
    """Chunks or a token at a time by the rows that a step plans for (64 and more, ``prompt_rows``): the same at the tokens that are
    launched and at the rows that are replayed, and scratch for no more rows than are there."""
    import types

    from nnis_amd.engine.graph import prompt_rows
    from nnis_amd.kernels import ops

    def scratch(batch, tokens, planned, decode=False, heads=4, longest=1279):
        ctx = types.SimpleNamespace(decode=decode, batch=batch, planned_rows=planned, planned_new=longest)
        return ops.chunked_scratch(ctx, tokens, heads, 64, 128, delta, "meta")

    for batch, first in least.items():
        for total in [batch, batch + 1, 63, 65, 100, 103, 104, first - 128, first - 64, first - 63, first - 1, first, first + 1, 4 * first]:
            if total < batch:
                continue
            rows = prompt_rows(total)
            longest = -(-rows // batch)
            launched, replayed = scratch(batch, total, rows, longest=longest), scratch(batch, rows, rows, longest=longest)
            assert (launched is not None) == (replayed is not None) == (rows >= first), (batch, total)
            if launched is not None:
                assert launched.numel() == ops.recurrent().nnis_chunked_scratch(total, batch, 4, 64, 128, int(delta)) <= replayed.numel()
    # whether there is memory enough goes by the planned rows too
    heads = ops.CHUNKED_MOST_BYTES // (4 * ops.recurrent().nnis_chunked_scratch(1280, 1, 1, 64, 128, int(delta)))
    assert scratch(1, 1279, 1280, heads=heads) is not None and scratch(1, 1280, 1280, heads=heads) is not None
    assert scratch(1, 1279, 1280, heads=heads + 1) is None and scratch(1, 1280, 1280, heads=heads + 1) is None
    assert scratch(8, 8, 4096, decode=True) is None  # single tokens


@pytest.mark.parametrize("heads, key_dim, value_dim, sequences, tokens, chunks", [
    (16, 128, 128, 1, 128, True), (16, 128, 128, 1, 1500, True), (16, 128, 128, 8, 2048, True), (16, 128, 128, 64, 300, True),  # 59 / 42, 602 / 135, 1,500 / 1,020, 1,788 / 1,646
    (16, 128, 128, 16, 101, False), (16, 128, 128, 32, 200, False), (16, 128, 128, 64, 170, False),  # 164 / 191, 575 / 659, 978 / 1,142
    (16, 64, 64, 64, 200, False), (8, 64, 128, 64, 170, False), (8, 32, 64, 64, 180, False), (8, 64, 128, 32, 200, False),  # 270 / 524, 219 / 345, 108 / 201, 140 / 196
    (8, 64, 128, 4, 120, True), (4, 32, 32, 16, 170, True), (4, 64, 64, 1, 64, False)])  # 52 / 34, 65 / 37; a chunk may hold two tokens
def test_the_delta_rule_goes_in_chunks_where_that_is_faster(heads, key_dim, value_dim, sequences, tokens, chunks):
    """Measured steps, microseconds a token at a time / in chunks: many walks fill the chip a token at a time."""
    import types

    from nnis_amd.kernels import ops

    ctx = types.SimpleNamespace(decode=False, batch=sequences, planned_rows=sequences * tokens, planned_new=tokens)
    assert (ops.chunked_scratch(ctx, sequences * tokens, heads, key_dim, value_dim, True, "meta") is not None) == chunks


@pytest.mark.parametrize("delta, heads, key_dim, value_dim, lengths, chunks", [
    (True, 16, 128, 128, [1500] + [100] * 15, True), (True, 16, 128, 128, [1500] + [16] * 15, True),  # 658 / 288, 608 / 225
    (True, 16, 128, 128, [700] + [30] * 15, True), (True, 8, 64, 128, [700] + [30] * 15, True),  # 305 / 178, 264 / 68
    (True, 16, 128, 128, [1500] + [16] * 63, False), (True, 16, 64, 64, [135] + [6] * 13, False),  # 635 / 687, 57 / 64
    (False, 8, 128, 256, [400] + [16] * 15, True), (False, 8, 128, 256, [1500] + [16] * 63, True),  # 136 / 61, 968 / 244
    (False, 8, 128, 256, [33] + [4] * 15, False), (False, 8, 128, 256, [47] + [10] * 15, False)])  # 38 / 51, 50 / 52
def test_matrix_recurrences_of_unequal_sequences_go_by_the_longest(delta, heads, key_dim, value_dim, lengths, chunks):
    """Measured steps, microseconds a token at a time / in chunks: a step lasts as long as its longest sequence's walk."""
    from nnis_amd.engine.graph import prompt_rows
    from nnis_amd.kernels import ops

    assert ops.chunks_pay(delta, len(lengths), prompt_rows(sum(lengths)), max(lengths), heads, key_dim, value_dim) == chunks


def test_32_bit_attention_of_small_heads():
    """One block for single tokens of small heads over few keys, and the row kernel for few rows of them, as measured."""
    from nnis_amd.kernels import ops

    for size, keys, splits in ((16, 100, 1), (32, 256, 1), (32, 320, 5), (16, 2048, 16), (48, 100, 2), (64, 1024, 16)):
        assert ops.attention_f32_splits(1, 9, 3, 0, keys, size) == splits
        assert ops.attention_f32_splits(1, 9, 3, keys - 15, 8192, size) == ops.attention_f32_splits(1, 9, 3, 15 - keys, 8192, size) == splits
    assert ops.attention_f32_least(16, 16) > 300 * 9 and ops.attention_f32_least(16, 16) < 600 * 9 and ops.attention_f32_least(16, 16) < 150 * 32
    assert ops.attention_f32_least(32, 16) == ops.attention_f32_least(16, 32) > 300 * 4 and ops.attention_f32_least(32, 32) <= 64 * 32
    assert ops.attention_f32_least(48, 16) == ops.attention_f32_least(64, 64) == 0


def test_the_tiles_of_products_into_the_stream():
    """A product into the residual stream goes by rates of its own (the parts of its rows' sums of squares follow the tile)."""
    from nnis_amd.kernels import ops

    width = {ops.TILE_64x128: 128, ops.TILE_64x64: 64, ops.TILE_256x256: 256, ops.TILE_256x192: 192, ops.TILE_128x128: 128, ops.TILE_256x128: 128,
             ops.TILE_128x192: 192}
    for (m, n, k), (tile, stream) in {
        (2048, 8192, 2048): (ops.TILE_256x256, ops.TILE_256x256),
        (2048, 2048, 8192): (ops.TILE_128x128, ops.TILE_128x128),
        (8192, 8192, 8192): (ops.TILE_256x256, ops.TILE_256x128),
        (4096, 4096, 14336): (ops.TILE_256x256, ops.TILE_256x128),
        (12288, 2048, 5632): (ops.TILE_256x128, ops.TILE_256x128),
        (2048, 576, 1536): (ops.TILE_64x64, ops.TILE_64x64),
    }.items():
        assert (ops.gemm_tile(m, n, k), ops.gemm_tile(m, n, k, residual=True)) == (tile, stream), (m, n, k)
        assert ops.core().nnis_gemm_residual_parts(m, n) >= 2 * -(-n // width[stream])  # (the room that any tile asks for)


@pytest.mark.parametrize("heads, kv_heads, head_dim", [(9, 3, 64), (32, 4, 64), (32, 32, 64), (16, 1, 256)])
def test_prefill_plans_of_short_prompts(heads, kv_heads, head_dim):
    """Up to 127 tokens: items of one column while a step has few, by the rows planned for and not by the length, which a replayed
    step knows by its class alone."""
    from nnis_amd.kernels.ops import prefill_plan

    for longest in (1, 24, 64, 65, 127):
        assert prefill_plan(longest, 64, heads, head_dim, kv_heads) == prefill_plan(longest, 128, heads, head_dim, kv_heads) == (1, 1)
        assert prefill_plan(longest, 65536, heads, head_dim, kv_heads) == (1, 0)
    assert prefill_plan(128, 128, heads, head_dim, kv_heads) == (2, 1)


@pytest.mark.parametrize("heads, kv_heads, head_dim", [(16, 4, 128), (32, 8, 96), (8, 8, 80)])
def test_prefill_plans_of_short_prompts_of_wide_heads(heads, kv_heads, head_dim):
    """Heads of 65 to 128 channels: items of one column up to 4,096 rows x heads, where they still find compute units without a block."""
    from nnis_amd.kernels.ops import prefill_plan

    most = 4096 // heads
    assert prefill_plan(100, most, heads, head_dim, kv_heads) == prefill_plan(1, 64, heads, head_dim, kv_heads) == (1, 1)
    assert prefill_plan(100, most + 1, heads, head_dim, kv_heads) == prefill_plan(24, 65024 // heads, heads, head_dim, kv_heads) == (1, 0)


@pytest.mark.parametrize("heads, kv_heads, width, dtype, batch, longest", [
    (9, 3, 576, torch.bfloat16, 1, 40960), (9, 3, 576, torch.bfloat16, 4, 37500), (9, 3, 576, torch.bfloat16, 8, 18750),
    (16, 16, 1024, torch.bfloat16, 1, 28125), (16, 16, 1024, torch.bfloat16, 4, 7031), (16, 16, 1024, torch.bfloat16, 16, 6144),
    (9, 3, 576, torch.bfloat16, 17, 4096), (9, 3, 576, torch.bfloat16, 32, 4096), (32, 4, 2048, torch.bfloat16, 4, 50000),
    (9, 3, 576, torch.float32, 8, 50000), (9, 3, 576, torch.float32, 16, 25000)])
def test_long_sequences_stay_with_the_layers_kernels(heads, kv_heads, width, dtype, batch, longest):
    """A step is launched as one up to the measured length and not from the next page on; wider models' at any length."""
    def taken(tokens):
        return chain_plan(2, batch, tokens, width=width, heads=heads, kv_heads=kv_heads, head_dim=64, inner=1536, dtype=dtype) is not None

    assert taken(1) and taken(longest) and not taken(longest + 1) and not taken(10 * longest)
    assert chain_plan(2, 16, 1 << 20, width=2048, heads=32, kv_heads=8, head_dim=64, inner=8192) is not None


def test_ways_to_cut_k_that_a_launched_step_does_not_have():
    def taken(batch, width, heads, inner):
        return chain_plan(2, batch, 500, width=width, heads=heads, kv_heads=heads, head_dim=64, inner=inner) is not None

    assert taken(16, 1024, 16, 2048) and not taken(1, 1024, 17, 2048) and not taken(16, 1024, 17, 2048)
    assert taken(16, 192, 4, 5056) and not taken(16, 192, 4, 5120) and taken(17, 192, 4, 5120)
    assert taken(1, 1088, 79, 8192) and not taken(1, 1088, 79, 8256) and not taken(1, 2048, 80, 2048) and taken(1, 2112, 80, 2048)


@pytest.mark.parametrize("batch, padded, taken", [(4, 4, True), (5, 7, True), (7, 7, True), (8, 8, False), (9, 12, False)])
def test_padding_keeps_large_groups_on_the_launch(batch, padded, taken, monkeypatch):
    """Five to seven sequences of more than four query heads a key head are padded to the most rows that the launch through all layers takes."""
    from nnis_amd.engine.graph import bucket
    from nnis_amd.kernels import ops

    monkeypatch.setattr(ops, "chain_takes", lambda *sizes: True)  # (the native side's sizes)
    assert bucket(batch) == padded
    assert (chain_plan(22, padded, 600, 2048, 32, 4, 64, 5632) is not None) == taken


@pytest.mark.parametrize("m, n, k, stored, others", [
    (12480, 2048, 5632, (8192, 160), (8192, 160)), (12480, 2048, 2048, (8192, 160), (8192, 160)), (12480, 2560, 2048, None, None),
    (9247, 8192, 5632, (8192, 160), None), (4348, 6144, 512, (2560, 192), None),  # 6% by the rule's model: into the stream 3 lost, behind a norm 6
    (12480, 11264, 2048, (11776, 128), None), (4862, 22016, 3072, None, None),     # 4%: stored 2 gained, and lost of weights beyond 128 MB
    (1106, 36864, 8192, None, None), (3862, 36864, 8192, None, None), (1388, 28672, 8192, None, None),  # weights beyond 256 MB: losses of 2 to 11%
    (8255, 3072, 14336, (5376, 160), (5376, 160)), (1568, 16384, 8128, (1024, 160), (1024, 160)), (1568, 16384, 8192, None, None)])
def test_lower_tiles_behind_large_ones(m, n, k, stored, others):
    from nnis_amd.kernels import ops

    for kind, want in ((True, stored), (False, others)):
        assert ops.gemm_large_rows(m, n, k, kind) == (want or (m, 256))


@pytest.mark.parametrize("m, n, k, tile", [(40, 5120, 2304, (64, 2)), (40, 5120, 2368, None), (48, 6144, 4096, None), (49, 5120, 2048, None),
                                           (64, 4096, 4096, (32, 4)), (64, 4096, 4160, None), (65, 4096, 4096, None)])
def test_products_that_share_k_in_groups(m, n, k, tile):
    """K in two parts between groups of waves loses 2 to 17% from 2,560 channels on, in four parts it gains as far as it was measured."""
    from nnis_amd.kernels import ops

    assert ops.gemm_grouped(m, n, k) == tile
