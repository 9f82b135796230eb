"""Which kernel instance serves a call, on both sides of the lines where the
measured order of the candidates changes (the comments at the rules hold the
times).  Names only: no GPU."""
import pytest

import kvbridge_amd as kvb

FAKE = kvb.device_input(*([0x1000] * 8))


def name(kv_heads, head_rows, dim, splits, tiles, fused=False, page=64):
    tokens = splits * tiles * 64
    s = kvb.make_shape(1, kv_heads * head_rows, kv_heads, dim, page, -(-tokens // page), tokens, 0, tokens, 0.1)
    return kvb.selected_kernel_name(s, FAKE, tiles * 64, fused)


def waves_chunk(*args):
    """(waves, one-tile chunks, single launch) of an int8 split kernel."""
    n = name(*args)
    assert n.startswith("split_i8_kernel<"), n
    f = n[len("split_i8_kernel<"):-1].split(",")
    return int(f[1]), f[2] == "1", f[5] == "true"


@pytest.mark.parametrize("head_rows", [1, 2, 4])
@pytest.mark.parametrize("dim", [64, 128])
def test_waves_of_short_splits(dim, head_rows):
    """Eight waves hold a tile each while a work-group has the CU to itself;
    with two per CU, and past 8 tiles (12 at dim 64), four waves are faster."""
    for tiles, one_per_cu, two_per_cu in [(4, (4, True), (4, True)), (5, (8, True), (4, True)), (8, (8, True), (4, True)),
                                          (9, (8, True) if dim == 64 else (4, False), (4, False)),
                                          (12, (8, True) if dim == 64 else (4, False), (4, False)),
                                          (13, (4, False), (4, False)), (15, (4, False), (4, False)),
                                          (16, (8, False), (8, False))]:
        assert waves_chunk(8, head_rows, dim, 32, tiles)[:2] == one_per_cu, tiles
        assert waves_chunk(8, head_rows, dim, 33, tiles)[:2] == two_per_cu, tiles
        assert waves_chunk(8, head_rows, dim, 64, tiles)[:2] == two_per_cu, tiles


def test_waves_of_the_single_launch():
    """The in-kernel merge wants a thread per output: eight waves to 12 tiles."""
    assert waves_chunk(8, 4, 128, 4, 12, True) == (8, True, True)
    assert waves_chunk(8, 1, 128, 4, 12, True) == (8, True, True)
    assert waves_chunk(8, 1, 128, 4, 13, True) == (4, False, True)
    assert waves_chunk(8, 4, 128, 4, 13, True) == (4, False, False)
    assert waves_chunk(8, 4, 128, 16, 12, True) == (4, False, False)  # 16 splits of four head-rows: two launches


def test_waves_at_dim_256():
    assert waves_chunk(8, 4, 256, 32, 3)[:2] == (4, True) and waves_chunk(8, 4, 256, 33, 3)[:2] == (2, False)
    assert waves_chunk(8, 4, 256, 33, 8)[:2] == (4, True) and waves_chunk(8, 4, 256, 32, 9)[:2] == (4, False)


def test_a_lone_split_is_one_launch():
    """At dim 256 the in-kernel merge serves one head-row; a split without
    others needs none."""
    for head_rows in (1, 2, 4):
        assert waves_chunk(8, head_rows, 256, 1, 20, True)[2]
        assert waves_chunk(8, head_rows, 256, 2, 20, True)[2] == (head_rows == 1)


@pytest.mark.parametrize("head_rows", [5, 8])
def test_wide_gqa_over_the_int8_kernels_round(head_rows):
    """5 to 8 head-rows over splits of up to 15 tiles: the generic MFMA kernel,
    but not where the grid all but fills the first round of the int8 kernel's
    one-wave work-groups at dim 128."""
    def generic(dim, groups, tiles):
        return ": split_generic_i8_kernel<" in name(8, head_rows, dim, groups // 8, tiles)

    for tiles in (4, 12, 15):
        assert [g for g in (64, 512, 760, 768, 1024, 1032, 1536, 2048) if not generic(128, g, tiles)] == [768, 1024]
        assert all(generic(64, g, tiles) for g in (64, 512, 776, 1024, 2048))
    assert not generic(128, 64, 16) and not generic(64, 64, 16)


def test_wide_gqa_batches():
    """The same grid of a batch: full sequences only."""
    def generic(batch, max_tokens, total):
        s = kvb.make_batch_shape(batch, 1, 64, 8, 128, 64, 1 << 14, max_tokens, total, 1 << 14, 512, 0.1, True)
        return ":" in kvb.batch_kernel_name(s, kvb.batch_input(*([0x1000] * 10)))

    assert not generic(8, 8192, 8 * 8192) and generic(8, 8192, 8 * 7000)
    assert generic(40, 8192, 40 * 8192) and generic(4, 8192, 4 * 8192)
