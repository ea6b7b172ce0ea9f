"""Which form the experts' products take, by their sizes and the chip."""
import pytest


def _tile(E, m, K, F, mode, units=256):
    from gpt_fast_amd.ops.routed_experts import rows_tile, tall_tiles_win
    sizes = (E, int(m * E), F, K, mode, units)
    return 4 if tall_tiles_win(*sizes) else rows_tile(*sizes)


# measured, a tile of 128 x 128 against one of 256 x 256: products where the one chosen is at least 3 % faster
@pytest.mark.parametrize("E,m,K,F,mode,tile", [
    (16, 120, 3584, 4096, 0, 4), (16, 140, 3584, 4096, 0, 2), (16, 222, 3584, 4096, 0, 4), (32, 64, 4096, 3584, 1, 2),
    (32, 100, 4096, 3584, 1, 4), (32, 222, 4096, 3584, 1, 4), (8, 180, 3584, 4096, 0, 2), (8, 222, 3584, 4096, 0, 4),
    (32, 140, 2816, 2048, 1, 2), (16, 222, 4096, 3584, 1, 2), (16, 80, 2048, 7168, 0, 2), (16, 140, 4096, 2048, 2, 2),
    (16, 80, 2048, 4096, 0, 4), (16, 222, 5120, 1536, 2, 4), (64, 180, 4096, 2048, 2, 4), (128, 140, 2048, 4096, 0, 4)])
def test_the_tile_that_was_measured_faster(E, m, K, F, mode, tile):
    assert _tile(E, m, K, F, mode) == tile


def test_tiles_by_rows_and_inner_size():
    assert [_tile(32, m, 4096, 3584, 1) for m in (0.5, 1, 35, 36)] == [2, 1, 1, 2]
    assert [_tile(128, m, 1024, 4096, 0) for m in (100, 399, 400)] == [0, 0, 4]
    assert [_tile(128, m, 1024, 4096, 1) for m in (100, 400)] == [0, 0]
    # a gated product's tiles make half the columns, and a chip of half the units is full with half the columns
    assert all(_tile(16, m, 4096, 2048, 2) == _tile(16, m, 4096, 4096, 0) == _tile(16, m, 4096, 2048, 0, 128)
               for m in (40, 80, 100, 140, 200, 300))


def test_two_pieces_ahead_where_every_workgroup_that_can_have_work_is_on_the_chip():
    from gpt_fast_amd.ops.routed_experts import _pieces_ahead
    # 32 tiles of 16 rows: 24 experts on 256 units, whether the experts or the pairs are fewer
    assert [_pieces_ahead(E, P, 512, 256) for E, P in ((24, 99), (25, 99), (64, 24), (64, 25))] == [2, 1, 2, 1]
    assert [_pieces_ahead(1, 1, rows, 1) for rows in (1, 48, 49)] == [2, 2, 1]


def test_the_routers_launch_orders_where_its_tokens_do_not_crowd_one_compute_unit():
    from gpt_fast_amd.ops.routed_experts import orders_sooner_with_route as sooner
    assert [sooner(n, 32, 4, 2) for n in (1, 8, 9, 16)] == [True, True, False, False]
    assert [sooner(n, 256, 8, 4) for n in (4, 5)] == [True, False]
    assert [sooner(n, 32, 4, 4) for n in (9, 16, 17)] == [True, True, False]
