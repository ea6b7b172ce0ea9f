"""Which form the experts' products take, by their sizes and the chip."""


def test_tall_tiles_by_rows_rounds_and_inner_size():
    from gpt_fast_amd.ops.routed_experts import tall_tiles_win

    def wins(E, F, K, mode, means, units=256):
        return [tall_tiles_win(E, int(m * E), F, K, mode, units) for m in means]
    assert wins(32, 3584, 4096, 1, (1, 63, 64, 100, 800)) == [False, False, True, True, True]
    # a round of 128 x 128 tiles; a round of these; a little more than one; clearly more
    assert wins(8, 3584, 4096, 1, (180, 300)) == [False, True]
    assert wins(16, 3584, 4096, 1, (180, 222, 300)) == [True, False, True]
    assert wins(128, 4096, 1024, 0, (100, 400)) == [False, False]
    # a gated product's tiles make half the columns
    assert wins(16, 2048, 4096, 2, (100,)) == wins(16, 4096, 4096, 0, (100,)) == [True]


def test_two_pieces_ahead_where_every_workgroup_that_can_have_work_is_on_the_chip():
    from gpt_fast_amd.ops.routed_experts import _pieces_ahead
    # 32 tiles of 16 rows: 24 experts on 256 units, whether the experts or the pairs are fewer
    assert [_pieces_ahead(E, P, 512, 256) for E, P in ((24, 99), (25, 99), (64, 24), (64, 25))] == [2, 1, 2, 1]
    assert [_pieces_ahead(1, 1, rows, 1) for rows in (1, 48, 49)] == [2, 2, 1]
