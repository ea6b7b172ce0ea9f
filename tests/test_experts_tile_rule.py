"""Where the experts' products take tiles of 256 x 256 that are as high as their rows."""


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
