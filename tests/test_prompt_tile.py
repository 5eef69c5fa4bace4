"""The rule behind the prompt matmul's tile, without a GPU: what ``prompt_tile`` names is what the launch takes."""

import pytest

from tensorfold_amd import _lib, qmm

CODES = {1, 2, 3, 4, 5, 6, 8, 9}


def test_the_rule_looks_at_rows_and_columns():
    assert qmm.prompt_tile(100, 4096, 4096) == 3           # 128 x 512 tiles would be 8 workgroups
    assert qmm.prompt_tile(512, 4096, 4096) == 6           # 31.0 us; 32 x 128 33.4
    assert qmm.prompt_tile(1000, 4096, 4096) == 6
    assert qmm.prompt_tile(2000, 4096, 4096) == 9
    assert qmm.prompt_tile(4096, 17408, 5120) == 9


def test_a_short_k_keeps_the_tiles_that_start_quickly():
    assert qmm.prompt_tile(4096, 17408, 96) == 8           # 62 us; 64 x 128 76
    assert qmm.prompt_tile(4096, 8192, 160) == 8           # 39 us; 47
    assert qmm.prompt_tile(200, 17408, 32) == 8            # 7.6 us; 32 x 128 11.3
    assert qmm.prompt_tile(1500, 2048, 96) == 6            # 6.8 us; 32 x 128 9.8
    assert qmm.prompt_tile(65, 65536, 64) == 9             # 11.7 us; 32 x 128 16.3
    assert qmm.prompt_tile(64, 17408, 64) == 4             # 4.9 us; 32 x 64 5.9
    assert qmm.prompt_tile(8, 17408, 64) == 1              # 3.6 us; 16 x 64 4.1
    assert qmm.prompt_tile(33, 8192, 64) == 3              # 4.2 us; four-wave 4.5
    assert qmm.prompt_tile(4096, 8192, 224) == 6           # from 192 inputs on the other rule


@pytest.mark.parametrize("m,n,k", [(400, 4096, 4096), (300, 6144, 4096), (256, 8192, 4096), (500, 4096, 5120), (98, 13184, 800),
                                   (2264, 730, 2272)])
def test_one_round_of_64_x_128_is_taken_where_32_x_128_takes_two(m, n, k):
    assert qmm.prompt_tile(m, n, k) == 6


def test_a_grid_that_an_xcd_takes_in_two_rounds_is_not_one():
    assert qmm.prompt_tile(512, 4000, 4096) == 6           # 32 tiles of columns, the faster index, x 8: 32 on each XCD
    assert qmm.prompt_tile(576, 3584, 4096) == 5           # 28, a grid of 32 x 9: 36 on the first
    assert qmm.prompt_tile(1000, 2047, 448) == 5           # (fewer than 512 inputs)


@pytest.mark.parametrize("k", [32, 64, 96, 4096, 4128, 5120])
def test_every_size_has_a_tile(k):
    for m in (0, 1, 16, 17, 64, 65, 300, 1000, 4096, 1 << 20, (1 << 31) - 1):
        for n in (1, 64, 130, 4096, 17408, 248320):
            tile = qmm.prompt_tile(m, n, k)
            assert tile in CODES and (tile != 9 or k % 64 == 0), (m, n)


@pytest.mark.parametrize("m,n,tiles,rows", [
    (2471, 5739, 20, 128), (1166, 12301, 10, 128), (1181, 12342, 10, 128), (2193, 6202, 18, 128), (953, 15629, 8, 128),      # of 128 rows
    (1858, 4352, 28, 80), (1329, 8768, 14, 96), (1362, 7808, 16, 96), (1554, 8372, 15, 112), (1300, 4096, 32, 48),          # dealt out
    (2543, 5248, 23, 112), (1000, 17408, 7, 144), (4096, 17408, 30, 144)])
def test_one_round_of_eight_wave_tiles_is_dealt_out_where_its_tallest_tile_is_shorter_for_it(m, n, tiles, rows):
    assert (_lib.lib().tf_qmm_prompt_row_tiles(m, n), _lib.lib().tf_qmm_prompt_rows(m, n)) == (tiles, rows)


def test_a_weight_past_a_32_bit_offset_keeps_off_the_eight_wave_tile():
    assert qmm.prompt_tile(4096, 1 << 20, 8128) == 9       # 0xFE000000 bytes of codes
    assert qmm.prompt_tile(4096, 1 << 20, 8192) != 9       # 2^32


def test_a_code_that_names_nothing_is_refused():
    for tile in (-1, 7, 10):
        with pytest.raises(ValueError, match="tile"):
            qmm.prefill_matmul(None, None, tile=tile)
