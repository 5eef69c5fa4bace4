"""The rule behind the EXL3 prompt matmul's workgroup heights, without a GPU."""

from tensorfold_amd.exl3 import prefill


def test_every_size_has_a_height_and_every_height_a_size():
    rows = [*range(1, 300, 13), *range(300, 6000, 97), 40000, 1 << 20, (1 << 31) - 1]
    seen = {prefill.row_tiles(m, n) for m in rows for n in (128, 1024, 4224, 5120, 6272, 9216, 17408, 152576)}
    assert seen == set(range(2, 10))


def test_few_rows_take_low_workgroups_and_past_eight_rounds_all_are_128_rows():
    assert prefill.row_tiles(1, 128) == prefill.row_tiles(31, 17408) == 2
    assert prefill.row_tiles(1000, 17408) == 9                       # 480 tiles in one round, where eight of 128 rows are 544
    for m in (16385, 100000):
        assert prefill.row_tiles(m, 8192) == 8
