"""The K splits of EXL3 routed experts: as many workgroups as fill the chip from the first row on, whatever the picks a row."""

from types import SimpleNamespace

import pytest

from tensorfold_amd.exl3 import experts


def pairs_allow(k: int) -> int:
    return max([1] + [sk for sk in (2, 4, 8) if k // 32 >= (3 if sk == 2 else 3.5) * experts.WAVES * sk])


# one row of few picks: the splits a wider row does not need
@pytest.mark.parametrize("dims,width,slots,splits", [
    (4096, 2048, 1, (8, 4)), (4096, 2048, 4, (4, 4)), (4096, 2048, 8, (4, 2)), (4096, 6144, 1, (8, 8)),
    (4096, 6144, 8, (2, 4)), (7168, 2048, 2, (8, 4)), (5120, 1536, 1, (8, 2)), (4096, 14336, 8, (1, 4))])
def test_a_layers_splits_follow_its_picks_a_row(dims, width, slots, splits):
    layer = SimpleNamespace(dims=dims, width=width, count=16)
    for rows in (1, 3):
        scratch = experts.Scratch(layer, rows, slots, device="cpu")
        assert (scratch.sk_gu, scratch.sk_d) == splits


def test_a_row_fills_the_chip_where_its_pairs_allow():
    for k in range(128, 20481, 128):
        for nb in (1, 4, 16, 48, 112, 600):
            for slots in (1, 2, 5, 8, 10, 96):
                for gateup in (False, True):
                    sk = experts.default_config(k, 128 * nb, gateup, slots)
                    row, most = nb * slots * (1 + gateup), pairs_allow(k)
                    assert sk in (1, 2, 4, 8) and sk <= most and sk * experts.WAVES <= k // 32
                    assert sk == most or row * sk >= 512                     # no fewer than fill the chip ...
                    assert sk == 1 or row * sk // 2 < 1024                    # ... and no more
