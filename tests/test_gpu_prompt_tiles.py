"""The prompt matmul's tiles against one another: the same bits over odd rows, columns and ragged K, both arithmetics, both
result types, rows with a stride, for the tile that the call chooses and for every tile asked for by its code."""

import pytest
import torch

from tensorfold_amd import qmm, synthetic

pytestmark = pytest.mark.gpu
DEV = "cuda"


# (rows, columns, K, group size) and the tile that the call takes: its row and column edges, one step and less of K, a
# step that ends inside (K = 32, 96, 736, 1056 are not whole steps of 128 or 256), more columns than rows and the reverse
SHAPES = [(1, 1, 32, 32, 1), (3, 130, 64, 64, 2), (16, 4096, 96, 32, 2), (17, 640, 256, 64, 2),
          (33, 1024, 736, 32, 2), (100, 4096, 1056, 32, 3), (129, 515, 320, 64, 2), (257, 4100, 448, 64, 3),
          (300, 8192, 512, 64, 5), (1000, 4096, 192, 64, 6), (999, 4099, 320, 64, 5), (1000, 2047, 192, 64, 5),
          (1030, 4096, 544, 32, 5), (2000, 130, 96, 32, 3), (2000, 4100, 192, 64, 9), (1999, 4096, 320, 32, 9),
          (4096, 513, 64, 64, 6)]


def operands(m, n, k, gs):
    q = qmm.pack(*(t.to(DEV) for t in synthetic.affine_general(n, k, gs, 7 * n + k)), gs)
    wide = synthetic.activations(m, k + 8, m + n).to(DEV)
    return q, (wide[:, :k].contiguous(), wide[:, :k])


@pytest.mark.parametrize("m,n,k,gs,tile", SHAPES)
def test_the_chosen_tile_has_the_bits_of_the_others(m, n, k, gs, tile):
    assert qmm.prompt_tile(m, n, k) == tile
    q, xs = operands(m, n, k, gs)
    for x in xs:
        for arith in (0, 1):
            for f32 in (False, True):
                got = qmm.prefill_matmul(x, q, f32=f32, arith=arith)
                assert torch.equal(got, qmm.prefill_matmul(x, q, f32=f32, arith=arith, tile=8)), (arith, f32)


# every tile on the same calls: its edges in rows and columns, less than a step of K, whole steps, one that ends inside
@pytest.mark.parametrize("m", [1, 15, 16, 31, 33, 63, 65, 129, 257])
@pytest.mark.parametrize("n,k,gs", [(515, 64, 64), (515, 192, 64), (1030, 320, 32), (130, 544, 32), (65, 1088, 64)])
def test_every_tile_has_the_same_bits(m, n, k, gs):
    q, xs = operands(m, n, k, gs)
    for x in xs:
        for arith in (0, 1):
            for f32 in (False, True):
                want = qmm.prefill_matmul(x, q, f32=f32, arith=arith, tile=8)
                for tile in (1, 2, 3, 4, 5, 6) + ((9,) if k % 64 == 0 else ()):
                    assert torch.equal(qmm.prefill_matmul(x, q, f32=f32, arith=arith, tile=tile), want), (tile, arith, f32)


def test_a_rows_infinity_stays_in_its_row_at_a_ragged_end():
    """The inputs past a ragged K count as nothing, also next to an infinity in the last piece of a row."""

    n, k, gs = 200, 96, 32
    q = qmm.pack(*(t.to(DEV) for t in synthetic.affine_general(n, k, gs, 5)), gs)
    x = synthetic.activations(40, k, 6).to(DEV)
    want = qmm.prefill_matmul(x, q, f32=True, arith=1)
    x[7, k - 1] = float("inf")
    got = qmm.prefill_matmul(x, q, f32=True, arith=1)
    others = [r for r in range(40) if r != 7]
    assert torch.equal(got[others], want[others])
    assert torch.equal(got[7].isnan(), qmm.prefill_matmul(x, q, f32=True, arith=1, tile=8)[7].isnan())
