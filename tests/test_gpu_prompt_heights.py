"""The eight-wave prompt kernel's row tiles, 32 to 144 rows by how a call's tiles fill the chip: every height, alone and beside
tiles of 16 rows less, against the four-wave kernel's bits."""

import pytest
import torch

from tensorfold_amd import _lib, qmm, synthetic

pytestmark = pytest.mark.gpu
DEV = "cuda"


# 65,536 columns are 128 tiles of 512: two row tiles fill the chip, so a call of u units of 16 rows takes tiles of half of them
@pytest.mark.parametrize("units,rows", [(2, 32), (4, 32), (5, 48), (6, 48), (7, 64), (9, 80), (12, 96), (13, 112), (15, 128),
                                        (16, 128), (17, 144), (18, 144)])
@pytest.mark.parametrize("gs", [32, 64])
def test_a_height_has_the_bits_of_the_others(units, rows, gs):
    n, k = 65536, 128
    assert _lib.lib().tf_qmm_prompt_rows(16 * units, n) == rows
    q = qmm.pack(*(t.to(DEV) for t in synthetic.affine_general(n, k, gs, units)), gs)
    for m in (16 * units, 16 * units - 15):                  # whole tiles, a last one of a row
        wide = synthetic.activations(m, k + 8, m).to(DEV)
        for x in (wide[:, :k].contiguous(), wide[:, :k]):
            for arith in (0, 1):
                got = qmm.prefill_matmul(x, q, arith=arith, tile=9)
                assert torch.equal(got, qmm.prefill_matmul(x, q, arith=arith, tile=8)), (m, arith)


@pytest.mark.parametrize("m,n,k", [(300, 17000, 64), (1000, 17408, 320), (1999, 5000, 192)])          # several rounds, ragged columns
def test_rounds_of_two_heights(m, n, k):
    q = qmm.pack(*(t.to(DEV) for t in synthetic.affine_general(n, k, 64, m)), 64)
    x = synthetic.activations(m, k, n).to(DEV)
    for f32 in (False, True):
        assert torch.equal(qmm.prefill_matmul(x, q, f32=f32, tile=9), qmm.prefill_matmul(x, q, f32=f32, tile=8)), f32


# tiles of 128 rows throughout: the last has 64 rows or less, 32 or less
@pytest.mark.parametrize("m,n", [(1472, 10240), (1457, 10230), (1712, 9216), (2080, 7680), (2065, 7675)])
@pytest.mark.parametrize("gs,k", [(64, 64), (32, 192)])
def test_a_short_last_tile(m, n, gs, k):
    assert _lib.lib().tf_qmm_prompt_rows(m, n) == 128
    q = qmm.pack(*(t.to(DEV) for t in synthetic.affine_general(n, k, gs, m)), gs)
    x = synthetic.activations(m, k, n).to(DEV)
    for arith in (0, 1):
        for f32 in (False, True):
            assert torch.equal(qmm.prefill_matmul(x, q, f32=f32, arith=arith, tile=9),
                               qmm.prefill_matmul(x, q, f32=f32, arith=arith, tile=8)), (arith, f32)
