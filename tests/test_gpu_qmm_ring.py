"""The decode matmul of 9 and more rows, whose operands go through LDS: the bits of the same rows in calls of their own (one
row takes another walk, which test_gpu_qmm holds to the oracle)."""

import dataclasses

import pytest
import torch

from tensorfold_amd import qmm, synthetic

pytestmark = pytest.mark.gpu
DEV = "cuda"


# one group (three waves of four without any), an odd number of them, K slices, a last column tile of 6 and of 63 columns, a K
# so deep that in groups of 64 9 and 10 rows take the walk of few rows, as up to 16 rows do where a wave has less than two groups
@pytest.mark.parametrize("gs", [32, 64])
@pytest.mark.parametrize("n,groups", [(70, 1), (64, 3), (129, 9), (1023, 16), (512, 80), (70, 129)])
def test_rows_have_the_bits_of_a_call_of_their_own(gs, n, groups):
    k = gs * groups
    q = qmm.pack(*(t.to(DEV) for t in synthetic.affine_general(n, k, gs, 3 + groups)), gs)
    x = synthetic.activations(65, k, 7).to(DEV)
    want = torch.cat([qmm.matmul(x[r:r + 1], q) for r in range(65)])
    assert torch.isfinite(want.float()).all() and want.float().abs().max() > 0
    for rows in (9, 10, 11, 15, 16, 17, 31, 32, 33, 65):
        assert torch.equal(qmm.matmul(x[:rows], q), want[:rows]), rows
    # inputs in rows of a wider tensor; scales in rows that do not start on whole dwords (the walk of few rows takes those)
    wide = torch.zeros((21, k + 8), dtype=torch.bfloat16, device=DEV)
    wide[:, 8:] = x[:21]
    assert torch.equal(qmm.matmul(wide[:, 8:], q), want[:21])
    odd = lambda t: torch.cat([t, t[:, :1]], 1)[:, :-1]
    ragged = dataclasses.replace(q, scales=odd(q.scales), biases=odd(q.biases))
    assert ragged.scales.stride(0) % 2 == 1
    for rows in (12, 21):
        assert torch.equal(qmm.matmul(x[:rows], ragged), want[:rows]), rows


@pytest.mark.parametrize("k", [1024, 5120])                  # waves of one group and of two or three
def test_a_group_of_weights_has_the_bits_of_each_alone(k):
    qs = [qmm.pack(*(t.to(DEV) for t in synthetic.affine_general(n, k, 64, n)), 64) for n in (512, 200, 64)]
    x = synthetic.activations(40, k, 5).to(DEV)
    for rows in (9, 16, 17, 40):
        for got, q in zip(qmm.matmul_group(x[:rows], qs), qs):
            assert torch.equal(got, qmm.matmul(x[:rows], q)), rows
