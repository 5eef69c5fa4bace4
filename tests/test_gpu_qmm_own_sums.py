"""The decode matmul that takes its group sums itself: the bits of the call that is given them, in every form of the launch
(arrival counters, whole column tiles, registers, LDS), and the sums by themselves at the edges of their tiles."""

import pytest
import torch

from tensorfold_amd import qmm, synthetic

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("gs", [32, 64])
# one group, three, an odd number, K slices, a K without counters' second launch, a deep one
@pytest.mark.parametrize("n,groups", [(1, 1), (70, 3), (129, 9), (1023, 16), (512, 80), (70, 129)])
def test_the_bits_of_the_call_that_is_given_the_sums(gs, n, groups):
    k = gs * groups
    q = qmm.pack(*(t.to(DEV) for t in synthetic.affine_general(n, k, gs, n + groups)), gs)
    wide = synthetic.activations(65, k + 8, 3).to(DEV)
    for m in (1, 4, 5, 8, 9, 16, 17, 33, 65):
        for x in (wide[:m, :k].contiguous(), wide[:m, 8:]):
            xs = qmm.group_sums(x, gs)
            for f32 in (False, True):
                assert torch.equal(qmm.matmul(x, q, f32=f32), qmm.matmul(x, q, xs, f32=f32)), (m, f32)
            assert torch.equal(qmm.matmul(x, q, reduce=False), qmm.matmul(x, q, xs, reduce=False)), m


@pytest.mark.parametrize("gs", [32, 64])
@pytest.mark.parametrize("m,groups", [(1, 1), (15, 15), (16, 16), (17, 17), (33, 64), (5, 65), (64, 130)])
def test_the_sums_at_the_edges_of_their_tiles(gs, m, groups):
    k = gs * groups
    wide = synthetic.activations(m, k + 8, m + groups).to(DEV)
    for x in (wide[:, :k].contiguous(), wide[:, 8:]):
        exact, size = x.double().reshape(m, groups, gs).sum(2), x.double().abs().reshape(m, groups, gs).sum(2)
        # each addition rounds a partial sum no larger than the magnitudes' by at most 2^-23 (the matrix unit truncates)
        assert bool(((qmm.group_sums(x, gs).double() - exact).abs() <= gs * 2.0 ** -23 * size).all())
