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
        # an addition loses at most 2^-23 of a partial sum no larger than the magnitudes' (the matrix unit cuts off, it does not
        # round: how close the sums are as a whole is below)
        assert bool(((qmm.group_sums(x, gs).double() - exact).abs() <= gs * 2.0 ** -23 * size).all())


@pytest.mark.parametrize("gs", [32, 64])
@pytest.mark.parametrize("kind", ["normal", "magnitudes", "relu2", "three decades"])
def test_the_sums_are_as_close_as_rounded_additions(gs, kind):
    """Against 64 bits: root mean square error over the magnitudes' sum no larger than that of rounded fp32 additions, eight inputs
    in order and a tree over the eights.  Over a quarter of a million groups an rms is known to 0.15 %; the 1 % is six of those."""

    m, k = 2048, 8192
    gen = torch.Generator(device=DEV).manual_seed(gs)
    z = torch.randn((m, k), generator=gen, device=DEV)
    x = {"normal": lambda: z, "magnitudes": lambda: z.abs(), "relu2": lambda: z.clamp(min=0) ** 2,
         "three decades": lambda: z.abs() * 10 ** (3 * torch.rand((m, k), generator=gen, device=DEV))}[kind]().bfloat16()
    wide = x.double().view(m, k // gs, gs)
    eights = x.float().view(m, k // gs, gs // 8, 8)
    rounded = eights[..., 0]
    for i in range(1, 8):
        rounded = rounded + eights[..., i]
    while rounded.shape[-1] > 1:
        rounded = rounded[..., 0::2] + rounded[..., 1::2]
    exact, size = wide.sum(2), wide.abs().sum(2)
    error = lambda sums: float(((sums.double() - exact) / size).square().mean().sqrt())
    assert 0 < error(qmm.group_sums(x, gs)) <= 1.01 * error(rounded[..., 0])
