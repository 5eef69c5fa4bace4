"""The bf16 prompt form of the experts: four waves a workgroup, waves past the last column staging activations only, against
the 16-row kernel, whose bits it shares whatever the split (that kernel is held to the oracle in test_gpu_experts)."""

import pytest
import torch

from tensorfold_amd import experts, synthetic
from tests.test_gpu_experts import DEV, run

pytestmark = pytest.mark.gpu


# widths of 1 to 9 column blocks (a wave takes two of one matrix, one of two), so that three, two, one and none of a unit's waves
# are idle; items of 1 to 128 rows; one step along K and many; units for less than a round of workgroups and, with 600
# experts, for those that stay
@pytest.mark.parametrize("gs,swiglu,e,rows,d,ni", [
    (64, False, 3, 130, 64, 64), (64, False, 5, 300, 192, 320), (32, False, 4, 97, 288, 128), (64, True, 5, 200, 256, 192),
    (32, True, 4, 33, 128, 288), (64, False, 600, 900, 320, 576), (32, True, 600, 700, 256, 224)])
def test_bits_do_not_depend_on_the_units(gs, swiglu, e, rows, d, ni):
    up = [synthetic.affine_general(ni, d, gs, 11 + i, (e,)) for i in range(2 if swiglu else 1)]
    down = synthetic.affine_general(d, ni, gs, 17, (e,))
    ex = experts.make([tuple(t.to(DEV) for t in m) for m in up], tuple(t.to(DEV) for t in down), gs,
                      arith=experts.ARITH_BF16)
    g = torch.Generator().manual_seed(5)
    picks = torch.stack([torch.randperm(e, generator=g)[:3] for _ in range(rows)]).to(torch.int32)
    picks[:, 0] = torch.where(picks[:, 1:].eq(1).any(1), picks[:, 0], torch.ones(rows, dtype=torch.int32))     # one expert most rows share
    x = synthetic.activations(rows, d, 23, 0.5).to(DEV)
    act, y, _ = run(ex, x, picks, prefill=True, tile=128)
    want_act, want, _ = run(ex, x, picks, prefill=True, tile=16)
    assert torch.isfinite(want).all() and want.abs().max() > 0
    assert torch.equal(act, want_act) and torch.equal(y, want)
