"""The row tiles of a prompt item, by its rows: every count at the edges of a tile, in both prompt arithmetics and in workgroups
that take one unit and that stay, against the 16-row kernel's bits (that kernel is held to the oracle in test_gpu_experts)."""

import pytest
import torch

from tensorfold_amd import experts, synthetic
from tests.test_gpu_experts import DEV, run

pytestmark = pytest.mark.gpu
COUNTS = [1, 15, 16, 17, 31, 32, 33, 48, 49, 64, 65, 80, 96, 97, 112, 113, 127, 128, 129, 160]


@pytest.mark.parametrize("arith", [experts.ARITH_F16, experts.ARITH_BF16])
@pytest.mark.parametrize("gs,swiglu,copies,d,ni", [(64, False, 1, 128, 192), (32, True, 1, 64, 96),
                                                   (64, True, 4, 64, 4096), (32, False, 4, 96, 4096)])
def test_every_row_count_has_the_bits_of_the_16_row_kernel(gs, swiglu, copies, d, ni, arith):
    counts = COUNTS * copies                                  # expert e is picked by counts[e] rows
    e = len(counts)
    up = [synthetic.affine_general(ni, d, gs, 3 + i, (e,)) for i in range(2 if swiglu else 1)]
    down = synthetic.affine_general(d, ni, gs, 7, (e,))
    ex = experts.make([tuple(t.to(DEV) for t in m) for m in up], tuple(t.to(DEV) for t in down), gs, arith=arith)
    picks = torch.repeat_interleave(torch.arange(e, dtype=torch.int32), torch.tensor(counts))
    picks = picks[torch.randperm(len(picks), generator=torch.Generator().manual_seed(1))][:, None].contiguous()
    x = synthetic.activations(len(picks), d, 9, 0.5).to(DEV)
    act, y, _ = run(ex, x, picks, prefill=True, tile=128)
    want_act, want, _ = run(ex, x, picks, prefill=True, tile=16)
    assert torch.isfinite(want).all() and want.abs().max() > 0
    assert torch.equal(act, want_act) and torch.equal(y, want)
