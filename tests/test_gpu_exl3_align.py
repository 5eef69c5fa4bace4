"""EXL3 routed experts whose trellises start on any 4-byte boundary (a view into a checkpoint's file) give the bits of the
same trellises on 16-byte ones: the walk's loads are wider than the alignment that is asked for."""

import pytest
import torch

from tensorfold_amd.exl3 import experts

pytestmark = pytest.mark.gpu
DEV = "cuda"


# one width of each way a run divides into a lane's loads: 32 K2 words = whole fours, ones to threes, a half wave more
@pytest.mark.parametrize("bits,cb", [(1, "mul1"), (1.5, "mul1"), (2, "mcg"), (3, "3inst"), (4, "mcg"), (4.5, "mul1"),
                                     (5.5, "mul1"), (6, "3inst"), (7, "mcg"), (7.5, "mul1"), (8, "3inst"), (8, "mul1")])
def test_any_word_alignment(bits, cb):
    n_exp, d, width, rows, top_k = 3, 128, 256, 5, 2
    gen = torch.Generator().manual_seed(int(2 * bits))
    mats = []
    for k, n in ((d, width), (d, width), (width, d)):
        mats.append([(torch.randint(-2 ** 15, 2 ** 15, (k // 16, n // 16, int(16 * bits)), generator=gen).to(torch.int16),
                      torch.randn(k, generator=gen).half().to(DEV), (torch.randn(n, generator=gen) * 0.1).half().to(DEV))
                     for _ in range(n_exp)])
    x = torch.randn((rows, d), generator=gen).bfloat16().to(DEV)
    pick = torch.stack([torch.randperm(n_exp, generator=gen)[:top_k] for _ in range(rows)]).int().to(DEV).contiguous()
    outs = []
    for words in range(4):
        placed, keep = [], []
        for triples in mats:
            row = []
            for t, suh, svh in triples:
                store = torch.zeros(t.numel() + 8, dtype=torch.int16, device=DEV)
                view = store[2 * words:2 * words + t.numel()].view(t.shape)
                view.copy_(t)
                keep.append(store)
                row.append((view, suh, svh))
            placed.append(row)
        ex = experts.prepare(*placed, cb)
        outs.append(experts.routed(x, pick, None, ex, experts.Scratch(ex, rows, top_k), None, rows).clone())
    assert torch.isfinite(outs[0]).all() and outs[0].abs().sum() > 0
    for words in range(1, 4):
        assert torch.equal(outs[0], outs[words]), words
