"""The combine of 16-bit pair outputs, eight columns a thread, against the two-column form's bits (rows of their own)."""

import pytest
import torch

from tensorfold_amd import moe

pytestmark = pytest.mark.gpu
DEV = "cuda"


# one slot, a batch of eight and one more, three batches; columns that end inside a workgroup; rows that share one
@pytest.mark.parametrize("rows,slots,d", [(600, 1, 512), (700, 8, 392), (521, 9, 520), (4096, 11, 64), (300, 17, 2688)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_rows_have_the_bits_of_a_call_of_their_own(rows, slots, d, dtype):
    gen = torch.Generator(device=DEV).manual_seed(rows)
    y = torch.randn((rows, slots, d), generator=gen, device=DEV).to(dtype)
    w = torch.rand((rows, slots), generator=gen, device=DEV)
    y[1, 0, 3], y[2, slots - 1, d - 1] = float("inf"), float("nan")
    got = moe.combine(y, w)
    one = lambda r: moe.combine(y[r:r + 1].contiguous(), w[r:r + 1].contiguous())[0]
    for r in (0, 1, 2, rows // 2, rows - 1):
        assert torch.equal(torch.nan_to_num(got[r].float()), torch.nan_to_num(one(r).float())), r
    # unaligned outputs take the other form, whose bits are the same
    odd = torch.empty((rows * slots * d + 2,), dtype=dtype, device=DEV)[2:].view(rows, slots, d).copy_(y)
    assert torch.equal(torch.nan_to_num(moe.combine(odd, w).float()), torch.nan_to_num(got.float()))


@pytest.mark.parametrize("slots", range(1, 17))
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_every_count_of_slots_has_those_bits(slots, dtype):
    rows, d = 520, 512                                        # 130 workgroups: the fewest that take eight columns a thread are 128
    gen = torch.Generator(device=DEV).manual_seed(slots)
    y = torch.randn((rows, slots, d), generator=gen, device=DEV).to(dtype)
    w = torch.rand((rows, slots), generator=gen, device=DEV)
    y[0, slots - 1], w[1, slots - 1] = float("inf"), float("nan")
    odd = torch.empty((rows * slots * d + 2,), dtype=dtype, device=DEV)[2:].view(rows, slots, d).copy_(y)
    got, want = moe.combine(y, w), moe.combine(odd, w)
    assert torch.equal(torch.nan_to_num(got.float()), torch.nan_to_num(want.float())) and bool(torch.isfinite(got[2:]).all())
