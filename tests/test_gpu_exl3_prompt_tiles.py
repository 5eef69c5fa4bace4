"""The EXL3 prompt matmul's workgroup heights: every count of 16-row tiles a call can be given, odd and even, with a ragged
last row tile and a last 128-column block of its own, holds the rows that 31-row calls (two row tiles) give, bit for bit.
Those are checked against the float64 forward in test_gpu_exl3_prefill.py."""

import pytest
import torch

from tensorfold_amd import synthetic
from tensorfold_amd.exl3 import linear, prefill

pytestmark = pytest.mark.gpu
DEV = "cuda"


# rows x columns whose calls take 3, 4, 5, 6, 7, 8 and 9 row tiles a workgroup
@pytest.mark.parametrize("tiles,rows,n", [(3, 700, 4224), (4, 777, 4224), (5, 1000, 4224), (6, 1400, 4224), (7, 1000, 6272),
                                          (8, 1400, 5120), (9, 2050, 4224)])
def test_rows_do_not_depend_on_the_tile(tiles, rows, n):
    assert prefill.row_tiles(rows, n) == tiles and prefill.row_tiles(31, n) == 2
    trellis, suh, svh = synthetic.exl3_layer(256, n, 3, n)
    layer = linear.Exl3Linear.from_tensors(trellis, suh, svh, "3inst", device=DEV)
    layer.bias = torch.linspace(-1, 1, n, device=DEV).half()
    ws = prefill.Workspace()
    x = synthetic.activations(rows, 256, rows, dtype=torch.float16).to(DEV)
    whole = prefill.matmul(layer, x, torch.empty((rows, n), dtype=torch.float16, device=DEV), ws).clone()
    wt = prefill.decode(layer, ws)
    for r in range(0, rows, 31):
        part = x[r:r + 31]
        few = prefill.matmul(layer, part, torch.empty((len(part), n), dtype=torch.float16, device=DEV), ws, wt=wt)
        assert torch.equal(few, whole[r:r + 31]), r


@pytest.mark.parametrize("rows,k", [(1, 128), (3, 384), (130, 5120), (511, 1024), (900, 2560)])
def test_the_rotation_of_few_and_many_blocks(rows, k):
    """xh of the rotation launch (one block of 128 a group of lanes, or two, the second missing at the end) against the
    transform in float64 of the same fp16 products."""

    from tensorfold_amd import _lib

    x = synthetic.activations(rows, k, rows + k, dtype=torch.float32).to(DEV)
    suh = (torch.rand((k,), device=DEV) + 0.5).half()
    xh = torch.empty((rows, k), dtype=torch.float16, device=DEV)
    _lib.call("tf_exl3_rot_in", _lib.ptr(x), linear._DTYPES[x.dtype], _lib.ptr(suh), _lib.ptr(xh), rows, k)
    i = torch.arange(128)
    ones = torch.zeros((128, 128), dtype=torch.int64)
    for b in range(7):
        ones += ((i[:, None] >> b) & 1) * ((i[None, :] >> b) & 1)
    h = (1.0 - 2.0 * (ones % 2)).double().to(DEV) / 128 ** 0.5
    products = (x * suh.float()).double().view(rows, k // 128, 128)
    want = (products @ h).view(rows, k)
    # seven fp32 additions and a scaling, each off by at most 2^-24 of what it holds, then one rounding to fp16
    sums = (products.abs().sum(2, keepdim=True) / 128 ** 0.5).expand(-1, -1, 128).reshape(rows, k)
    assert torch.all((xh.double() - want).abs() <= want.abs() * 2 ** -11 + 2 ** -25 + 9 * 2 ** -24 * sums)
