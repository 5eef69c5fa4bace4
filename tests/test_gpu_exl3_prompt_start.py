"""The launch that rotates a prompt's inputs and decodes the weight against the two launches: every bit of both, and of the
product behind them."""

import pytest
import torch

from tensorfold_amd import _lib, synthetic
from tensorfold_amd.exl3 import linear, prefill
from tests.test_gpu_exl3_prefill import DEV, layer_of

pytestmark = pytest.mark.gpu


# kt, nt: tiles of 16; one column block and an odd number of them, rows for less than a row of the grid, for many, and (2,100 x 1024
# inputs) past the count from which a workgroup takes 32 blocks
@pytest.mark.parametrize("codebook,bits,kt,nt,m", [("3inst", 3, 8, 8, 1), ("mcg", 4, 16, 24, 17), ("mul1", 2.5, 24, 8, 300),
                                                   ("3inst", 6, 64, 40, 129), ("mul1", 2, 64, 8, 2100), ("mcg", 8, 8, 136, 5)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_one_launch_has_the_bits_of_two(codebook, bits, kt, nt, m, dtype):
    layer = layer_of(codebook, bits, kt, nt, 11)[0]
    x = synthetic.activations(m, layer.k, 3).to(DEV).to(dtype)
    ws, ws2 = prefill.Workspace(), prefill.Workspace()
    out, out2 = (torch.empty((m, layer.n), dtype=torch.float16, device=DEV) for _ in range(2))
    prefill.matmul(layer, x, out, ws)
    xh = torch.empty((m, layer.k), dtype=torch.float16, device=DEV)
    _lib.call("tf_exl3_rot_in", x, linear._DTYPES[dtype], layer.suh, xh, m, layer.k)
    wt = prefill.decode(layer, ws2)
    assert torch.equal(ws.xh[:m * layer.k].view(torch.int16), xh.view(-1).view(torch.int16))
    assert torch.equal(ws.w[:layer.k * layer.n].view(torch.int16), wt.reshape(-1).view(torch.int16))
    assert torch.equal(prefill.matmul(layer, x, out2, ws2, wt), out) and torch.isfinite(out).all() and out.abs().max() > 0
