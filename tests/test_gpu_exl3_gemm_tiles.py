"""The EXL3 prompt matmul's row tiles (32, 64, 96 or 128 rows a workgroup, chosen from rows and columns): a row has the
same bits whichever tile it falls in, at the edges of every tile, and the values of a float64 product."""

import math

import pytest
import torch

from tensorfold_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"


def gemm(x, w8, svh):
    m, k, n = x.shape[0], x.shape[1], w8.shape[1]
    y = torch.full((m + 1, n), 7.0, dtype=torch.float32, device=DEV)
    _lib.call("tf_exl3_gemm", x.data_ptr(), w8.data_ptr(), svh.data_ptr(), None, y.data_ptr(), 2, n, m, k, n)
    assert (y[m] == 7.0).all()                                   # nothing past the last row
    return y[:m]


# columns and rows at which the rule takes each tile, and the rows around a tile's edge
@pytest.mark.parametrize("n", [128, 1024, 3072, 5120, 9216])
def test_a_row_does_not_depend_on_the_tile(n):
    k, most = 256, 3000
    gen = torch.Generator(device=DEV).manual_seed(n)
    x = torch.randn((most, k), generator=gen, device=DEV).half()
    w8 = (torch.randn((k // 8, n, 8), generator=gen, device=DEV) * 0.05).half()
    svh = (torch.rand((n,), generator=gen, device=DEV) + 0.5).half()
    whole = gemm(x, w8, svh)
    for m in (1, 31, 32, 33, 63, 65, 95, 96, 97, 127, 128, 129, 333, 777, 1000, 1400, 2048):
        assert torch.equal(gemm(x[:m].contiguous(), w8, svh), whole[:m]), m
    dense = w8.permute(0, 2, 1).reshape(k, n).double()
    h = torch.tensor([[(-1.0) ** bin(i & j).count("1") for j in range(128)] for i in range(128)], device=DEV).double()
    rows = x[:200].double() @ dense
    want = (rows.view(200, n // 128, 128) @ h).reshape(200, n) / math.sqrt(128) * svh.double()
    # fp32 sums of k = 256 exact products and a 128-point butterfly: k 2^-24 at the worst, far less in the 2-norm
    assert (whole[:200].double() - want).norm() / want.norm() < 256 * 2.0 ** -24
