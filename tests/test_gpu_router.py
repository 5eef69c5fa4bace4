"""The router's logits at the edges of its kernels' tiles, against float64 products; a row's bits whatever the call."""

import pytest
import torch

from tensorfold_amd import moe, synthetic

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("rows,d,ne", [(1, 32, 1), (2, 96, 5), (16, 2688, 128), (17, 512, 129), (70, 2048, 513),
                                       (257, 2720, 33), (65, 64, 1024), (1030, 480, 513), (4096, 256, 145)])
def test_router_against_float64_and_row_by_row(rows, d, ne):
    x = synthetic.activations(rows, d, 3 * rows + d).to(DEV)
    r = synthetic.activations(ne, d, 5 * ne + d, scale=d ** -0.5).to(DEV)
    got = moe.router(x, r)
    want = x.double() @ r.double().t().contiguous()
    # d products of bf16 values, exact in fp32, added in fp32: each addition rounds by at most 2^-24 of a partial sum
    bound = d * 2.0 ** -23 * (x.double().abs() @ r.double().abs().t().contiguous())
    assert bool(((got.double() - want).abs() <= bound).all())
    for at in {0, rows // 2, rows - 1}:
        assert torch.equal(moe.router(x[at:at + 1], r)[0], got[at])
    part = rows - rows // 3
    assert torch.equal(moe.router(x[:part], r), got[:part])


# slices of 2 to 28 chunks: fewer than a workgroup requests together, as many, and one to a few more (each tile's kernel)
@pytest.mark.parametrize("rows,d,ne", [(32, 512, 128), (8, 896, 16), (40, 2080, 64), (8, 4096, 128), (3, 7168, 17),
                                       (300, 736, 513), (290, 1504, 257), (777, 1056, 513), (530, 3104, 500)])
def test_slices_of_any_length(rows, d, ne):
    test_router_against_float64_and_row_by_row(rows, d, ne)


# the edges between the kernels that the rows and experts choose: many rows of few experts, and either side of where the
# wide kernel starts (512 workgroups of 32 x 64)
@pytest.mark.parametrize("rows,d,ne", [(16390, 96, 8), (16400, 352, 16), (33000, 64, 1), (16385, 160, 17), (16400, 512, 32),
                                       (4100, 256, 128), (4096, 512, 129), (1055, 288, 513), (5460, 96, 145),
                                       (5471, 352, 180), (8192, 128, 128), (8193, 288, 128)])
def test_many_rows_of_few_experts(rows, d, ne):
    test_router_against_float64_and_row_by_row(rows, d, ne)


# 32 x 16 tiles, a compute unit each: from the first call past 256 tiles of 16 x 16 to 256 such tiles and one more; slices that
# are requested in one go, and in two
@pytest.mark.parametrize("rows,d,ne", [(257, 2688, 241), (513, 2048, 113), (1024, 2080, 128), (1025, 352, 128), (8192, 64, 9),
                                       (8193, 64, 9), (17, 4096, 2044), (250, 3104, 500), (4000, 32, 17)])
def test_tiles_of_32_rows_and_16_experts(rows, d, ne):
    test_router_against_float64_and_row_by_row(rows, d, ne)
