"""The decode matmul's rows on the matrix instruction: every row tile's edges against float64, groups fewer than the
waves that share them, and a row's infinity kept to its row."""

import pytest
import torch

from tensorfold_amd import qmm, synthetic

pytestmark = pytest.mark.gpu
DEV = "cuda"


def exact(x, w, gs):
    words, scales, biases = (t.to(DEV) for t in w)
    n, k8 = words.shape
    codes = ((words[:, :, None] >> (4 * torch.arange(8, device=DEV))) & 15).reshape(n, 8 * k8 // gs, gs).double()
    weight = (codes * scales.double()[:, :, None] + biases.double()[:, :, None]).reshape(n, 8 * k8)
    size = (codes * scales.double().abs()[:, :, None] + biases.double().abs()[:, :, None]).reshape(n, 8 * k8)
    return x.double() @ weight.t().contiguous(), x.double().abs() @ size.t().contiguous()


@pytest.mark.parametrize("n,k,gs", [(1, 32, 32), (70, 64, 64), (64, 192, 64), (129, 4992, 32), (512, 2048, 64)])
def test_rows_against_float64(n, k, gs):
    w = synthetic.affine_general(n, k, gs, n + 3 * k)
    q = qmm.pack(*(t.to(DEV) for t in w), gs)
    x = synthetic.activations(49, k, n).to(DEV)
    want, size = exact(x, w, gs)
    # products of a bf16 input and a whole code are exact in fp32; k / gs group terms, gs inputs and the group sums are
    # added in fp32, each step rounding by at most 2^-24 of a partial sum no larger than `size`
    bound = (k // gs + 2 * gs + 24) * 2.0 ** -24 * size
    for m in (1, 3, 4, 5, 8, 9, 16, 17, 32, 33, 49):
        got = qmm.matmul(x[:m], q, f32=True)
        assert bool(((got.double() - want[:m]).abs() <= bound[:m]).all()), m
        assert torch.equal(qmm.matmul(x[:m], q), got.bfloat16()), m


def test_a_rows_infinity_stays_in_its_row():
    q = qmm.pack(*(t.to(DEV) for t in synthetic.affine_general(130, 256, 64, 5)), 64)
    x = synthetic.activations(20, 256, 6).to(DEV)
    for m in (3, 7, 20):
        want = qmm.matmul(x[:m], q)
        y = x[:m].clone()
        y[1, 100] = float("inf")
        got = qmm.matmul(y, q)
        others = [r for r in range(m) if r != 1]
        assert torch.equal(got[others], want[others]) and not torch.isfinite(got[1]).any()
