"""A grouped matmul's partial sums in one buffer of its own, in the caller's buffers, or some of each: the bits of separate
calls, at column counts whose parts do not end on a 256-byte step; and launches on the stream that is current."""

import pytest
import torch

from tensorfold_amd import _lib, qmm

pytestmark = pytest.mark.gpu
DEV = "cuda"


def weight(gen, n, k, gs):
    words = torch.randint(-2 ** 31, 2 ** 31, (n, k // 8), generator=gen, dtype=torch.int64).to(torch.int32)
    scales = (torch.rand((n, k // gs), generator=gen) * 0.02).bfloat16()
    return qmm.pack(words.to(DEV), scales.to(DEV), (scales.float() * -8).bfloat16().to(DEV), gs)


@pytest.mark.parametrize("rows", [1, 8, 9, 33])
@pytest.mark.parametrize("given", [(), (1,), (0, 2), (0, 1, 2)])
def test_parts_of_the_call_and_of_the_caller(rows, given):
    gen = torch.Generator().manual_seed(rows)
    k, gs = 1024, 32
    ws = [weight(gen, n, k, gs) for n in (513, 100, 65)]
    x = torch.randn((rows, k), generator=gen).bfloat16().to(DEV)
    sks = [qmm.split_k(w.n, k, gs) for w in ws]
    assert min(sks) > 1
    parts = [torch.empty((sk, rows, w.n), device=DEV) if i in given else None for i, (w, sk) in enumerate(zip(ws, sks))]
    want = [qmm.matmul(x, w) for w in ws]
    for _ in range(2):
        got = qmm.matmul_group(x, ws, parts=parts if given else None)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert all(torch.equal(a, b) for a, b in zip(qmm.matmul_group(x, ws, sks=[1, sks[1], 1], parts=parts),
                                                 [qmm.matmul(x, w, sk=sk) for w, sk in zip(ws, (1, sks[1], 1))]))


def test_the_current_stream():
    assert _lib.stream() == torch.cuda.current_stream().cuda_stream
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert _lib.stream() == side.cuda_stream
    assert _lib.stream() == torch.cuda.current_stream().cuda_stream
