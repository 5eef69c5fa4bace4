"""Decode matmuls of few rows without arrival counters: the bits of the call that has them, whichever form the launch
takes (a workgroup with all of K, or the slices and a reduce)."""

import ctypes

import pytest
import torch

from tensorfold_amd import _lib, qmm, synthetic

pytestmark = pytest.mark.gpu
DEV = "cuda"

# (columns, K, group size, slices): two, four and eight slices, slices of one to three groups (runs without one), runs of
# unequal length, a K and a width on either side of where the split launch takes over, a last tile of one column
SHAPES = [(64, 64, 32, 2), (65, 128, 32, 4), (130, 192, 32, 2), (1030, 256, 32, 8), (515, 768, 64, 4), (1024, 1024, 32, 8),
          (1000, 1024, 64, 2), (2048, 1536, 64, 4), (100, 1600, 32, 2), (8191, 3072, 64, 4), (8193, 3200, 64, 2),
          (16385, 512, 64, 4), (960, 1024, 32, 8)]


def weight(n, k, gs, seed):
    return qmm.pack(*(t.to(DEV) for t in synthetic.affine_general(n, k, gs, seed)), gs)


@pytest.mark.parametrize("n,k,gs,sk", SHAPES)
def test_without_counters_the_same_bits(n, k, gs, sk):
    q = weight(n, k, gs, n + k)
    wide = synthetic.activations(8, k + 8, n).to(DEV)
    for m in (1, 2, 4, 5, 8):
        for x in (wide[:m, :k].contiguous(), wide[:m, :k]):
            xs = qmm.group_sums(x, gs)
            for f32 in (False, True):
                out = torch.full((m + 1, n), 7, device=DEV, dtype=torch.float32 if f32 else torch.bfloat16)
                part = torch.empty((sk, m, n), device=DEV)
                _lib.call("tf_qmm", x.data_ptr(), x.stride(0), xs.data_ptr(), q.weight.data_ptr(), q.scales.data_ptr(),
                          q.biases.data_ptr(), q.scales.stride(0), out.data_ptr(), part.data_ptr(), None, 0, m, n, k, sk,
                          gs, 16, int(f32), 1)
                assert torch.equal(out[:m], qmm.matmul(x, q, xs, sk=sk, f32=f32)), (m, f32)
                assert bool((out[m] == 7).all())


@pytest.mark.parametrize("ns,k,gs,sks", [((512, 65, 130), 512, 32, (4, 4, 4)), ((1024, 515), 1024, 32, (8, 4)),
                                         ((64, 4100, 1000, 130), 1536, 64, (4, 4, 4, 4)), ((130, 65), 128, 32, (4, 4)),
                                         ((1000, 513), 1536, 32, (8, 8)), ((512, 512), 512, 64, (2, 4))])
def test_a_group_without_counters_the_same_bits(ns, k, gs, sks):
    qs = [weight(n, k, gs, n + k + i) for i, n in enumerate(ns)]
    count = len(ns)
    pointers = lambda ts: (ctypes.c_void_p * count)(*[t.data_ptr() for t in ts])
    ints = lambda v: (ctypes.c_int * count)(*v)
    at = ctypes.addressof
    for m in (1, 4, 5, 8):
        x = synthetic.activations(m, k, m).to(DEV)
        xs = qmm.group_sums(x, gs)
        outs = [torch.empty((m, n), device=DEV, dtype=torch.bfloat16) for n in ns]
        parts = [torch.empty((sk, m, n), device=DEV) for sk, n in zip(sks, ns)]
        tables = [pointers([q.weight for q in qs]), pointers([q.scales for q in qs]), pointers([q.biases for q in qs]),
                  (ctypes.c_int64 * count)(*[q.scales.stride(0) for q in qs]), pointers(outs), pointers(parts)]
        columns, slices = ints(ns), ints(sks)
        _lib.call("tf_qmm_group", x.data_ptr(), x.stride(0), xs.data_ptr(), count, *map(at, tables), None, None,
                  at(columns), at(slices), m, k, gs, 16, 0)
        for out, q, sk in zip(outs, qs, sks):
            assert torch.equal(out, qmm.matmul(x, q, xs, sk=sk)), m
