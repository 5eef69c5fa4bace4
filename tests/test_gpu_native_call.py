"""The calls that csrc/call.cpp makes as a whole against the general way (ctypes, torch's own allocations): the same results, and
whatever is not ordinary left to the general way, which copies or raises."""

import dataclasses

import pytest
import torch

from tensorfold_amd import _lib, build, glue, qmm, synthetic

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture
def general(monkeypatch):
    """Run a function with nothing native: every launch through ctypes."""

    _lib._start()

    def run(f):
        with monkeypatch.context() as m:
            m.setattr(_lib, "_native", {})
            return f()

    return run


def weight(n, k, gs, seed=1):
    return qmm.pack(*(t.to(DEV) for t in synthetic.affine_general(n, k, gs, seed)), gs)


def same(a, b):
    a, b = ([t] if isinstance(t, torch.Tensor) else list(t) for t in (a, b))
    return len(a) == len(b) and all(x.shape == y.shape and x.dtype == y.dtype and x.is_contiguous() and torch.equal(x, y)
                                    for x, y in zip(a, b))


def test_the_built_library_is_what_runs():
    assert build.call_lib() is not None and set(_lib.WHOLE) < set(_lib._start())


@pytest.mark.parametrize("gs", [32, 64])
@pytest.mark.parametrize("m", [1, 8, 9, 40])
def test_results(general, m, gs):
    k = 1024
    qs = [weight(n, k, gs, n) for n in (4096, 65, 640)]
    wide = synthetic.activations(m, k + 8, m).to(DEV)
    r, w = synthetic.activations(m, k, 5).to(DEV), synthetic.activations(1, k, 6).to(DEV)[0].contiguous()
    for x in (wide[:, :k].contiguous(), wide[:, 8:]):
        xs = qmm.group_sums(x, gs)
        for f32 in (False, True):
            for q in qs:
                assert _lib.whole("matmul", x, q, 1, f32) is not None
                for f in (lambda: qmm.matmul(x, q, f32=f32), lambda: qmm.matmul(x, q, f32=f32, sk=2),
                          lambda: qmm.prefill_matmul(x, q, f32=f32), lambda: qmm.prefill_matmul(x, q, f32=f32, tile=8)):
                    assert same(f(), general(f)), (q.n, f32)
            group = lambda: qmm.matmul_group(x, qs, xs, f32=f32)
            assert _lib.whole("matmul_group", x, xs, qs, [1, 1, 1], f32) is not None and same(group(), general(group)), f32
            assert not any(q.counters.any() for q in qs)
    x = wide[:, :k].contiguous()
    norm = lambda: glue.add_rmsnorm(x, r, w, 1e-6, gs)
    assert _lib.whole("add_rmsnorm", x, r, w, 1e-6, gs) is not None and same(norm(), general(norm))


def test_what_is_not_ordinary_goes_the_general_way(general):
    k, gs = 512, 64
    q, other = weight(130, k, gs), weight(130, k + 64, gs)
    x, xs = synthetic.activations(3, k, 1).to(DEV), None
    odd_start = torch.zeros((3, k + 1), dtype=torch.bfloat16, device=DEV)[:, 1:].copy_(x)       # rows off 16 bytes
    columns = x.t().contiguous().t()
    for bad in (odd_start, columns, x.half(), x.cpu(), x[0], x[:, :k - 64]):
        assert _lib.whole("matmul", bad, q, 1, False) is None and _lib.whole("prefill_matmul", bad, q, False, 0) is None
    for copied in (odd_start, columns):
        assert same(qmm.matmul(copied, q), qmm.matmul(x, q)) and same(qmm.prefill_matmul(copied, q), qmm.prefill_matmul(x, q))
    for bad, error in ((x.half(), ValueError), (x[0], ValueError), (x[:, :k - 64], ValueError), (x.cpu(), RuntimeError)):
        for f in (lambda: qmm.matmul(bad, q), lambda: qmm.prefill_matmul(bad, q)):
            with pytest.raises(error):
                f()
    xs = qmm.group_sums(x, gs)
    for bad in ([q, q], [q, other], [q] * 5, (q,), [None], []):
        assert _lib.whole("matmul_group", x, xs, bad, [1] * len(bad), False) is None
    for bad in (xs.half(), xs[:2], xs.t().contiguous().t(), xs.cpu()):
        assert _lib.whole("matmul_group", x, bad, [q], [1], False) is None
    # strided scales: taken as they lie by the decode form, copied for the prompt's
    wide = lambda t: torch.cat([t] * 2, 1)[:, :t.shape[1]]
    ragged = dataclasses.replace(q, scales=wide(q.scales), biases=wide(q.biases))
    assert _lib.whole("prefill_matmul", x, ragged, False, 0) is None
    assert same(qmm.prefill_matmul(x, ragged), qmm.prefill_matmul(x, q)) and same(qmm.matmul(x, ragged), qmm.matmul(x, q))
    r, w = synthetic.activations(3, k, 2).to(DEV), synthetic.activations(1, k, 3).to(DEV)[0].contiguous()
    for args in ((x.t().contiguous().t(), r, w, 1e-6, 64), (x, r[:2], w, 1e-6, 64), (x, r, w.float(), 1e-6, 64),
                 (x, r, w, 1e-6, 48), (x, r.cpu(), w, 1e-6, 64), (x, r, w[:64], 1e-6, 64)):
        assert _lib.whole("add_rmsnorm", *args) is None
        with pytest.raises((ValueError, RuntimeError)):
            glue.add_rmsnorm(*args)
    with pytest.raises(RuntimeError, match="whole groups a slice"):                              # the library's own sentence
        qmm.matmul(x, q, sk=3)


def test_results_of_a_subclass_are_of_its_class():
    class Named(torch.Tensor):
        pass

    qs, x = [weight(130, 512, 64), weight(64, 512, 64)], synthetic.activations(3, 512, 1).to(DEV)
    r, w = synthetic.activations(3, 512, 2).to(DEV), synthetic.activations(1, 512, 3).to(DEV)[0].contiguous()
    named, xs = x.as_subclass(Named), qmm.group_sums(x, 64)
    for f in (lambda t: [qmm.matmul(t, qs[0])], lambda t: [qmm.prefill_matmul(t, qs[0])], lambda t: qmm.matmul_group(t, qs, xs),
              lambda t: list(glue.add_rmsnorm(t, r, w, 1e-6))[:2]):
        for got, want in zip(f(named), f(x), strict=True):
            assert type(got) is Named and type(want) is torch.Tensor and torch.equal(got.as_subclass(torch.Tensor), want)


def test_under_capture_and_on_another_stream():
    q, x = weight(640, 2048, 64), synthetic.activations(3, 2048, 4).to(DEV)
    want = qmm.matmul(x, q)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = qmm.matmul(x, q)
    for _ in range(3):
        got.zero_()
        graph.replay()
        assert torch.equal(got, want)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        y = qmm.matmul(x, q)
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(y, want)


def test_a_full_device_raises_torch_s_own_error():
    x = torch.zeros((1, 64), dtype=torch.bfloat16, device=DEV)
    assert "empties" in _lib._start()
    with pytest.raises(torch.OutOfMemoryError):                            # 4 PiB: refused as it is asked for
        _lib.empties(x, [(1 << 20, 1 << 30, True)])
    with pytest.raises(torch.OutOfMemoryError):
        qmm.matmul(x, weight(130, 64, 64), sk=1 << 30)


def test_numbers_past_32_bits_are_not_cut_down():
    q, x = weight(130, 512, 64), synthetic.activations(3, 512, 1).to(DEV)
    for sk in (2 ** 32 + 1, 2 ** 32 + 2):
        assert _lib.whole("matmul", x, q, sk, False) is None
        with pytest.raises(RuntimeError):                                  # a workspace of some terabytes, refused
            qmm.matmul(x, q, sk=sk)
    r, w = synthetic.activations(3, 512, 2).to(DEV), synthetic.activations(1, 512, 3).to(DEV)[0].contiguous()
    for gs in (2 ** 32 + 64, 2 ** 70):
        with pytest.raises(ValueError, match="whole groups"):
            glue.add_rmsnorm(x, r, w, 1e-6, gs)
