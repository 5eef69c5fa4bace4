"""The entry points as Python functions (csrc/call.cpp) against ctypes: the same names, argument counts, values and sentences,
without a GPU (what the library refuses before it launches)."""

import shutil

import numpy as np
import pytest
import torch

from tensorfold_amd import _lib, build

NATIVE = _lib._bound() if build.call_lib() else None
pytestmark = pytest.mark.skipif(NATIVE is None, reason="no C++ compiler, Python headers or torch headers")
QUERIES = {"tf_qmm_prompt_tile", "tf_qmm_prompt_rows", "tf_qmm_prompt_row_tiles", "tf_exl3_gemm_tile"}          # launch nothing: called on the library itself


def sentence(name, *args):
    with pytest.raises(RuntimeError) as caught:
        NATIVE[name](*args)
    assert getattr(_lib.lib(), name)(*[a.data_ptr() if isinstance(a, torch.Tensor) else a for a in args]) != 0
    assert _lib.lib().tf_last_error().decode() == str(caught.value)
    return str(caught.value)


def test_every_launch_is_there_with_its_arguments():
    assert set(NATIVE) - {"empties", *_lib.WHOLE} == set(_lib.PROTOTYPES) - QUERIES
    for name, args in _lib.PROTOTYPES.items():
        if name not in QUERIES:
            for given in (0, len(args) - 1, len(args) + 1):
                with pytest.raises(TypeError, match=f"takes {len(args)}"):
                    NATIVE[name](*[0] * given)


def test_values_arrive_as_ctypes_passes_them():
    x = torch.zeros((2, 64), dtype=torch.bfloat16)
    assert "not 48" in sentence("tf_group_sums", x, 64, 2, 64, 48, x, None)
    assert "16-byte" in sentence("tf_group_sums", x.data_ptr() + 2, 64, 2, 64, 64, x, None)          # an address
    assert "a multiple of the group" in sentence("tf_group_sums", None, 64, 2, 64, 64, x, None)      # no pointer
    assert "not -3" in sentence("tf_moe_topk", x, 64, 1, 64, -3, True, x, x, None)                   # signs and truth values
    # 64-bit strides, a float among the whole numbers, the last of many arguments
    assert "exceed the grid limit" in sentence("tf_experts_prefill", 64, 1, x, 1 << 40, 0, x, 1, 1, x, x, x, x, 32, 0.5, 1 << 40,
                                               64, 0, None)


@pytest.mark.parametrize("number", [np.int32, np.int64, np.uint16, torch.tensor])
@pytest.mark.parametrize("native", [True, False])
def test_whole_numbers_of_other_types_are_taken_as_ctypes_takes_them(monkeypatch, number, native):
    monkeypatch.setattr(_lib, "_native", NATIVE if native else {})
    monkeypatch.setattr(_lib, "stream", lambda: 0)
    x, w = torch.zeros((2, 64), dtype=torch.bfloat16), torch.zeros((64,), dtype=torch.int32)
    with pytest.raises(RuntimeError, match="not 48"):
        _lib.call("tf_group_sums", x, number(64), number(2), number(64), number(48), x)
    with pytest.raises(RuntimeError, match="whole groups a slice"):
        _lib.call("tf_qmm_group", x, 64, x, 1, [w], [w], [w], [number(128)], [w], [None], [None], [number(0)], [number(64)], [number(3)],
                  number(2), number(64), 64, 16, 0)


def test_tables_are_lists():
    x = torch.zeros((2, 64), dtype=torch.bfloat16)
    w = torch.zeros((64,), dtype=torch.int32)
    group = lambda ws, sks, gs: NATIVE["tf_qmm_group"](x, 64, x, len(ws), ws, ws, ws, [128] * len(ws), ws, [None] * len(ws),
                                                       [None] * len(ws), [0] * len(ws), [64] * len(ws), sks, 2, 64, gs, 16, 0, None)
    for ws, sks, gs, text in (([w], [1], 48, "groups of 32 or 64"), ([w] * 5, [1] * 5, 64, "1 to 4 weights, not 5"),
                              ([w, None], [1, 1], 64, "null pointer"), ([w, w], [1, 3], 64, "whole groups a slice"),
                              ([w, w], [1, 70000], 64, "whole groups a slice")):
        with pytest.raises(RuntimeError, match=text):
            group(ws, sks, gs)
    with pytest.raises(TypeError, match="longer list"):
        group([w] * 9, [1] * 9, 64)


@pytest.mark.parametrize("bad", [1.5, "1", (1,), object()])
def test_what_is_no_number_and_no_tensor_is_refused(bad):
    x = torch.zeros((2, 64), dtype=torch.bfloat16)
    for args in ((bad, 64, 2, 64, 64, x, None), (x, bad, 2, 64, 64, x, None)):
        with pytest.raises(TypeError):
            NATIVE["tf_group_sums"](*args)


def test_empties():
    x = torch.zeros((2, 64), dtype=torch.bfloat16)
    made = NATIVE["empties"](x, [(3, 5, False), (2, 7, True), (0, 4, 0)])
    assert [(tuple(t.shape), t.dtype, t.is_contiguous(), t.requires_grad) for t in made] == \
        [((3, 5), torch.bfloat16, True, False), ((2, 7), torch.float32, True, False), ((0, 4), torch.bfloat16, True, False)]
    for bad in ((x, [(1, 2)]), (x, [(-1, 2, 0)]), (x, 3), (3, []), (x,)):
        with pytest.raises((TypeError, RuntimeError)):
            NATIVE["empties"](*bad)


def test_results_of_a_subclass_are_of_its_class(monkeypatch):
    class Named(torch.Tensor):
        pass

    monkeypatch.setattr(_lib, "_native", NATIVE)
    x = torch.zeros((2, 64), dtype=torch.bfloat16)
    for given, kind in ((x, torch.Tensor), (torch.nn.Parameter(x), torch.Tensor), (x.as_subclass(Named), Named)):
        for made, dtype in zip(_lib.empties(given, [(3, 5, False), (2, 7, True)]), (torch.bfloat16, torch.float32)):
            assert type(made) is kind and made.dtype == dtype and not made.requires_grad


def test_a_tensor_without_storage_raises():
    x = torch.zeros((2, 64), dtype=torch.bfloat16)
    nowhere = torch.empty((2, 64), dtype=torch.bfloat16, device="meta")          # torch hands out an address of 0
    for args in ((nowhere, 64, 2, 64, 64, x, None), (x, 64, 2, 64, 64, nowhere, None)):
        assert "x must be" in sentence("tf_group_sums", *args)
    for args in ((x.to_sparse(), 64, 2, 64, 64, x, None), (x, 64, 2, 64, 64, x.to_sparse(), None)):
        with pytest.raises(RuntimeError, match="storage"):
            NATIVE["tf_group_sums"](*args)


def test_what_an_allocation_raises_keeps_its_type():
    class Elsewhere(torch.Tensor):
        __torch_dispatch__ = classmethod(lambda *_: None)

    # a device that this torch has no allocator for: torch.empty raises NotImplementedError, a type of torch's own in C++
    x = torch.Tensor._make_wrapper_subclass(Elsewhere, (2, 64), dtype=torch.bfloat16, device="vulkan")
    with pytest.raises(NotImplementedError):
        torch.empty((2, 64), device="vulkan")
    with pytest.raises(NotImplementedError):
        NATIVE["empties"](x, [(2, 64, False)])


@pytest.mark.parametrize("gs", [2 ** 70, -2 ** 70, 2 ** 40])
def test_a_whole_call_leaves_numbers_past_32_bits_to_the_general_way(gs):
    x, w = torch.zeros((2, 64), dtype=torch.bfloat16), torch.zeros((64,), dtype=torch.bfloat16)
    assert NATIVE["add_rmsnorm"](x, x, w, 1e-6, gs, 0) is None


WATCH = """
#include <Python.h>
#include <c10/core/CPUAllocator.h>
struct Watch : c10::Allocator {
  c10::Allocator* inner = c10::GetCPUAllocator();
  int held = 0, calls = 0;
  c10::DataPtr allocate(size_t n) override { return ++calls, held += PyGILState_Check(), inner->allocate(n); }
  void copy_data(void* to, const void* from, size_t n) const override { inner->copy_data(to, from, n); }
};
static Watch watch;
extern "C" void begin() { c10::SetCPUAllocator(&watch, 100); }
extern "C" int calls() { return watch.calls; }
extern "C" int held() { c10::SetCPUAllocator(watch.inner, 100); return watch.held; }
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no C++ compiler")
def test_other_threads_go_on_while_memory_is_allocated(tmp_path):
    import ctypes
    import subprocess
    import sysconfig
    from pathlib import Path

    root = Path(torch.__file__).parent
    (tmp_path / "watch.cpp").write_text(WATCH)
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
                    f"-I{sysconfig.get_paths()['include']}", f"-I{root / 'include'}", str(tmp_path / "watch.cpp"), "-o",
                    str(tmp_path / "watch.so"), f"-L{root / 'lib'}", "-lc10"], check=True, capture_output=True)
    watch, x = ctypes.PyDLL(str(tmp_path / "watch.so")), torch.zeros((2, 64), dtype=torch.bfloat16)
    watch.begin()
    try:
        made = NATIVE["empties"](x, [(3, 64, False), (2, 5, True)])
        calls = watch.calls()
    finally:
        held = watch.held()
    assert len(made) == calls == 2 and held == 0


def test_the_module_has_no_thread_local_storage():
    import struct

    image = build.CALL_LIB.read_bytes()
    at, size, count = struct.unpack_from("<Q", image, 0x20)[0], *struct.unpack_from("<HH", image, 0x36)          # ELF64 program headers
    kinds = [struct.unpack_from("<I", image, at + i * size)[0] for i in range(count)]
    assert 1 in kinds and 7 not in kinds          # PT_LOAD, PT_TLS


def test_threads_that_start_together_bind_it_once(monkeypatch):
    import threading
    import time

    bound = []
    monkeypatch.setattr(_lib, "_ready", lambda: True)
    monkeypatch.setattr(_lib, "_native", None)
    monkeypatch.setattr(_lib, "_bound", lambda: (bound.append(1), time.sleep(0.05), dict(NATIVE))[2])
    got = []
    threads = [threading.Thread(target=lambda: got.append(_lib._start())) for _ in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(bound) == 1 and len(got) == 6 and all(g is got[0] for g in got)
