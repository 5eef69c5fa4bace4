"""ctypes prototypes of ``include/tfmi.h`` and the call helper every op goes through."""

from __future__ import annotations

import contextlib
import ctypes
import threading
from ctypes import c_float, c_int, c_int64, c_void_p
from functools import lru_cache
from pathlib import Path

import torch

from . import build

P, I, L, F = c_void_p, c_int, c_int64, c_float

# name -> argument types, in the header's order (the trailing stream included)
PROTOTYPES = {
    "tf_qmm_pack": [P, P, P, I, I, I, P, P, P, P],
    "tf_qmm_unpack": [P, P, P, I, I, I, P, P, P, P],
    "tf_group_sums": [P, L, I, I, I, P, P],
    "tf_qmm": [P, L, P, P, P, P, L, P, P, P, I, I, I, I, I, I, I, I, I, P],
    "tf_qmm_own_sums": [P, L, P, P, P, L, P, P, P, I, I, I, I, I, I, I, I, I, P],
    "tf_qmm_static": [P, L, P, P, P, P, L, P, I, I, I, I, I, I, I, P],
    "tf_qmm_group": [P, L, P, I, P, P, P, P, P, P, P, P, P, P, I, I, I, I, I, P],
    "tf_qmm_prompt_tile": [I, I, I],
    "tf_qmm_prompt_rows": [I, I],
    "tf_qmm_prompt_row_tiles": [I, I],
    "tf_qmm_prefill": [P, L, P, P, P, P, I, I, I, I, I, I, I, P],
    "tf_quantize_rows": [P, L, I, I, I, P, P, P, P],
    "tf_qmm_prefill8": [P, P, P, P, P, P, P, I, I, I, I, I, I, P],
    "tf_experts_pack": [P, P, P, I, I, I, I, P, P],
    "tf_experts_unpack": [P, L, I, I, I, I, P, P, P, P],
    "tf_experts_plan": [P, L, I, I, P, P, P, P, P, P],
    "tf_experts_run": [I, I, P, L, I, P, I, I, P, P, P, P, I, F, L, P],
    "tf_experts_run_desc": [I, I, P, L, I, P, I, I, P, P, P, I, F, L, P],
    "tf_experts_prefill": [I, I, P, L, I, P, I, I, P, P, P, P, I, F, L, I, I, P],
    "tf_moe_route_up": [P, L, I, I, I, I, I, I, P, L, P, I, I, P, P, P, P, P, P, P, F, I, P, I, P],
    "tf_moe_down_combine": [I, P, I, I, P, I, I, P, P, P, P, P, I, P],
    "tf_moe_decode_sliced": [P, L, I, I, I, I, I, I, P, L, P, P, I, I, P, P, P, P, P, P, P, P, P, P, P, F, I, P],
    "tf_moe_route_decode": [P, L, I, I, I, I, P, P, P, P, P, P, P, I, P],
    "tf_moe_decode_experts": [I, I, P, L, I, I, P, P, I, I, P, P, P, P, P, P, P, P, P, F, I, P],
    "tf_moe_router": [P, L, P, P, I, I, I, P],
    "tf_moe_topk": [P, L, I, I, I, I, P, P, P],
    "tf_moe_combine": [P, I, P, P, I, I, I, P],
    "tf_exl3x_rot_in": [P, I, L, P, P, P, P, P, I, I, I, I, P],
    "tf_exl3x_grouped": [P, P, P, P, P, P, P, P, P, P, I, I, I, I, I, I, I, I, P],
    "tf_exl3x_gateup_epilogue": [P, P, P, P, P, P, I, I, I, I, F, I, P],
    "tf_exl3x_down_combine": [P, P, P, P, P, P, I, I, I, I, I, P],
    "tf_exl3x_plan_rot_in": [P, I, L, P, P, P, P, P, I, I, I, I, I, P, P, P, P],
    "tf_add_norm": [P, P, I, P, I, I, P, F, P, P, P, I, I, I, P],
    "tf_exl3_rot_in": [P, I, P, P, I, I, P],
    "tf_exl3_linear": [P, P, L, L, P, P, P, I, P, P, I, I, I, I, I, I, I, P],
    "tf_exl3_rot_in_stacked": [P, I, P, P, I, I, I, P],
    "tf_exl3_linear_stacked": [P, P, L, L, L, P, P, P, I, P, P, I, I, I, I, I, I, I, I, P],
    "tf_exl3_gate_up": [P, P, L, L, L, P, P, P, I, P, P, P, P, I, I, I, I, I, I, I, P],
    "tf_exl3_swiglu_rot_in": [P, I, P, P, I, I, P],
    "tf_exl3_unpack": [P, P, I, I, L, L, I, I, P],
    "tf_exl3_unpack_k8": [P, P, I, I, L, L, I, I, P],
    "tf_exl3_rot_in_unpack_k8": [P, I, P, P, I, P, P, I, I, L, L, I, I, P],
    "tf_exl3_gemm_tile": [I, I],
    "tf_exl3_gemm": [P, P, P, P, P, I, L, I, I, I, P],
}


def _declare(so: ctypes.CDLL) -> ctypes.CDLL:
    so.tf_last_error.restype = ctypes.c_char_p
    so.tf_last_error.argtypes = []
    so.tf_version.restype = c_int
    so.tf_check_device.restype = c_int
    for name, args in PROTOTYPES.items():
        fn = getattr(so, name)
        fn.argtypes = args
        fn.restype = c_int
    return so


@lru_cache(maxsize=1)
def lib() -> ctypes.CDLL:
    return _declare(build.load())


_other: ctypes.CDLL | None = None


@contextlib.contextmanager
def through(path):
    """Route ``call`` through another build of the library (the timeline build) inside the block; yields it.  The
    other build must carry the digest of the sources beside it: one built before an entry point changed its
    arguments would be called with shifted pointers."""

    global _other
    if not Path(path).exists():
        raise RuntimeError(f"tensorfold-amd: {path} is missing (build.timeline_lib() builds the timeline library)")
    if build.built_id(Path(path)) != build.source_id():
        raise RuntimeError(f"tensorfold-amd: {path} was built from other sources than the ones beside it")
    _other = _declare(ctypes.CDLL(str(path)))
    try:
        yield _other
    finally:
        _other = None


@lru_cache(maxsize=1)
def _ready() -> bool:
    """First GPU call: the device must be the one the kernels were built for."""

    if not torch.cuda.is_available():
        raise RuntimeError("tensorfold-amd: its kernels run on an MI355X GPU only; none is available "
                           "(there is no CPU path)")
    so = lib()
    if so.tf_check_device():
        raise RuntimeError(so.tf_last_error().decode())
    return True


def ptr(t: torch.Tensor | None) -> int | None:
    return None if t is None else t.data_ptr()


def stream() -> int:
    # the handle of torch.cuda.current_stream() without the Stream object around it: every launch asks for it.  The two
    # names are torch's own and not public: a build that lacks them is asked the public way
    try:
        return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())
    except AttributeError:
        return torch.cuda.current_stream().cuda_stream


_native: dict | None = None          # entry point -> its Python function of csrc/call.cpp; empty where that is not built


def _bound() -> dict:
    """The functions of ``tfmi_call.so``, bound to the library that ``lib`` has loaded; none where it cannot be had."""

    from importlib.machinery import ExtensionFileLoader
    from importlib.util import module_from_spec, spec_from_loader

    path = build.call_lib()
    if path is None:
        return {}
    loader = ExtensionFileLoader("tfmi_call", str(path))
    try:
        module = module_from_spec(spec_from_loader("tfmi_call", loader))
        loader.exec_module(module)
        module.bind(str(build.LIB))
    except (ImportError, RuntimeError) as e:          # not loadable here: the kernels do not need it
        build.say(f"{e}: launches go through ctypes, a few microseconds slower")
        return {}
    return {name: getattr(module, name) for name in (*PROTOTYPES, "empties", *WHOLE) if hasattr(module, name)}


_starting = threading.Lock()


def _start() -> dict:
    """The first call's part: the device looked at and the native functions bound, once whatever threads ask."""

    global _native
    with _starting:
        if _native is None:
            _ready()
            _native = _bound()
        return _native


def empties(x: torch.Tensor, sizes: list[tuple[int, int, bool]]) -> list[torch.Tensor]:
    """Uninitialised tensors [rows, columns] on x's device, of its type or fp32, one for each (rows, columns, fp32?); of
    x's class where that is a subclass."""

    make = (_native if _native is not None else _start()).get("empties")
    if make is not None and type(x) in (torch.Tensor, torch.nn.Parameter):
        return make(x, sizes)
    return [x.new_empty((r, c), dtype=torch.float32) if wide else x.new_empty((r, c)) for r, c, wide in sizes]


# calls that csrc/call.cpp makes as a whole where every argument is the ordinary one
WHOLE = ("matmul", "matmul_group", "prefill_matmul", "add_rmsnorm")


def whole(name: str, *args):
    """What ``name`` of ``WHOLE`` returns, launch and all, or None: some argument wants the general way."""

    if _native is None:
        if not (isinstance(args[0], torch.Tensor) and args[0].is_cuda):
            return None
        _start()
    make = _native.get(name)
    return None if make is None or _other is not None else make(*args, stream())


def call(name: str, *args) -> None:
    """Run entry point ``name`` on the current stream; a non-zero status raises with the library's sentence.  A pointer
    is a tensor, an address or None; where the entry point takes a table (of pointers, strides or counts) a list."""

    entry = (_native if _native is not None else _start()).get(name)
    if entry is not None and _other is None:
        entry(*args, stream())
        return
    so, kinds = _other or lib(), TABLES.get(name, {})
    # (a tensor of one number may stand for a whole number: only where a pointer belongs is it an address)
    plain = lambda a, kind: a.data_ptr() if kind is P and isinstance(a, torch.Tensor) else a
    args = [(kinds[i] * len(a))(*(plain(t, kinds[i]) for t in a)) if i in kinds and isinstance(a, list) else plain(a, kind)
            for i, (a, kind) in enumerate(zip((*args, stream()), PROTOTYPES[name], strict=True))]
    if getattr(so, name)(*args):
        raise RuntimeError(so.tf_last_error().decode())


# the element types of an entry point's tables, by argument, for the ctypes path
TABLES = {"tf_qmm_group": {4: c_void_p, 5: c_void_p, 6: c_void_p, 7: c_int64, 8: c_void_p, 9: c_void_p, 10: c_void_p,
                           11: c_int, 12: c_int, 13: c_int}}


def on_gpu(*tensors: torch.Tensor) -> None:
    for t in tensors:
        if t is not None and not t.is_cuda:
            raise RuntimeError("tensorfold-amd: expected a GPU tensor (its kernels have no CPU path)")
