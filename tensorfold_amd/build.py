"""Build and load ``libtfmi.so``: hipcc for gfx950, nothing else (the counterpart of the reference's cuda/build.py).

The reference JIT-builds one pybind11 module per kernel family for whatever NVIDIA GPU is present and refuses GPUs
under compute capability 8.9 (cuda/build.py:20-69).  Here one shared library with a C ABI is compiled ahead of
time, in the tree, for the one target this package supports, and a GPU that is not gfx950 is refused by name.
"""

from __future__ import annotations

import contextlib
import ctypes
import os
import shutil
import subprocess
import sys
import tempfile
from functools import lru_cache
from pathlib import Path

ARCH = "gfx950"
HERE = Path(__file__).resolve().parent
CSRC = HERE / "csrc"
LIB = HERE / "libtfmi.so"
TIMELINE_LIB = HERE / "libtfmi_timeline.so"      # the same kernels with per-workgroup timestamps (see compile)
SOURCES = ("api.hip", "pack.hip", "decode.hip", "fused.hip", "route.hip", "norm.hip", "prefill.hip", "prefill8.hip", "exl3.hip", "exl3_experts.hip")
CALL_LIB = HERE / "tfmi_call.so"                 # the entry points as Python functions (csrc/call.cpp); host code alone
# NDEBUG: without it pybind11 (under torch's headers) brings a thread-local counter, and a library with thread-local storage
# that is loaded late and never touches its own puts every other library's access to theirs on glibc's slow path (before 2.39):
# a torch.randint and a conversion take 22.7 us beside such a tfmi_call.so, 20.3 without
CALL_FLAGS = ("-O2", "-DNDEBUG", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden")
# packed-fp32 VALU forms are switched off for the device pass (the host pass warns that it does not know the feature)
FLAGS = ("-O3", "-std=c++17", "-fPIC", "-shared", f"--offload-arch={ARCH}",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops")


def say(text: str) -> None:
    print(f"[tensorfold-amd] {text}", file=sys.stderr, flush=True)


def hipcc() -> str | None:
    return shutil.which("hipcc") or (str(Path("/opt/rocm/bin/hipcc")) if Path("/opt/rocm/bin/hipcc").exists() else None)


def source_id() -> str:
    """16 hex digits over every file the library is built from and the compiler flags."""

    import hashlib

    h = hashlib.sha256(" ".join(FLAGS).encode())
    for path in [CSRC / s for s in SOURCES] + sorted(CSRC.glob("*.h")) + [HERE.parent / "include" / "tfmi.h"]:
        h.update(path.name.encode())
        h.update(path.read_bytes())
    return h.hexdigest()[:16]


def call_for() -> str:
    """16 hex digits over what ``tfmi_call.so`` is built for: another Python or torch may lay out its objects otherwise."""

    import hashlib

    import torch

    return hashlib.sha256(f"{sys.version} {torch.__version__}".encode()).hexdigest()[:16]


def call_id() -> str:
    """16 hex digits over what ``tfmi_call.so`` is built from and for."""

    import hashlib

    h = hashlib.sha256(f"{call_for()} {CALL_FLAGS}".encode())
    for path in (CSRC / "call.cpp", HERE.parent / "include" / "tfmi.h"):
        h.update(path.read_bytes())
    return h.hexdigest()[:16]


def built_id(path: Path = LIB, mark: bytes = b"TFMI_BUILD_ID=") -> str | None:
    """The digest a library file carries (``tf_build_id``), read from the file without loading it."""

    if not path.exists():
        return None
    blob = path.read_bytes()
    at = blob.find(mark)
    return None if at < 0 else blob[at + len(mark):at + len(mark) + 16].decode(errors="replace")


@contextlib.contextmanager
def beside(target: Path):
    """Where to write ``target``'s next version: it takes the old one's place in one step at the block's end, so that other
    processes (ranks that find it out of date all build it) load the whole old file or the whole new one."""

    with tempfile.TemporaryDirectory(dir=target.parent, prefix=".tfmi-build-") as tmp:
        made = Path(tmp) / target.name
        yield made
        os.replace(made, target)


def stale() -> bool:
    """Whether the library is missing or was built from other sources than the ones beside it."""

    if LIB.exists() and not (CSRC / SOURCES[0]).exists():
        return False                       # a library shipped without its sources is taken as it is
    return built_id() != source_id()


def timeline_lib() -> Path:
    """``libtfmi_timeline.so`` for the sources beside it: built on request only (``bench_configs.py timeline*`` asks),
    and again whenever its digest is not the sources'.  A timeline build of other sources is never loaded: its entry
    points may take other arguments than the prototypes of this tree."""

    if built_id(TIMELINE_LIB) != source_id():
        if hipcc() is None:
            raise RuntimeError(f"tensorfold-amd: {TIMELINE_LIB} is missing or was built from other sources, and there "
                               "is no hipcc to build it")
        compile(timeline=True)
    return TIMELINE_LIB


def compile(verbose: bool = False, timeline: bool = False) -> Path:
    """Compile every kernel for gfx950 into ``libtfmi.so`` (cross-compiles without a GPU): one hipcc per source,
    side by side, then a link.  ``timeline``: the same sources with -DTF_TIMELINE into ``libtfmi_timeline.so``, whose
    decode expert kernels note per-workgroup timestamps (an instrument: only ``timeline_lib`` builds it)."""

    from concurrent.futures import ThreadPoolExecutor

    cc = hipcc()
    if cc is None:
        raise RuntimeError("tensorfold-amd: hipcc was not found; ROCm's compiler is needed to build libtfmi.so")
    target = TIMELINE_LIB if timeline else LIB
    say(f"building {target.name} for {ARCH} (about half a minute)")
    noise = "packed-fp32-ops"

    def run(cmd: list[str]) -> str:
        done = subprocess.run(cmd, capture_output=True, text=True)
        err = "\n".join(line for line in done.stderr.splitlines() if noise not in line)
        if done.returncode:
            raise RuntimeError(f"tensorfold-amd: hipcc failed:\n{err}")
        return err

    compile_flags = [f for f in FLAGS if f != "-shared"] + [f'-DTF_BUILD_ID="{source_id()}"']
    if timeline:
        compile_flags.append("-DTF_TIMELINE")
    with tempfile.TemporaryDirectory(prefix="tfmi-build-") as tmp:
        objects = [str(Path(tmp) / (Path(s).stem + ".o")) for s in SOURCES]
        with ThreadPoolExecutor(max_workers=min(8, len(SOURCES))) as pool:
            logs = list(pool.map(lambda so: run([cc, *compile_flags, "-c", str(CSRC / so[0]), "-o", so[1]]),
                                 zip(SOURCES, objects)))
        with beside(target) as made:
            logs.append(run([cc, "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", str(made), *objects]))
    if verbose:
        for text in logs:
            if text:
                say(text)
    if not timeline:
        _try_call()
    return target


def compile_call() -> Path | None:
    """``tfmi_call.so`` with the host's C++ compiler; None where that, Python's headers or torch's are missing."""

    import sysconfig

    import torch

    cc, python, root = shutil.which("g++") or shutil.which("c++"), Path(sysconfig.get_paths()["include"]), Path(torch.__file__).parent
    if cc is None or not (python / "Python.h").exists() or not (root / "include/torch/csrc/autograd/python_variable.h").exists():
        return None
    with beside(CALL_LIB) as made:
        done = subprocess.run([cc, *CALL_FLAGS, f"-I{python}",
                               f"-I{root / 'include'}", f"-I{root / 'include/torch/csrc/api/include'}",
                               f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f'-DTF_CALL_ID="{call_id()}"',
                               f'-DTF_CALL_FOR="{call_for()}"',
                               str(CSRC / "call.cpp"), "-o", str(made), f"-L{root / 'lib'}", "-ltorch_python", "-ltorch_cpu",
                               "-lc10", "-ldl"], capture_output=True, text=True)
        if done.returncode:
            raise RuntimeError(f"tensorfold-amd: {cc} failed:\n{done.stderr}")
    return CALL_LIB


def _try_call() -> Path | None:
    """``compile_call`` where a failure (a compiler that cannot, a folder that is not written to) is said and not raised: the
    kernels do not need this library."""

    try:
        made, why = compile_call(), "no C++ compiler, Python headers or torch headers"
    except (RuntimeError, OSError) as e:
        made, why = None, str(e)
    if made is None:
        say(f"{why}: launches go through ctypes, a few microseconds slower")
    return made


def call_lib() -> Path | None:
    """``tfmi_call.so`` for the sources beside it, built first if it is missing or out of date; None where it cannot be
    (``_lib.call`` then goes through ctypes: the same launches, a few microseconds later)."""

    if not (CSRC / "call.cpp").exists():          # shipped without its sources: taken where it was built for this Python and torch
        return CALL_LIB if built_id(CALL_LIB, b"TFMI_CALL_FOR=") == call_for() else None
    return CALL_LIB if built_id(CALL_LIB, b"TFMI_CALL_ID=") == call_id() else _try_call()


@lru_cache(maxsize=1)
def load() -> ctypes.CDLL:
    """The library, built first if it is missing or out of date (its digest differs from the sources') and hipcc is
    here; a missing or stale library never falls back to anything."""

    if stale():
        if hipcc() is None:
            what = "is missing" if not LIB.exists() else "was built from other sources than the ones beside it"
            raise RuntimeError(f"tensorfold-amd: {LIB} {what} and there is no hipcc to build it; "
                               "run `python -c 'import __graft_entry__ as g; g.build()'` where ROCm is installed")
        compile()
    return ctypes.CDLL(str(LIB))


def refuse_other_gpu() -> None:
    """With a GPU present, refuse by name one the kernels were not built for (cuda/build.py:35-46 in spirit)."""

    import torch

    if not torch.cuda.is_available():
        return
    lib = load()
    lib.tf_last_error.restype = ctypes.c_char_p
    if lib.tf_check_device():
        raise ValueError(lib.tf_last_error().decode())
