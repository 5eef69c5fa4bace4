"""How the two libraries come to be built, with the compilers stood in for (nothing is compiled here)."""

import subprocess
from pathlib import Path

import pytest

from tensorfold_amd import build


@pytest.fixture
def tree(tmp_path, monkeypatch):
    """The libraries of an older build in a folder of their own, and a compiler that does what the test says."""

    class Tree:
        kernels, call, ran = tmp_path / "libtfmi.so", tmp_path / "tfmi_call.so", []
        status, during = 0, staticmethod(lambda output: None)

    def run(cmd, **_):
        Tree.ran.append(cmd)
        output = Path(cmd[cmd.index("-o") + 1])
        Tree.during(output)
        if not Tree.status:
            output.write_bytes(b"new")
        return subprocess.CompletedProcess(cmd, Tree.status, "", "no such luck")

    Tree.ran = []
    for path in (Tree.kernels, Tree.call):
        path.write_bytes(b"old")
    monkeypatch.setattr(build, "LIB", Tree.kernels)
    monkeypatch.setattr(build, "CALL_LIB", Tree.call)
    monkeypatch.setattr(build, "hipcc", lambda: "hipcc")
    monkeypatch.setattr(build.shutil, "which", lambda name: name)
    monkeypatch.setattr(build.subprocess, "run", run)
    return Tree


def test_a_library_takes_its_place_whole(tree):
    """While it is linked the old file is there for whoever loads it; a link that fails leaves the old file and nothing else."""

    seen = []
    tree.during = lambda output: seen.append((output.name, tree.kernels.read_bytes(), tree.call.read_bytes()))
    build.compile()
    assert ("libtfmi.so", b"old", b"old") in seen and ("tfmi_call.so", b"new", b"old") in seen
    assert tree.kernels.read_bytes() == tree.call.read_bytes() == b"new"
    tree.status, tree.during = 1, lambda output: output.write_bytes(b"half")
    with pytest.raises(RuntimeError, match="no such luck"):
        build.compile_call()
    assert tree.call.read_bytes() == b"new" and {p.name for p in tree.call.parent.iterdir()} == {"libtfmi.so", "tfmi_call.so"}
