"""How the two libraries come to be built, with the compilers stood in for (nothing is compiled here)."""

import subprocess
from pathlib import Path

import pytest

from tensorfold_amd import _lib, build


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

    _lib.lib()                                               # the built kernels, as the calls below find them
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


def _says(capfd, *texts):
    err = capfd.readouterr().err
    return all(t in err for t in (*texts, "launches go through ctypes")) and err.count("ctypes") == 1


def test_without_a_call_library_launches_go_through_ctypes(tree, monkeypatch, capfd):
    """A compiler that fails, a folder that is not there to write to, a file that does not load: said once, and the kernels
    run."""

    monkeypatch.setattr(_lib, "_ready", lambda: True)
    monkeypatch.setattr(_lib, "_native", None)
    monkeypatch.setattr(_lib, "stream", lambda: 0)
    x = __import__("torch").zeros((2, 64)).bfloat16()

    def refused():
        for _ in range(2):
            with pytest.raises(RuntimeError, match="not 48"):
                _lib.call("tf_group_sums", x, 64, 2, 64, 48, x)
        assert _lib._native == {}
        _lib._native = None

    tree.status = 1
    refused()
    assert len(tree.ran) == 1 and _says(capfd, "no such luck") and tree.call.read_bytes() == b"old"
    tree.status = 0
    refused()                                                # "new" is no library
    assert tree.call.read_bytes() == b"new" and _says(capfd, "tfmi_call.so")
    monkeypatch.setattr(build, "CALL_LIB", tree.call / "below" / "tfmi_call.so")
    refused()
    assert _says(capfd, "Not a directory")
    monkeypatch.setattr(build.shutil, "which", lambda name: None)
    refused()
    assert _says(capfd, "no C++ compiler")


def test_a_build_of_the_kernels_does_without_it(tree, capfd):
    def run(output):
        tree.status = int(output.name == "tfmi_call.so")

    tree.during = run
    assert build.compile() == tree.kernels and tree.kernels.read_bytes() == b"new" and tree.call.read_bytes() == b"old"
    assert _says(capfd, "no such luck")


def test_a_call_library_without_sources_is_taken_for_its_python_and_torch_alone(tree, monkeypatch):
    monkeypatch.setattr(build, "CSRC", tree.call.parent)
    for text, taken in ((b"TFMI_CALL_ID=0123456789abcdef TFMI_CALL_FOR=" + build.call_for().encode(), tree.call),
                        (b"TFMI_CALL_ID=0123456789abcdef TFMI_CALL_FOR=0123456789abcdef", None), (b"an older build's", None)):
        tree.call.write_bytes(text)
        assert build.call_lib() == taken and not tree.ran


def test_the_built_call_library_names_both():
    if build.call_lib() is None:
        pytest.skip("no C++ compiler, Python headers or torch headers")
    assert build.built_id(build.CALL_LIB, b"TFMI_CALL_ID=") == build.call_id()
    assert build.built_id(build.CALL_LIB, b"TFMI_CALL_FOR=") == build.call_for()
