"""The stream a launch goes to, on a torch build without the internal names that give its handle directly."""

import types

import pytest
import torch

from tensorfold_amd import _lib


@pytest.mark.parametrize("name", ["_cuda_getCurrentRawStream", "_cuda_getDevice"])
def test_without_torchs_internal_names_the_public_call_is_asked(monkeypatch, name):
    for internal in ("_cuda_getCurrentRawStream", "_cuda_getDevice"):
        monkeypatch.setattr(torch._C, internal, lambda *device: 0, raising=False)
    monkeypatch.delattr(torch._C, name)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(cuda_stream=7))
    assert _lib.stream() == 7
