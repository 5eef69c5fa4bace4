"""The decode layer's scratch against the layer it is given for, with the launches stood in for."""

import types

import pytest
import torch

from tensorfold_amd import _lib, experts, moe


@pytest.mark.parametrize("switch", [None, "SLICED_DECODE", "ROUTING_LAUNCH"])
@pytest.mark.parametrize("width,taken", [(256, True), (128, True), (512, False), (192, False), (320, False)])
def test_activations_that_are_not_whole_rows_of_the_layer_are_refused(monkeypatch, switch, width, taken):
    launched = []
    monkeypatch.setattr(_lib, "on_gpu", lambda *_: None)
    monkeypatch.setattr(_lib, "call", lambda name, *args: launched.append(name))
    if switch:
        monkeypatch.setattr(moe, switch, True)
    d, ne, rows = 128, 4, 2
    cfg = types.SimpleNamespace(num_experts_per_tok=2, num_experts=ne, moe_intermediate_size=256, hidden_size=d)
    buf = moe.MoEBuffers(rows, cfg, "cpu", shared=False)               # 2 x 2 rows of 256 values
    ex = experts.Experts(torch.zeros((ne, 1, 1, 1, 1)), torch.zeros((ne, 1, 1, 1, 1)), 64, width, d)
    x, logits = torch.zeros((rows, d), dtype=torch.bfloat16), torch.zeros((rows, ne))
    if taken:
        moe.decode(x, logits, ex, buf, 2, ne)
        assert launched
    else:
        with pytest.raises(RuntimeError):
            moe.decode(x, logits, ex, buf, 2, ne)
        assert not launched
