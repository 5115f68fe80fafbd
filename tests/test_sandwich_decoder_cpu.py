"""What the host does between two sublayers of several rows, whose prompts are bound by it where tokens are few."""
import sys
from types import SimpleNamespace

import torch

from muillm_amd import hybrid_ops
from muillm_amd.modules.decoder import sandwichdecoder


def test_calls_per_sublayer(monkeypatch):
    """Of Python functions: the sublayer itself, the join behind it and its library call, and one that puts them together."""
    monkeypatch.setattr(hybrid_ops, "residual_norm", lambda x, y, *args, **kw: (x, y))
    norm, calls = SimpleNamespace(weight=None), []

    def sublayer(h, *cache):
        return h

    layer = SimpleNamespace(mixer=sublayer, mlp=sublayer, branch_scale=1.0, pre_mixer_norm=norm, post_mixer_norm=norm, pre_mlp_norm=norm, post_mlp_norm=norm)
    x = torch.zeros(3, 2, 8)
    sys.setprofile(lambda frame, event, arg: calls.append(frame.f_code.co_name) if event == "call" else None)
    try:
        sandwichdecoder.run_layers([layer] * 5, x, x, norm, 1e-5, None, None)
    finally:
        sys.setprofile(None)
    assert calls.count("sublayer") == 20  # (the stub's and the loop's)
    assert len(calls) <= 4 * 10 + 4, calls
