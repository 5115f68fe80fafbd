"""The boundary that a linear's call takes along is only used for the very output it was made from."""

import pytest
import torch

from muillm_amd import hybrid_ops
from muillm_amd.engineconfig import MuiEngineConfig
from muillm_amd.modules.decoder import sandwichdecoder
from muillm_amd.modules.linear import MuiLinear
from muillm_amd.modules.recurrent.mlstm import MuiMLstm
from muillm_amd.muillm_ext import ResidualBehind


def _behind(gain, stream=None, after=None):
    return ResidualBehind(torch.zeros(17, 8) if stream is None else stream, gain, 1.0, after, 1.0, 1e-5)


def _filled():
    y = torch.zeros(17, 8)
    with torch.no_grad():
        behind = _behind(torch.ones(8))
        assert behind.linear(y, lambda name, args: None)
    return behind, y


def test_taken_for_the_output_itself_only():
    behind, y = _filled()
    assert behind.take(y.clone()) is None and behind.take(y.view(17, 8)) is None
    assert behind.take(y) is not None
    y.add_(1)
    assert behind.take(y) is None
    assert _behind(torch.ones(8)).take(y) is None  # never filled


def test_not_filled_where_it_cannot_be_checked_or_does_not_fit():
    y = torch.zeros(17, 8)

    def tried(*args, **kw):
        return _behind(*args, **kw).linear(y, lambda name, args: None)

    assert not tried(torch.ones(8))  # gradients are on
    with torch.no_grad():
        assert tried(torch.ones(8)) and tried(torch.ones(8), after=torch.ones(8))
        assert not tried(torch.ones(8).half()) and not tried(torch.ones(4)) and not tried(torch.ones(16)[::2])
        assert not tried(torch.ones(8), after=torch.ones(9))
        assert not tried(torch.ones(8), torch.zeros(17, 8).half()) and not tried(torch.ones(8), torch.zeros(16, 8))
        assert not tried(torch.ones(8), torch.zeros(8, 17).T)
    with torch.inference_mode():
        assert not _behind(torch.ones(8)).linear(torch.zeros(17, 8), lambda name, args: None)


@pytest.mark.parametrize("tokens,worth", [(1, False), (16, False), (17, True), (128, True), (129, False)])
def test_number_of_tokens(tokens, worth):
    with torch.no_grad():
        assert ResidualBehind.worth_it(tokens) == worth
    assert not ResidualBehind.worth_it(tokens)


class _Mixer(MuiMLstm):
    """y = out_proj(h), with the boundary filled in as the library's call does it."""
    takes_behind = MuiMLstm.takes_behind

    def __init__(self):
        super(MuiMLstm, self).__init__(engine_config=MuiEngineConfig())
        self.out_proj = MuiLinear(MuiEngineConfig(), 8, 8, bias=False)
        self.got = []

    def forward(self, h, cache, cache_position, behind=None):
        self.got.append(behind)
        y = self.out_proj(h)
        if behind is not None:
            assert behind.linear(y, lambda name, args: None)
            behind.result = (behind.stream + y, y.clone())
        return y


@pytest.fixture
def layer(monkeypatch):
    monkeypatch.setattr(hybrid_ops, "residual_norm", lambda x, y, *a, **kw: (x + y, y.clone()))
    return sandwichdecoder.MuiSandwichDecoderLayer(MuiEngineConfig(), 8, _Mixer(), None, 1e-5, pre_norms=False)


def _through(layer):
    """The residual stream behind the layer, and whether its mixer was given the boundary."""
    out = []
    with torch.no_grad():
        h = torch.ones(1, 17, 8)
        sandwichdecoder.run_layers([layer], torch.zeros_like(h), h, layer.post_mixer_norm, 1e-5, None, None, collect=out)
    return out[0], layer.mixer.got.pop() is not None


def _write_unseen(mod, args, out):
    out.data.mul_(2.0)


def test_a_hooks_write_is_heard(layer):
    plain, given = _through(layer)
    assert given
    for m in (layer.mixer, layer.mixer.out_proj):
        handle = m.register_forward_hook(_write_unseen)
        assert torch.equal(_through(layer)[0], 2 * plain)
        handle.remove()
        handle = m.register_forward_pre_hook(lambda mod, args: (args[0] * 2,) + args[1:])
        assert torch.equal(_through(layer)[0], 2 * plain) and torch.equal(_through(layer)[0], 2 * plain)
        handle.remove()
    handle = torch.nn.modules.module.register_module_forward_hook(lambda mod, args, out: _write_unseen(mod, args, out) if mod is layer.mixer else None)
    assert torch.equal(_through(layer)[0], 2 * plain)
    handle.remove()
    got, given = _through(layer)
    assert given and torch.equal(got, plain)


def test_a_forward_of_an_instance_is_called_as_documented(layer):
    plain, _ = _through(layer)
    mixer, linear = layer.mixer, layer.mixer.out_proj
    linear.forward = lambda x: 2 * torch.nn.functional.linear(x, linear.weight)
    assert torch.equal(_through(layer)[0], 2 * plain)
    del linear.forward
    mixer.forward = lambda h, cache, cache_position: mixer.got.append(None) or 2 * linear(h)
    assert torch.equal(_through(layer)[0], 2 * plain)
    del mixer.forward
    got, given = _through(layer)
    assert given and torch.equal(got, plain)
