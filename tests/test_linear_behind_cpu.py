"""The boundary that a linear's call takes along is only used for the very output it was made from."""

import pytest
import torch

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
