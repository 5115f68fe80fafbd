"""Scratch of linears beyond MUI_MAX_TOKENS tokens: whose it is (no GPU needed)."""
import torch

from muillm_amd import muillm_ext


def test_captured_calls_never_take_a_streams_scratch(monkeypatch):
    """A graph keeps its scratch's address and may be replayed on any stream: while a stream captures, the scratch that
    eager calls on it use stays out, whichever streams ran what before; what linear_workspace() sets is used."""
    capturing, stream = [False], 7
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing[0])
    monkeypatch.setattr(muillm_ext, "_PROMPT_WORKSPACES", {})
    monkeypatch.setattr(muillm_ext, "new_linear_workspace", lambda device: torch.zeros(8, dtype=torch.uint8, device=device))
    x = torch.zeros(32, 8)
    eager = muillm_ext._prompt_workspace(x, stream)
    assert eager is not None and muillm_ext._prompt_workspace(x, stream) is eager
    capturing[0] = True
    assert muillm_ext._prompt_workspace(x, stream) is None
    own = muillm_ext.new_linear_workspace("cpu")
    with muillm_ext.linear_workspace(own):
        assert muillm_ext._prompt_workspace(x, stream) is own
    assert muillm_ext._prompt_workspace(x, stream) is None
    stream, capturing[0] = 8, False
    other = muillm_ext._prompt_workspace(x, stream)
    assert other is not None and other is not eager and other is not own
