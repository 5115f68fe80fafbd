"""Delta rule of prompts where four columns of y cannot be written at once: rows that start at multiples of eight bytes."""

import pytest
import torch

from muillm_amd import hybrid_ops as ops
from tests.test_zufadra_ops_gpu import Y_REL, _close, _Delta

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads,dv", [(1, 4), (1, 12), (3, 68)])
def test_delta_rule_of_unaligned_segments(heads, dv, dtype, monkeypatch):
    d = _Delta(dtype, heads, 1, 16, dv, 4, seed=dv)
    proj = d.inputs(1, 107)
    ref, s_ref = d.reference(proj[0])
    for segment in (17, 33, 65):  # later segments of y start at odd tokens
        monkeypatch.setattr(ops, "DELTA_SEGMENT", segment)
        y, s = d.run(proj, [107])
        _close(y[0], ref, Y_REL[dtype], segment)
        _close(s[0], s_ref, 2e-5, segment)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("t", [17, 31, 65, 81, 113])
@pytest.mark.parametrize("rank", [16, 20])  # (read 16 bytes at a time, and not)
def test_last_chunk_with_few_tokens(t, rank, dtype):
    """Waves of the last chunk without tokens, where the workgroup loads the gate's matrix together and where it does not."""
    d = _Delta(dtype, 3, 3, 32, 24, 4, rg=rank, seed=t)
    proj = d.inputs(2, t)
    y, s = d.run(proj, [t])
    for b in range(2):
        ref, s_ref = d.reference(proj[b])
        _close(y[b], ref, Y_REL[dtype], b)
        _close(s[b], s_ref, 2e-5, b)
