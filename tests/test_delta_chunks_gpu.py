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
