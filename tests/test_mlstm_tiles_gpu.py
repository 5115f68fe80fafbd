"""Matrix memory of prompts with enough workgroups that they take several value tiles each: row by row, which takes one, the same."""

import pytest
import torch

from tests.test_hybrid_ops_gpu import _close, _mlstm_case, _mlstm_oracle, _mlstm_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads,dk,dv", [(8, 16, 128), (8, 70, 121), (8, 40, 190), (6, 24, 256)])
def test_mlstm_of_many_workgroups(heads, dk, dv, dtype):
    rows, t, cap = 24, 330, 7.0
    proj, gates = _mlstm_case(dv, dtype, rows, t, heads, dk, dv)
    o, state = _mlstm_run(proj, gates, heads, dk, dv, cap, [t])
    for b in (0, 7, rows - 1):
        ob, sb = _mlstm_run(proj[b:b + 1], gates[b:b + 1], heads, dk, dv, cap, [t])
        assert torch.equal(o[b], ob[0])
        for x, y in zip(state, sb):
            assert torch.equal(x[b], y[0])
    ref, (rs, _, _) = _mlstm_oracle(proj[7], gates[7], heads, dk, dv, cap)
    _close(o[7], ref, 5e-5)
    _close(state[0][7], rs, 2e-5)
