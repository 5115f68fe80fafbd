"""Delta rule steps of a single token: their inputs go into the ring of the convolutions from registers, which comes round after 19 of them (taps 4)."""

import pytest
import torch

from tests.test_zufadra_ops_gpu import Y_REL, _close, _Delta

pytestmark = pytest.mark.gpu

# (heads, kv_heads, dk, dv, taps, ranks of decay and gate): four and eight rows of S per thread, shared query heads, one tap, as many channels as threads, and one more of one
SIZES = [(4, 2, 64, 64, 4, 16, 8), (4, 1, 128, 128, 4, 128, 128), (3, 1, 100, 72, 2, 72, 136), (2, 1, 16, 4, 1, 8, 8), (2, 2, 16, 512, 3, 8, 8), (2, 1, 16, 516, 3, 8, 8),
         (2, 2, 128, 128, 4, 8, 256)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", range(len(SIZES)))
@pytest.mark.parametrize("batch", [3, 260])
def test_single_tokens_round_the_ring(case, batch, dtype):
    d = _Delta(dtype, *SIZES[case], seed=case)
    pads = torch.zeros(batch, dtype=torch.int64)
    pads[1] = 3
    proj = d.inputs(batch, 24)
    y, s = d.run(proj, [1] * 22 + [2], pads)  # (a call of two reads what single ones have left)
    for b in (0, 1, batch - 1):
        ref, s_ref = d.reference(proj[b, pads[b]:])
        _close(y[b, pads[b]:], ref, Y_REL[dtype], b)
        _close(s[b], s_ref, 2e-5, b)
