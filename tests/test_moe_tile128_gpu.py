"""Experts' products on 128-pair tiles, whose k-steps start at another place for every expert and row tile: at the edges of their pairs, experts of one tile and of
several side by side, weights below and above 32 MB, a K that the loads into LDS do not take, against float64."""
import pytest
import torch

from muillm_amd import hybrid_ops as ops
from tests.test_moe_tiles_gpu import DEV, REL

pytestmark = pytest.mark.gpu
COUNTS = [1, 8, 9, 63, 64, 65, 32, 33, 127, 128, 129, 0, 200, 16, 257, 31]


@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16))
@pytest.mark.parametrize("width,ff", [(64, 64), (128, 192), (320, 576), (2048, 576), (576, 2048), (104, 72)])
def test_products_of_uneven_experts(width, ff, dtype):
    g = torch.Generator(device=DEV).manual_seed(width)
    n, tokens = len(COUNTS), sum(COUNTS)
    chosen = torch.repeat_interleave(torch.arange(n), torch.tensor(COUNTS))[torch.randperm(tokens, generator=torch.Generator().manual_seed(1))].to(DEV)
    logits = torch.full((tokens, n), -4.0, device=DEV).scatter_(1, chosen[:, None], 4.0)
    rand = lambda *s, std=1.0: torch.empty(s, device=DEV).normal_(0.0, std, generator=g).to(dtype)  # noqa: E731
    x, gate, up, down = rand(tokens, width), rand(n, ff, width, std=width ** -0.5), rand(n, ff, width, std=width ** -0.5), rand(n, width, ff, std=ff ** -0.5)
    expert, _, pairs, tiles = ops.moe_route(logits, None, n, 1, 128)
    out = ops.moe_experts(x, gate, up, down, 7.0, expert, pairs, tiles, 128)
    for e in range(n):
        rows = (chosen == e).nonzero()[:, 0]
        if not len(rows):
            continue
        xe = x[rows].double()
        a, u = (xe @ gate[e].double().T).clamp(max=7.0), (xe @ up[e].double().T).clamp(-7.0, 7.0)
        ref = (a * torch.sigmoid(1.702 * a) * (u + 1.0)).to(dtype).double() @ down[e].double().T
        err = float((out[rows].double() - ref).abs().max() / ref.abs().max())
        assert err <= REL[dtype], f"expert {e}, {COUNTS[e]} pairs: {err:.2e}"
    # the same rows among others: the same bits
    some = (chosen == 3) | (chosen == 10)
    expert, _, pairs, tiles = ops.moe_route(logits[some].contiguous(), None, n, 1, 128)
    assert torch.equal(ops.moe_experts(x[some].contiguous(), gate, up, down, 7.0, expert, pairs, tiles, 128), out[some])
