"""Experts' products on 256-pair tiles at the edges of their 32-pair strips, their row tiles and their k-steps, against float64."""

import pytest
import torch

from muillm_amd import _lib
from muillm_amd import hybrid_ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
COUNTS = [1, 31, 32, 33, 64, 65, 96, 97, 129, 160, 193, 0, 224, 225, 255, 256, 257, 300]
# the output's rounding (half a unit: 2^-9, 2^-12 of the value) and as much again for values of the activation that round the
# other way, against the largest output
REL = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16))
@pytest.mark.parametrize("width,ff", [(64, 64), (128, 192), (192, 128), (320, 576)])
def test_products_of_uneven_experts(width, ff, dtype):
    g = torch.Generator().manual_seed(width)
    n, tokens = len(COUNTS), sum(COUNTS)
    chosen = torch.repeat_interleave(torch.arange(n), torch.tensor(COUNTS))[torch.randperm(tokens, generator=g)]
    logits = torch.full((tokens, n), -4.0).scatter_(1, chosen[:, None], 4.0)
    x = torch.randn(tokens, width, generator=g).to(dtype).to(DEV)
    gate, up = (torch.randn(n, ff, width, generator=g).mul_(width ** -0.5).to(dtype).to(DEV) for _ in range(2))
    down = torch.randn(n, width, ff, generator=g).mul_(ff ** -0.5).to(dtype).to(DEV)
    expert, _, pairs, tiles = ops.moe_route(logits.to(DEV), None, n, 1, 256)
    assert torch.equal(expert[:, 0].cpu().long(), chosen)
    for _ in range(2):
        out = ops.moe_experts(x, gate, up, down, 7.0, expert, pairs, tiles, 256)
        for e in range(n):
            rows = (chosen == e).nonzero()[:, 0].to(DEV)
            if not len(rows):
                continue
            xe = x[rows].double()
            a = (xe @ gate[e].double().T).clamp(max=7.0)
            u = (xe @ up[e].double().T).clamp(-7.0, 7.0)
            act = (a * torch.sigmoid(1.702 * a) * (u + 1.0)).to(dtype).double()
            ref = act @ down[e].double().T
            err = float((out[rows].double() - ref).abs().max() / ref.abs().max())
            assert err <= REL[dtype], f"expert {e}, {COUNTS[e]} pairs: {err:.2e}"


@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16))
@pytest.mark.parametrize("width,ff,experts", [(64, 48, 11), (2048, 520, 20), (2008, 520, 20)])  # (gate and up below and above 32 MB, rows of no whole cache lines)
def test_neighbouring_tiles_of_one_expert(width, ff, experts, dtype):
    """16-pair tiles: experts with one tile and with several, side by side, at the first and the last place."""
    counts = ([17, 16, 1, 0, 33, 48, 15, 32, 2, 0, 20] + [0] * experts)[:experts]
    counts[-1] = max(counts[-1], 31)
    g = torch.Generator().manual_seed(width)
    tokens = sum(counts)
    chosen = torch.repeat_interleave(torch.arange(experts), torch.tensor(counts))[torch.randperm(tokens, generator=g)]
    logits = torch.full((tokens, experts), -4.0).scatter_(1, chosen[:, None], 4.0)
    x = torch.randn(tokens, width, generator=g).to(dtype).to(DEV)
    gate, up = (torch.randn(experts, ff, width, generator=g).mul_(width ** -0.5).to(dtype).to(DEV) for _ in range(2))
    down = torch.randn(experts, width, ff, generator=g).mul_(ff ** -0.5).to(dtype).to(DEV)
    expert, _, pairs, tiles = ops.moe_route(logits.to(DEV), None, experts, 1, 16)
    assert torch.equal(expert[:, 0].cpu().long(), chosen)
    out = ops.moe_experts(x, gate, up, down, 7.0, expert, pairs, tiles, 16)
    for e in range(experts):
        rows = (chosen == e).nonzero()[:, 0].to(DEV)
        if not len(rows):
            continue
        xe = x[rows].double()
        a = (xe @ gate[e].double().T).clamp(max=7.0)
        u = (xe @ up[e].double().T).clamp(-7.0, 7.0)
        ref = (a * torch.sigmoid(1.702 * a) * (u + 1.0)).to(dtype).double() @ down[e].double().T
        err = float((out[rows].double() - ref).abs().max() / ref.abs().max())
        assert err <= REL[dtype], f"expert {e}, {counts[e]} pairs: {err:.2e}"


@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16))
@pytest.mark.parametrize("width,ff,experts,counts", [
    (512, 640, 5, [3, 0, 16, 1, 2]),               # four and five segments: every wave has one of every unit; fewer units than workgroups
    (768, 520, 7, [0, 0, 0, 0, 0, 0, 1]),          # one tile; k of down in no whole segments (a workgroup per block)
    (2048, 1152, 24, [1] * 24),                    # more units than workgroups, gate and up beyond 32 MB: all rows non-temporal
    (2048, 1152, 24, [2, 17, 0, 40] + [1] * 20),   # ... and by unit: experts with one tile and with several
    (1032, 2056, 12, [5, 1, 33] + [0] * 9)])       # blocks that end inside the matrix; no whole segments
def test_units_of_a_round_of_workgroups(width, ff, experts, counts, dtype):
    g = torch.Generator().manual_seed(width + ff)
    tokens = sum(counts)
    chosen = torch.repeat_interleave(torch.arange(experts), torch.tensor(counts))[torch.randperm(tokens, generator=g)]
    logits = torch.full((tokens, experts), -4.0).scatter_(1, chosen[:, None], 4.0)
    x = torch.randn(tokens, width, generator=g).to(dtype).to(DEV)
    gate, up = (torch.randn(experts, ff, width, generator=g).mul_(width ** -0.5).to(dtype).to(DEV) for _ in range(2))
    down = torch.randn(experts, width, ff, generator=g).mul_(ff ** -0.5).to(dtype).to(DEV)
    expert, _, pairs, tiles = ops.moe_route(logits.to(DEV), None, experts, 1, 16)
    assert int(tiles[0, 3]) == (max(counts) > 16)
    for _ in range(2):
        out = ops.moe_experts(x, gate, up, down, 7.0, expert, pairs, tiles, 16)
        for e in range(experts):
            rows = (chosen == e).nonzero()[:, 0].to(DEV)
            if not len(rows):
                continue
            xe = x[rows].double()
            a = (xe @ gate[e].double().T).clamp(max=7.0)
            u = (xe @ up[e].double().T).clamp(-7.0, 7.0)
            ref = (a * torch.sigmoid(1.702 * a) * (u + 1.0)).to(dtype).double() @ down[e].double().T
            err = float((out[rows].double() - ref).abs().max() / ref.abs().max())
            assert err <= REL[dtype], f"expert {e}, {counts[e]} pairs: {err:.2e}"


def test_units_without_a_tile():
    """All tokens choose identity experts: nothing is written."""
    experts, width, ff, tokens = 4, 512, 512, 3
    logits = torch.full((tokens, experts + 1), -4.0)
    logits[:, experts] = 4.0
    expert, _, pairs, tiles = ops.moe_route(logits.to(DEV), None, experts, 1, 16)
    assert int(tiles[0, 2]) == 0
    w = torch.ones(experts, ff, width, dtype=torch.bfloat16, device=DEV)
    x, act = torch.ones(tokens, width, dtype=torch.bfloat16, device=DEV), torch.full((tokens, ff), 7.0, dtype=torch.bfloat16, device=DEV)
    out = torch.full((tokens, width), 7.0, dtype=torch.bfloat16, device=DEV)
    lib, s, code = _lib.load(), torch.cuda.current_stream().cuda_stream, _lib.MUI_DTYPE_BF16
    _lib.check(lib.mui_moe_gateup(s, code, w.data_ptr(), w.data_ptr(), ff * width, x.data_ptr(), 7.0, expert.data_ptr(), pairs.data_ptr(), tiles.data_ptr(), 16, act.data_ptr(),
                                  experts, ff, width, 1, tokens), "gateup")
    _lib.check(lib.mui_moe_down(s, code, w.data_ptr(), ff * width, act.data_ptr(), expert.data_ptr(), pairs.data_ptr(), tiles.data_ptr(), 16, out.data_ptr(),
                                experts, width, ff, 1, tokens), "down")
    assert bool((act == 7.0).all()) and bool((out == 7.0).all())


@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16))
@pytest.mark.parametrize("width,ff", [(2176, 1152), (2048, 1408), (2304, 1280)])  # gate/up, down: 17 and 9 segments, 16 and 11, 18 and 10
def test_a_rows_bits_beside_other_rows(width, ff, dtype):
    """Alone a token's units are a workgroup's first; among others they come later, where the waves hold other segments of them."""
    experts = 24
    g = torch.Generator().manual_seed(width + ff)
    x = torch.randn(experts, width, generator=g).to(dtype).to(DEV)
    gate, up = (torch.randn(experts, ff, width, generator=g).mul_(width ** -0.5).to(dtype).to(DEV) for _ in range(2))
    down = torch.randn(experts, width, ff, generator=g).mul_(ff ** -0.5).to(dtype).to(DEV)
    logits = torch.full((experts, experts), -4.0).fill_diagonal_(4.0).to(DEV)

    def run(rows):
        expert, _, pairs, tiles = ops.moe_route(logits[rows].contiguous(), None, experts, 1, 16)
        return ops.moe_experts(x[rows].contiguous(), gate, up, down, 7.0, expert, pairs, tiles, 16)

    together = run(list(range(experts)))
    for e in (3, 11, 19, 23):
        assert torch.equal(run([e])[0], together[e]), f"expert {e}"
        assert torch.equal(run(list(range(e, experts)))[0], together[e]), f"expert {e} first"
