"""A single token's routing with its gate and up product in one launch, against the same in 64 bits: row ends, experts that are not there, sizes that the launch
declines, ties. Gate: the roundings to 16 bits of the activation and of the result, in proportion."""
import pytest
import torch

from muillm_amd import _lib
from muillm_amd import hybrid_ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
ULP = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}


def _make(experts, identity, top, width, ff, dtype, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed + width + ff + experts)
    rand = lambda *s, std=1.0: torch.empty(s, device=DEV).normal_(0.0, std, generator=g).to(dtype)  # noqa: E731
    return (rand(1, width), torch.empty(1, experts + identity, device=DEV).normal_(generator=g), rand(experts + identity, std=0.05),
            rand(experts, ff, width, std=width ** -0.5), rand(experts, ff, width, std=width ** -0.5), rand(experts, width, ff, std=ff ** -0.5))


def _reference(x, logits, corr, gate, up, down, limit, top):
    share = torch.softmax(logits.double(), -1)[0]
    chosen = torch.sort(share + corr.double(), descending=True, stable=True).indices[:top]
    y = torch.zeros(x.shape[1], dtype=torch.float64, device=DEV)
    for e in chosen.tolist():
        if e >= gate.shape[0]:
            y += share[e] * x[0].double()
            continue
        a, u = (gate[e].double() @ x[0].double()).clamp(max=limit), (up[e].double() @ x[0].double()).clamp(-limit, limit)
        y += share[e] * (down[e].double() @ (a * torch.sigmoid(1.702 * a) * (u + 1)))
    return chosen, share[chosen], y


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("experts,identity,top,width,ff", [
    (64, 8, 8, 4096, 1792), (64, 8, 6, 2048, 1408), (3, 1, 4, 8, 2), (2, 6, 5, 264, 64), (200, 56, 8, 2056, 30), (16, 0, 1, 4088, 512), (5, 0, 5, 512, 2000),
    (70, 200, 3, 256, 64), (16, 2, 9, 256, 64), (8, 1, 2, 4104, 64), (8, 0, 2, 256, 65), (8, 0, 2, 256, 72)])
def test_against_64_bits(experts, identity, top, width, ff, dtype):
    """The last ones but one are sizes that go the general way: 270 outputs, nine chosen, a long row, an odd number of activations."""
    x, logits, corr, gate, up, down = _make(experts, identity, top, width, ff, dtype)
    out = ops.moe(x, logits, corr, gate, up, down, 7.0, top)
    chosen, share, want = _reference(x, logits, corr, gate, up, down, 7.0, top)
    assert out.expert[0].tolist() == chosen.tolist()
    assert float((out.weight[0].double() - share).abs().max() / share.max()) < 1e-5
    got = out.dense()[0].double()
    assert float((got - want).norm() / want.norm()) < ULP[dtype]


@pytest.mark.parametrize("outputs,top,width,ff,one", [
    (72, 8, 4096, 1792, True), (72, 6, 2048, 1408, True), (128, 8, 2048, 1024, True), (64, 2, 512, 512, True), (8, 2, 256, 4096, True),
    (128, 4, 256, 1024, False), (256, 2, 512, 1024, False), (64, 8, 512, 4096, False), (192, 2, 1024, 1024, False)])
def test_one_launch_where_it_is_faster(outputs, top, width, ff, one):
    """Its tiles are in the order of the choice, those of the general way sorted by expert (which follows where rows are short, outputs many)."""
    lib, bf16 = _lib.load(), torch.bfloat16
    logits = torch.arange(outputs, 0, -1, device=DEV).mul(-1.0)[None].contiguous()  # the last one is chosen first
    w, x, act = torch.zeros(outputs, ff, width, dtype=bf16, device=DEV), torch.zeros(1, width, dtype=bf16, device=DEV), torch.empty(top, ff, dtype=bf16, device=DEV)
    expert, weight, pairs, tiles = ops._routing(1, top, outputs, 16, x.device)
    _lib.check(lib.mui_moe_route_gateup(torch.cuda.current_stream().cuda_stream, ops.dtype_code(bf16), logits.data_ptr(), None, 0, w.data_ptr(), w.data_ptr(), ff * width, x.data_ptr(), 7.0,
                                        16, expert.data_ptr(), weight.data_ptr(), pairs.data_ptr(), tiles.data_ptr(), act.data_ptr(), outputs, ff, width, top, 1), "mui_moe_route_gateup")
    chosen = list(range(outputs - 1, outputs - 1 - top, -1))
    assert expert[0].tolist() == chosen
    assert tiles[1:1 + top, 0].tolist() == (chosen if one else chosen[::-1])


@pytest.mark.parametrize("width,ff,once", [(2048, 1408, True), (512, 64, False)])
def test_same_as_apart(width, ff, once):
    """The general way gives the same choice, and the same values but for the order of sums; the down product takes the tiles as they are left."""
    x, logits, corr, gate, up, down = _make(64, 8, 8, width, ff, torch.bfloat16)
    assert (64 * ff * width * 4 > 32 << 20) == once
    tile = ops.moe_tile_pairs(x.dtype, 1, 8, 64, width, ff)
    expert, weight, pairs, tiles = ops.moe_route(logits, corr, 64, 8, tile)
    apart = ops.MoEOutput(ops.moe_experts(x, gate, up, down, 7.0, expert, pairs, tiles, tile), x, expert, weight, 64).dense()
    out = ops.moe(x, logits, corr, gate, up, down, 7.0, 8)
    assert torch.equal(out.expert, expert)
    assert float(((out.weight - weight) / weight).abs().max()) <= 72 * 2.0 ** -24  # (a sum of 72 in another order)
    assert float((out.dense() - apart).norm() / apart.norm()) < 2 * ULP[torch.bfloat16]


def test_ties_nothing_real_and_nan():
    x, logits, corr, gate, up, down = _make(6, 4, 4, 64, 16, torch.bfloat16)
    logits.fill_(1.0)
    assert ops.moe(x, logits, None, gate, up, down, 7.0, 4).expert[0].tolist() == [0, 1, 2, 3]  # the lowest of equals
    logits[0, :6] = -50.0
    out = ops.moe(x, logits, None, gate, up, down, 7.0, 4)  # identity experts only
    assert out.expert[0].tolist() == [6, 7, 8, 9]
    assert float((out.dense() - x.float()).abs().max()) < 1e-5
    logits.fill_(float("nan"))
    out = ops.moe(x, logits, None, gate, up, down, 7.0, 4)
    assert int(out.expert.max()) < 10 and int(out.expert.min()) >= 0
    assert bool(torch.isnan(out.weight).any()) or float(out.weight.abs().max()) == 0.0
    torch.cuda.synchronize()


def test_refused():
    lib = _lib.load()
    x, logits, corr, gate, up, down = _make(4, 0, 2, 64, 16, torch.bfloat16)
    args = [torch.empty(64, dtype=torch.int32, device=DEV).data_ptr() for _ in range(4)]
    act = torch.empty(2, 16, dtype=torch.bfloat16, device=DEV)
    for top, n_identity in ((5, 0), (0, 0), (2, -1)):
        assert lib.mui_moe_route_gateup(None, 1, logits.data_ptr(), None, n_identity, gate.data_ptr(), up.data_ptr(), 16 * 64, x.data_ptr(), 7.0, 16, *args, act.data_ptr(),
                                        4, 16, 64, top, 1) == -1
    with pytest.raises(RuntimeError):
        ops.moe(x, logits, corr, gate, up[:2], down, 7.0, 2)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("experts,chosen,ff,width", [
    (16, [3, 20, 0, 15], 768, 8), (16, [20, 20, 5], 768, 4104), (9, [8, 7, 6, 5, 4, 3, 2, 1, 0, 9], 2048, 264), (6, [5], 2056, 512), (4, [0, 9, 3], 4096, 1000),
    (4, [0, 3], 760, 64), (4, [3, 9, 1], 4104, 64), (4, [2, 1], 1024, 12), (4, [9, 9], 1024, 64)])
def test_down_against_64_bits(experts, chosen, ff, width, dtype):
    """Rows of one and two chunks per thread, whole and part filled; the first and the last expert; identity experts in front, between and alone, whose rows stay as they
    are; from (760 ..) on sizes that go the general way, and nothing chosen that has a matrix. Gate: the rounding of the result to 16 bits."""
    g = torch.Generator(device=DEV).manual_seed(ff + width)
    act = torch.empty(len(chosen), ff, device=DEV).normal_(generator=g).to(dtype)
    down = torch.empty(experts, width, ff, device=DEV).normal_(0.0, ff ** -0.5, generator=g).to(dtype)
    expert = torch.tensor([chosen], dtype=torch.int32, device=DEV)
    real = [(i, e) for i, e in enumerate(chosen) if e < experts]
    pairs = torch.tensor([i for i, _ in real] + [0], dtype=torch.int32, device=DEV)
    most = _lib.load().mui_moe_max_tiles(1, len(chosen), experts, 16)
    tiles = torch.zeros(most + 1, 4, dtype=torch.int32)
    tiles[0, 2] = len(real)
    for j, (_, e) in enumerate(real):
        tiles[1 + j] = torch.tensor([e, j, 1, 0])
    tiles, out = tiles.to(DEV), torch.full((len(chosen), width), 7.0, dtype=dtype, device=DEV)
    st = torch.cuda.current_stream().cuda_stream
    _lib.check(_lib.load().mui_moe_one_down(st, ops.dtype_code(dtype), down.data_ptr(), width * ff, act.data_ptr(), expert.data_ptr(), pairs.data_ptr(), tiles.data_ptr(), 16,
                                            out.data_ptr(), experts, width, ff, len(chosen)), "mui_moe_one_down")
    for i, e in enumerate(chosen):
        if e >= experts:
            assert bool((out[i] == 7.0).all())
            continue
        want = down[e].double() @ act[i].double()
        assert float((out[i].double() - want).norm() / want.norm()) < ULP[dtype] / 2


@pytest.mark.parametrize("experts,top,width,ff,general", [(32, 8, 4096, 768, True), (32, 32, 1024, 1272, True), (8, 4, 8192, 1024, True), (32, 8, 4088, 768, False), (8, 8, 4096, 1280, False)])
def test_down_of_many_short_rows(experts, top, width, ff, general):
    """Short rows, 32768 of them and more, go the general way, whose sums are others."""
    g, st = torch.Generator(device=DEV).manual_seed(ff + width), torch.cuda.current_stream().cuda_stream
    act, down = (torch.empty(s, device=DEV).normal_(generator=g).bfloat16() for s in ((top, ff), (experts, width, ff)))
    logits = torch.empty(1, experts, device=DEV).normal_(generator=g)
    expert, _, pairs, tiles = ops.moe_route(logits, None, experts, top, 16)
    one, apart = (torch.empty(top, width, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    args = (st, ops.dtype_code(act.dtype), down.data_ptr(), width * ff, act.data_ptr(), expert.data_ptr(), pairs.data_ptr(), tiles.data_ptr(), 16)
    _lib.check(_lib.load().mui_moe_one_down(*args, one.data_ptr(), experts, width, ff, top), "mui_moe_one_down")
    _lib.check(_lib.load().mui_moe_down(*args, apart.data_ptr(), experts, width, ff, top, 1), "mui_moe_down")
    assert torch.equal(one, apart) == general
    assert float((one.double() - apart.double()).norm() / apart.double().norm()) < ULP[torch.bfloat16]
