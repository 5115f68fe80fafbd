"""Small kernels of a decode step where their fast forms begin and end, against float64: experts' sums of up to 256 rows and eight
experts, chunks of eight values per thread; and the grouping of few pairs by expert."""

import pytest
import torch

from muillm_amd import hybrid_ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
REL = {torch.float32: 3e-6, torch.bfloat16: 5e-3, torch.float16: 7e-4}


def _close(got, ref, rel):
    assert bool(torch.isfinite(got).all())
    err = float((got.double() - ref).abs().max() / ref.abs().max())
    assert err <= rel, f"{err:.2e} > {rel:.1e}"


def _rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,top,k", [(1, 8, 4096), (256, 8, 2048), (257, 8, 2048), (3, 9, 2056), (2, 1, 8), (5, 7, 4104), (2, 8, 4088),
                                        (3, 4, 4096), (3, 5, 2056), (200, 8, 4096), (201, 8, 4096), (3, 8, 1024), (3, 8, 1032)])
def test_moe_residual_norm_edges(rows, top, k, dtype):
    g = _gen(rows + top + k)
    n_exp = 5
    expert = torch.randint(0, n_exp + 3, (rows, top), generator=g, device=DEV, dtype=torch.int32)
    weight = torch.rand(rows, top, generator=g, device=DEV)
    pairs, own = torch.randn(rows * top, k, generator=g, device=DEV).to(dtype), torch.randn(rows, k, generator=g, device=DEV).to(dtype)
    pairs[(expert.reshape(-1) >= n_exp)] = float("nan")  # never written
    x = torch.randn(rows, k, generator=g, device=DEV)
    gp, gn = ((1 + 0.2 * torch.randn(k, generator=g, device=DEV)).to(dtype) for _ in range(2))
    src = torch.where((expert < n_exp)[..., None], pairs.double().reshape(rows, top, k), own.double()[:, None])
    y = (weight.double()[..., None] * src).sum(1)
    ref = x.double() + _rms(y, 1e-3) * gp.double() * 0.5
    out, h = ops.residual_norm(x, ops.MoEOutput(pairs, own, expert, weight, n_exp), gp, gn, 1e-3, branch_scale=0.5)
    _close(out, ref, 3e-6)
    _close(h, _rms(ref, 1e-3) * gn.double(), REL[dtype])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("following", [True, False])
@pytest.mark.parametrize("k", [2048, 2056, 4104, 8192, 8200])
def test_residual_norm_without_a_first_norm(k, following, dtype):
    g = _gen(k)
    x, y = torch.randn(3, k, generator=g, device=DEV), torch.randn(3, k, generator=g, device=DEV).to(dtype)
    gain = (1 + 0.2 * torch.randn(k, generator=g, device=DEV)).to(dtype) if following else None
    ref = x.double() + 0.5 * y.double()
    out, h = ops.residual_norm(x, y, None, gain, 1e-3, y_scale=0.5, emit=True)
    _close(out, ref, 3e-6)
    _close(h, _rms(ref, 1e-3) * gain.double() if following else ref, REL[dtype])


@pytest.mark.parametrize("tokens,top,experts,identity", [(1, 8, 64, 8), (8, 8, 64, 8), (13, 5, 64, 8), (64, 1, 3, 1), (32, 2, 2, 0), (65, 1, 7, 1)])
@pytest.mark.parametrize("skew", [0.0, 30.0])
def test_grouping_of_few_pairs(tokens, top, experts, identity, skew):
    """Pairs in the experts' order, cut into tiles of one expert; `skew` sends everybody to the same experts."""
    logits = torch.randn(tokens, experts + identity, generator=_gen(tokens), device=DEV)
    logits[:, :top] += skew
    expert, _, pairs, tiles = ops.moe_route(logits, None, experts, top, 16)
    flat, tiles, pairs = expert.cpu().reshape(-1).long(), tiles.cpu(), pairs.cpu().long()
    n, at, covered = int(tiles[0, 2]), 0, []
    assert bool((tiles[1 + n:, 2] == 0).all())
    sizes = torch.bincount(flat[flat < experts], minlength=experts)
    want = [(e, min(16, int(sizes[e]) - i)) for e in range(experts) for i in range(0, int(sizes[e]), 16)]
    assert [(e, c) for e, _, c, _ in tiles[1:1 + n].tolist()] == want
    for e, first, count, _ in tiles[1:1 + n].tolist():
        assert first == at and bool((flat[pairs[first:first + count]] == e).all())
        at += count
        covered += pairs[first:first + count].tolist()
    assert sorted(covered) == (flat < experts).nonzero().flatten().tolist()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("q_rank,kv_rank,rot", [(1536, 512, 64), (8, 8, 2), (1984, 64, 6), (1992, 64, 6), (520, 1528, 512), (40, 20, 4)])
def test_latent_prepare_edges(q_rank, kv_rank, rot, dtype):
    g = _gen(q_rank)
    down = torch.randn(2, 3, q_rank + kv_rank + rot, generator=g, device=DEV).to(dtype)
    qg, kg = ((1 + 0.2 * torch.randn(n, generator=g, device=DEV)).to(dtype) for n in (q_rank, kv_rank))
    inv = 100.0 ** (-torch.arange(rot // 2, dtype=torch.float64, device=DEV) / rot)
    cc, rc = torch.zeros(2, 9, kv_rank, dtype=dtype, device=DEV), torch.zeros(2, 9, rot, dtype=dtype, device=DEV)
    ql, cs = ops.latent_prepare(down, qg, kg, 0.05, inv, torch.arange(4, 7, device=DEV), None, cc, rc)
    rel = REL[dtype] if dtype != torch.float32 else 3e-6
    _close(ql, _rms(down[..., :q_rank].double(), 0.05) * qg.double(), rel)
    _close(cc[:, 4:7], _rms(down[..., q_rank:q_rank + kv_rank].double(), 0.05) * kg.double(), rel)
    angle = torch.arange(4, 7, device=DEV).double()[:, None] * inv
    _close(cs.reshape(2, 3, rot)[1], torch.cat([angle.cos(), angle.sin()], -1), 1e-6)
    u, v = down[..., q_rank + kv_rank:].double().split(rot // 2, -1)
    _close(rc[:, 4:7], torch.cat([u * angle.cos() - v * angle.sin(), v * angle.cos() + u * angle.sin()], -1), rel)
    assert float(cc[:, :4].abs().max()) == 0 and float(cc[:, 7:].abs().max()) == 0


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads,dv", [(8, 512), (3, 504), (2, 520), (5, 8), (3, 12)])
def test_mlstm_output_edges(heads, dv, dtype):
    g = _gen(dv)
    o, gain = torch.randn(1, 7, heads, dv, generator=g, device=DEV), (1 + 0.2 * torch.randn(heads * dv, generator=g, device=DEV)).to(dtype)
    gate = torch.randn(1, 7, heads * dv + 8, generator=g, device=DEV).to(dtype)[..., 8:]
    ref = _rms(o.double(), 0.02).reshape(1, 7, -1) * gain.double() * torch.sigmoid(gate.double())
    _close(ops.mlstm_output(o, gain, gate, 0.02), ref, REL[dtype])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads,dv", [(8, 24), (8, 64), (3, 128), (5, 184), (5, 192), (2, 200), (3, 256), (3, 264)])
def test_mlstm_output_of_narrow_heads(heads, dv, dtype):
    """Both sides of the widths from which a lane holds eight values and a wave one head; the last wave of two heads has one."""
    g = _gen(dv)
    o, gain = torch.randn(1, 301, heads, dv, generator=g, device=DEV), (1 + 0.2 * torch.randn(heads * dv, generator=g, device=DEV)).to(dtype)
    gate = torch.randn(1, 301, heads * dv, generator=g, device=DEV).to(dtype)
    ref = _rms(o.double(), 0.02).reshape(1, 301, -1) * gain.double() * torch.sigmoid(gate.double())
    _close(ops.mlstm_output(o, gain, gate, 0.02), ref, REL[dtype])


def _turned(x, n, freq):
    """x [t, n * dim] in slots 5 .., pairs of neighbours turned by their slot's angles"""
    x = x.reshape(x.shape[0], n, -1, 2)
    angle = torch.zeros(x.shape[0], x.shape[2], dtype=torch.float64, device=DEV)
    angle[:, :len(freq)] = torch.arange(5, 5 + x.shape[0], device=DEV).double()[:, None] * freq
    c, s = angle.cos()[:, None], angle.sin()[:, None]
    return torch.stack([x[..., 0] * c - x[..., 1] * s, x[..., 1] * c + x[..., 0] * s], -1).reshape(x.shape[0], -1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads,kv_heads", [(4, 1), (32, 8), (33, 3), (66, 33), (97, 97)])
def test_hybrid_prepare_wide_rows(heads, kv_heads, dtype):
    """Rows of less than a round of 512 chunks, of exactly one, and of up to three, with a ragged last one."""
    g, dim, rot, t = _gen(heads), 128, 32, 3
    nq, nk = heads * dim, kv_heads * dim
    proj = torch.randn(1, t, nq + 2 * nk, generator=g, device=DEV).to(dtype)
    qg, kg = ((1 + 0.2 * torch.randn(n, generator=g, device=DEV)).to(dtype) for n in (nq, nk))
    freq = 100.0 ** (-torch.arange(rot // 2, dtype=torch.float64, device=DEV) * 2 / rot)
    kc, vc = (torch.zeros(1, t + 6, nk, dtype=dtype, device=DEV) for _ in range(2))
    q = ops.hybrid_prepare(proj, heads, kv_heads, dim, dim, qg, kg, 0.1, freq, torch.arange(5, 5 + t, device=DEV), None, kc, vc)

    _close(q[0], _turned(_rms(proj[0, :, :nq].double(), 0.1) * qg.double(), heads, freq), REL[dtype])
    _close(kc[0, 5:5 + t], _turned(_rms(proj[0, :, nq:nq + nk].double(), 0.1) * kg.double(), kv_heads, freq), REL[dtype])
    assert torch.equal(vc[0, 5:5 + t], proj[0, :, nq + nk:]) and float(kc[0, :5].abs().max()) == 0


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads,kv_heads", [(8, 2), (33, 3)])
@pytest.mark.parametrize("t", [1024, 1025])
def test_hybrid_prepare_without_gains(t, heads, kv_heads, dtype):
    """Both sides of the number of tokens from which nothing is requested early (256 CUs), with and without a second round of chunks."""
    g, dim, rot = _gen(heads), 128, 32
    nq, nk = heads * dim, kv_heads * dim
    proj = torch.randn(1, t, nq + 2 * nk, generator=g, device=DEV).to(dtype)
    freq = 100.0 ** (-torch.arange(rot // 2, dtype=torch.float64, device=DEV) * 2 / rot)
    kc, vc = (torch.zeros(1, t + 6, nk, dtype=dtype, device=DEV) for _ in range(2))
    q = ops.hybrid_prepare(proj, heads, kv_heads, dim, dim, None, None, 0.1, freq, torch.arange(5, 5 + t, device=DEV), None, kc, vc)
    _close(q[0], _turned(proj[0, :, :nq].double(), heads, freq), REL[dtype])
    _close(kc[0, 5:5 + t], _turned(proj[0, :, nq:nq + nk].double(), kv_heads, freq), REL[dtype])
    assert torch.equal(vc[0, 5:5 + t], proj[0, :, nq + nk:]) and float(kc[0, :5].abs().max()) == 0
