"""Latent attention of one new token in one launch: against 64-bit arithmetic over the same stored rows, and the rows that it stores against latent_prepare's."""
import pytest
import torch

from oracle import salepel as oracle
from muillm_amd import hybrid_ops as ops
from muillm_amd.modules.attention.latentattention import MuiLatentAttention
from tests.salepel_util import assert_rows, build, config, latent, mlstm, moe, random_weights, row_error

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rotated(x, cos, sin):
    u, w = x.double().chunk(2, -1)
    return torch.cat([u * cos - w * sin, w * cos + u * sin], -1)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("own", [True, False])
@pytest.mark.parametrize("heads,dim,rot,vdim,kv_rank", [(16, 128, 64, 128, 512), (5, 20, 16, 12, 40), (3, 1, 48, 1, 8), (2, 127, 32, 121, 504)])
@pytest.mark.parametrize("batch,cap,pos,window,padded", [(1, 9, 0, 0, False), (1, 256, 255, 0, False), (1, 300, 299, 256, False), (3, 70, 64, 9, True), (8, 72, 65, 0, True), (2, 40, 45, 0, False),
                                                         (2, 40, -1, 0, False)])
def test_one_launch(batch, cap, pos, window, padded, heads, dim, rot, vdim, kv_rank, own, dtype):
    g = torch.Generator(device=DEV).manual_seed(batch + cap + heads)
    rand = lambda *s, std=1.0: torch.randn(*s, generator=g, device=DEV).mul_(std).to(dtype)  # noqa: E731
    q, down = rand(batch, 1, heads * (dim + rot)), rand(batch, 1, 24 + kv_rank + rot)
    uk, uv, gain = rand(heads * dim, kv_rank, std=kv_rank ** -0.5), rand(heads * vdim, kv_rank, std=kv_rank ** -0.5), rand(kv_rank)
    c, r = rand(batch, cap, kv_rank), rand(batch, cap, rot)
    starts = torch.arange(batch, device=DEV) * (pos + 1) // 2 if padded else None  # (the third row of three holds the new token alone)
    c[:, max(pos, 0) + (not own):], r[:, max(pos, 0) + (not own):] = float("nan"), float("nan")
    for i in range(batch if padded else 0):
        c[i, :starts[i]], r[i, :starts[i]] = float("nan"), float("nan")
    half = torch.arange(rot // 2, device=DEV, dtype=torch.float64)
    inv_freq, at = 10000.0 ** (-2.0 * half / rot), torch.tensor([pos], device=DEV)
    scale, eps = (dim + rot) ** -0.5, 1e-5
    assert ops.latent_step_serves(q, batch, heads, dim, rot, vdim, uk, uv, c, r, window)
    cs, rs = c.clone(), r.clone()
    out = ops.latent_step(q, down[..., 24:] if own else None, gain if own else None, eps, inv_freq, uk, uv, cs, rs, at, starts, heads, dim, vdim, scale, window)
    if own:
        cp, rp = c.clone(), r.clone()
        ops.latent_prepare(down, torch.ones(24, dtype=dtype, device=DEV), gain, eps, inv_freq, at, starts, cp, rp)
        u = torch.finfo(dtype).eps  # one value rounded to either side
        assert torch.allclose(cs.float(), cp.float(), rtol=u, atol=0, equal_nan=True) and torch.allclose(rs.float(), rp.float(), rtol=u, atol=2e-7, equal_nan=True)
    u = torch.finfo(dtype).eps / 2
    for i in range(batch):
        start = int(starts[i]) if padded else 0
        hi = min(pos, cap - 1)
        lo = max(hi - window + 1 if window else 0, start, 0)
        got = out[i, 0].double().reshape(heads, vdim)
        if hi < lo:
            assert not got.any()
            continue
        qi = q[i, 0].reshape(heads, dim + rot)
        angle = max(pos - start, 0) * inv_freq
        qr = rotated(qi[:, dim:], angle.cos(), angle.sin()).to(dtype).double()
        ci, ri = cs[i, lo:hi + 1].double(), rs[i, lo:hi + 1].double()
        kc = (uk.double() @ ci.T).reshape(heads, dim, -1)
        p = ((torch.matmul(qi[:, None, :dim].double(), kc)[:, 0] + qr @ ri.T) * scale).softmax(-1)
        v = torch.matmul(uv.double(), ci.T).reshape(heads, vdim, -1)
        ref = torch.matmul(v, p[:, :, None])[..., 0]
        # scores: a rotated query value may round to its other neighbour (2 u); fp32 sums of dim + kv_rank products over their magnitudes
        terms = (torch.matmul(uk.double().abs().reshape(heads, dim, -1).transpose(1, 2), qi[:, :dim, None].double().abs())[..., 0] @ ci.abs().T)
        off = scale * (2 * u * (qr.abs() @ ri.abs().T) + (dim + kv_rank) * 2.0 ** -24 * (terms + qr.abs() @ ri.abs().T)).amax(-1) + 4 * 2.0 ** -24
        most = torch.matmul(torch.matmul(uv.double().abs(), ci.abs().T).reshape(heads, vdim, -1), p[:, :, None])[..., 0]
        tol = u * ref.abs() + (2 * off[:, None] + (kv_rank + hi - lo + 16) * 2.0 ** -24) * most + 6e-8  # (the last: fp16's steps below its normal range)
        assert ((got - ref).abs() <= tol).all(), (i, ((got - ref).abs() / tol).max())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_what_it_leaves_alone(dtype):
    def serves(batch=1, heads=4, dim=16, rot=16, vdim=16, kv_rank=64, window=0, cap=64, off=0):
        n = heads * dim * kv_rank
        uk = torch.zeros(n + 8, dtype=dtype, device=DEV)[off:off + n].view(heads * dim, kv_rank)
        c, r = (torch.zeros(batch, cap, w, dtype=dtype, device=DEV) for w in (kv_rank, rot))
        return ops.latent_step_serves(uk, batch, heads, dim, rot, vdim, uk, torch.zeros(heads * vdim, kv_rank, dtype=dtype, device=DEV), c, r, window)

    half = dtype != torch.float32
    assert serves() == half and serves(window=256, cap=400) == half
    for kw in (dict(dim=129), dict(vdim=129), dict(kv_rank=520), dict(kv_rank=60), dict(rot=80), dict(rot=8), dict(rot=0), dict(cap=257), dict(cap=400, window=257), dict(batch=65), dict(off=1)):
        assert not serves(**kw), kw


@pytest.mark.parametrize("listened", [False, True])
def test_decoder(listened):
    """A decoder whose latent layers are served, own rows and another layer's, token by token against the float64 oracle; and with a hook of the query's projection, which hears it."""
    cfg = config([(latent(rot=16), moe()), (latent(rot=16, window=21, kv_from=0), None), (mlstm(), None), (latent(heads=5, rot=16, window=57), None)])
    w = random_weights(cfg, seed=4, close_calls=False)
    tokens = torch.randint(0, cfg["vocab"], (150,), generator=torch.Generator().manual_seed(4)).tolist()
    lm = build(cfg, w, torch.bfloat16)
    heard = []
    for m in lm.modules():
        if listened and isinstance(m, MuiLatentAttention):
            m.up_q.register_forward_hook(lambda m, args, out: heard.append(args[0].shape[1]))
    cache = lm.create_cache(1, 200)
    outs = [lm(input_ids=torch.tensor([tokens[:40]], device=DEV), past_key_values=cache).logits[0]]
    outs += [lm(input_ids=torch.tensor([[t]], device=DEV), past_key_values=cache).logits[0] for t in tokens[40:]]
    assert_rows(row_error(torch.cat(outs), oracle.forward(cfg, w, tokens)[0]), torch.bfloat16)
    assert heard == (([40] * 3 + [1] * 3 * 110) if listened else [])


@pytest.mark.parametrize("window,used", [(160, True), (200, False)])
def test_decoder_beyond_the_keys_of_one_launch(window, used, monkeypatch):
    cfg = config([(latent(rot=16, window=window), None), (latent(rot=16, window=window, kv_from=0), None)])
    w = random_weights(cfg, seed=5, close_calls=False)
    tokens = torch.randint(0, cfg["vocab"], (230,), generator=torch.Generator().manual_seed(5)).tolist()
    calls, step = [], ops.latent_step
    monkeypatch.setattr(ops, "latent_step", lambda *a, **kw: calls.append(1) or step(*a, **kw))
    lm = build(cfg, w, torch.bfloat16)
    cache = lm.create_cache(1, 240)
    outs = [lm(input_ids=torch.tensor([tokens[:210]], device=DEV), past_key_values=cache).logits[0]]
    outs += [lm(input_ids=torch.tensor([[t]], device=DEV), past_key_values=cache).logits[0] for t in tokens[210:]]
    assert_rows(row_error(torch.cat(outs), oracle.forward(cfg, w, tokens)[0]), torch.bfloat16)
    assert len(calls) == (2 * 20 if used else 0)


def _logits(lm, tokens, first):
    cache = lm.create_cache(1, 200)
    outs = [lm(input_ids=torch.tensor([tokens[:first]], device=DEV), past_key_values=cache).logits[0]]
    return torch.cat(outs + [lm(input_ids=torch.tensor([[t]], device=DEV), past_key_values=cache).logits[0] for t in tokens[first:]])


def _assert_fp16(err):
    """fp16 rounds eight times finer than bf16, for which the gate is 0.08; every single token for itself."""
    assert float(err[20:].max()) <= 0.08 / 8, err


@pytest.mark.parametrize("latents,gains", [(1.0, 1.0), (2.0 ** 11, 2.0 ** 7), (2.0 ** -10, 2.0 ** -10)])
def test_latents_and_gains_whose_product_is_out_of_fp16s_range(latents, gains):
    """The normed query latent is gain times latent times the norm's scale: the first two alone need not fit."""
    cfg = config([(latent(rot=16), None), (latent(rot=16, window=21, kv_from=0), None)])
    w = random_weights(cfg, seed=6, close_calls=False)
    for i in range(2):
        w[f"l{i}.mix.dq"] *= latents
        w[f"l{i}.mix.dq.norm"] *= gains
        w[f"l{i}.mix.uq"] /= gains
    tokens = torch.randint(0, cfg["vocab"], (30,), generator=torch.Generator().manual_seed(6)).tolist()
    _assert_fp16(row_error(_logits(build(cfg, w, torch.float16), tokens, 20), oracle.forward(cfg, w, tokens)[0]))


@pytest.mark.parametrize("name", ["q_norm", "kv_norm"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_gains_in_the_middle_of_a_buffer(dtype, name):
    """Where a parameter lies (views into one flat buffer) is no matter to the single token."""
    cfg = config([(latent(rot=16), None)])
    w = random_weights(cfg, seed=7, close_calls=False)
    tokens = torch.randint(0, cfg["vocab"], (30,), generator=torch.Generator().manual_seed(7)).tolist()
    lm = build(cfg, w, dtype)
    for m in lm.modules():
        if isinstance(m, MuiLatentAttention):
            gain = getattr(m, name)
            flat = torch.zeros(gain.numel() + 8, dtype=dtype, device=DEV)
            flat[1:1 + gain.numel()] = gain
            setattr(m, name, torch.nn.Parameter(flat[1:1 + gain.numel()], requires_grad=False))
            assert getattr(m, name).data_ptr() % 16
    err = row_error(_logits(lm, tokens, 20), oracle.forward(cfg, w, tokens)[0])
    _assert_fp16(err) if dtype == torch.float16 else assert_rows(err, dtype)
