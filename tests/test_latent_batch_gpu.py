"""Prompt attention over latent rows: the rows of a batch in one launch are the rows one at a time, bit for bit."""

import pytest
import torch

from muillm_amd import _lib
from muillm_amd import hybrid_ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("heads,dim,rot,vdim", [(3, 24, 8, 40), (1, 6, 2, 10), (16, 128, 64, 128), (5, 20, 6, 12)])
@pytest.mark.parametrize("batch,t,q_first,window", [(2, 17, 0, 0), (3, 130, 21, 40), (8, 150, 0, 64), (32, 33, 5, 0)])
def test_one_launch_is_the_rows_one_at_a_time(batch, t, q_first, window, heads, dim, rot, vdim, dtype):
    g = torch.Generator(device=DEV).manual_seed(batch + t)
    first = max(0, q_first - window + 1) if window else 0
    rows, cap = q_first + t - first, q_first + t + 3
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dtype)  # noqa: E731
    q, kv, r = rand(batch, t, heads * (dim + rot)), rand(batch, rows, heads * (dim + vdim)), rand(batch, cap, rot)
    cos_sin = torch.randn(batch * t, rot, generator=g, device=DEV)
    for starts in (None, torch.arange(batch, device=DEV) % (q_first + t)):
        # per row: batches of one cannot tell their place, so every row's buffers are its own
        apart = torch.cat([ops.latent_prefill_attention(q[i:i + 1], cos_sin[i * t:(i + 1) * t].contiguous(), [kv[i].clone()], first,
                                                        r[i:i + 1].clone(), None if starts is None else starts[i:i + 1].contiguous(), q_first,
                                                        heads, dim, vdim, (dim + rot) ** -0.5, window) for i in range(batch)])
        listed = ops.latent_prefill_attention(q, cos_sin, [k.clone() for k in kv], first, r, starts, q_first, heads, dim, vdim,
                                              (dim + rot) ** -0.5, window)
        got = ops.latent_prefill_attention(q, cos_sin, kv, first, r, starts, q_first, heads, dim, vdim, (dim + rot) ** -0.5, window)
        assert torch.equal(got, listed) and torch.equal(got, apart)


def test_more_rows_than_a_launch_holds():
    """The grid's third dimension ends at 65535."""
    batch, t, heads, dim, rot, vdim, cut = 65535 + 3, 17, 1, 6, 2, 10, 65535
    g = torch.Generator(device=DEV).manual_seed(1)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV).to(torch.float16)  # noqa: E731
    q, kv, r = rand(batch, t, heads * (dim + rot)), rand(batch, t, heads * (dim + vdim)), rand(batch, t, rot)
    cos_sin, starts = torch.randn(batch * t, rot, generator=g, device=DEV), torch.arange(batch, device=DEV) % t
    call = lambda a, b: ops.latent_prefill_attention(q[a:b], cos_sin[a * t:b * t], kv[a:b], 0, r[a:b].clone(), starts[a:b], 0,  # noqa: E731
                                                     heads, dim, vdim, (dim + rot) ** -0.5, 0)
    assert torch.equal(call(0, batch), torch.cat([call(0, 40000), call(40000, cut - 1), call(cut - 1, batch - 1), call(batch - 1, batch)]))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kv_rank", [8, 64, 120, 128, 136, 256, 264, 512])
@pytest.mark.parametrize("tokens", [1, 400])
def test_value_map_of_decode_steps(kv_rank, tokens, dtype):
    """Columns of the value map that are requested early, and those behind them, with few and with many workgroups: against the
    plain kernel on the same values in fp32."""
    heads, dim, rot, vdim, keys = 5, 16, 8, 40, 9
    g = torch.Generator(device=DEV).manual_seed(kv_rank + tokens)
    rand = lambda *s, std=1.0: torch.randn(*s, generator=g, device=DEV).mul_(std).to(dtype)  # noqa: E731
    q, c, r = rand(tokens, 1, heads * (dim + rot)), rand(tokens, keys, kv_rank), rand(tokens, keys, rot)
    uk, uv = rand(heads * dim, kv_rank, std=kv_rank ** -0.5), rand(heads * vdim, kv_rank, std=kv_rank ** -0.5)
    cos_sin, pos = torch.randn(tokens, rot, generator=g, device=DEV), torch.tensor([keys - 1], device=DEV)
    args = (pos, None, heads, dim, vdim, (dim + rot) ** -0.5, 0)
    got = ops.latent_attention(q, cos_sin, uk, uv, c, r, *args, _lib.MUI_LATENT_DECODE)
    ref = ops.latent_attention(q.float(), cos_sin, uk.float(), uv.float(), c.float(), r.float(), *args, _lib.MUI_LATENT_PLAIN)
    err = float((got.double() - ref.double()).abs().max() / ref.double().abs().max())
    # rounded to 16 bits: the absorbed query, the probabilities and the output
    assert err <= {torch.float16: 3.0 * 2.0 ** -10, torch.bfloat16: 3.0 * 2.0 ** -7}[dtype], f"{err:.1e}"


@pytest.mark.parametrize("kv_rank,rot", [(520, 8), (568, 8), (512, 72)])
def test_ranks_beyond_the_decode_kernel(kv_rank, rot):
    heads, dim, vdim, keys, tokens = 3, 16, 40, 9, 4
    g = torch.Generator(device=DEV).manual_seed(kv_rank)
    rand = lambda *s, std=1.0: torch.randn(*s, generator=g, device=DEV).mul_(std).to(torch.bfloat16)  # noqa: E731
    q, c, r = rand(tokens, 1, heads * (dim + rot)), rand(tokens, keys, kv_rank), rand(tokens, keys, rot)
    uk, uv = rand(heads * dim, kv_rank, std=kv_rank ** -0.5), rand(heads * vdim, kv_rank, std=kv_rank ** -0.5)
    cos_sin, pos = torch.randn(tokens, rot, generator=g, device=DEV), torch.tensor([keys - 1], device=DEV)
    args = (pos, None, heads, dim, vdim, (dim + rot) ** -0.5, 0)
    route = ops.latent_route(torch.bfloat16, 1, heads, dim, rot, vdim, kv_rank)
    got = ops.latent_attention(q, cos_sin, uk, uv, c, r, *args, route)
    ref = ops.latent_attention(q.float(), cos_sin, uk.float(), uv.float(), c.float(), r.float(), *args, _lib.MUI_LATENT_PLAIN)
    assert float((got.double() - ref.double()).abs().max() / ref.double().abs().max()) <= 3.0 * 2.0 ** -7
    with pytest.raises(_lib.MuiLibraryError):
        ops.latent_attention(q, cos_sin, uk, uv, c, r, *args, _lib.MUI_LATENT_DECODE)
