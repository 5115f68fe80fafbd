"""Gate/up projections of prompts that end a little beyond whole 256-token tiles (two launches where that is cheaper): around the ends of what the
second launch takes, against float64 products and against one launch."""
import pytest
import torch

from muillm_amd import _lib, muillm_ext

pytestmark = pytest.mark.gpu
DEV = "cuda"
REL = {torch.bfloat16: 2 ** -7, torch.float16: 2 ** -10}  # as a share of the largest output: four times one rounding to 16 bits
K = 128


@pytest.fixture
def one_launch():
    lib = _lib.load()
    yield lambda on: lib.mui_tune_prefill(3200 if on else 0, 0)
    lib.mui_tune_prefill(0, 0)


@pytest.mark.parametrize("weights", ["bf16", "fp16", "int8", "int8_group"])
@pytest.mark.parametrize("n", [8192, 14336, 14320])
@pytest.mark.parametrize("tokens", [511, 513, 544, 576, 577, 640, 641, 1025, 1152, 2049, 2176])
def test_two_launches(weights, n, tokens, one_launch):
    dtype, g = torch.bfloat16 if weights == "bf16" else torch.float16, torch.Generator(device=DEV).manual_seed(n + tokens)
    x = torch.randn(tokens, K, device=DEV, generator=g).to(dtype)
    if "int8" in weights:
        q = torch.randint(-128, 128, (2 * n, K), device=DEV, generator=g, dtype=torch.int32)
        s = (torch.rand(2 * n, device=DEV, generator=g) * 2e-3 + 1e-3).to(dtype)
        w = q.float() * s.float()[:, None]
    if weights == "int8":
        c = q.to(torch.int8).view(n, 2, K)
        call = lambda: muillm_ext.mui_int8_channel_gateupsilu_forward(None, 0.0, c[:, 0], c[:, 1], s.view(n, 2)[:, 0], s.view(n, 2)[:, 1], x)
    elif weights == "int8_group":  # one group of 128 per row: (scale, smallest value)
        c, low = (q + 128).to(torch.uint8).view(n, 2, K), (s.float() * -128).to(dtype)
        pairs = torch.stack([s, low], 1).view(n, 2, 1, 2).contiguous()
        w = (q + 128).float() * s.float()[:, None] + low.float()[:, None]
        call = lambda: muillm_ext.muillm_int8_gateupsilu_forward(None, 0.0, c, pairs, 7, x)
    else:
        w = (torch.randn(2 * n, K, device=DEV, generator=g) * 0.1).to(dtype)
        pair = w.view(n, 2, K)
        call = lambda: muillm_ext.mui_gateup_silu(None, 0.0, pair[:, 0], pair[:, 1], x)
        w = w.float()
    a, b = x.double() @ w[0::2].double().T, x.double() @ w[1::2].double().T
    ref = a * torch.sigmoid(a) * b
    assert one_launch(False) == 0
    y = call()
    assert one_launch(True) == 0
    assert float((y.double() - ref).abs().max() / ref.abs().max()) <= REL[dtype]
    assert float((call().double() - ref).abs().max() / ref.abs().max()) <= REL[dtype]
