"""Gate/up of 65 to 128 tokens on streamed bands of weight rows: the first and last number of tokens of six and eight token tiles, bands of both widths, one band and
all that one round of workgroups takes and one more, against float64 products."""
import pytest
import torch

from muillm_amd import _lib, muillm_ext

pytestmark = pytest.mark.gpu
DEV = "cuda"
REL = {torch.bfloat16: 2 ** -7, torch.float16: 2 ** -10}  # as a share of the largest output: four times one rounding to 16 bits


@pytest.mark.parametrize("dtype", list(REL))
@pytest.mark.parametrize("tokens", [65, 96, 97, 128])
@pytest.mark.parametrize("rows", [0, 48, 64])  # of a band; 0: as the call chooses
@pytest.mark.parametrize("n,k", [(8, 256), (40, 768), (6144, 256), (8192, 1024), (8200, 512)])
def test_gateup_of_many_tokens(dtype, tokens, rows, n, k):
    g = torch.Generator(device=DEV).manual_seed(n + k + tokens)
    w, x = (torch.randn(n, 2, k, device=DEV, generator=g) * k ** -0.5).to(dtype), torch.randn(tokens, k, device=DEV, generator=g).to(dtype)
    bg, bu = (torch.randn(n, device=DEV, generator=g).to(dtype) for _ in range(2))
    a, b = x.double() @ w[:, 0].double().T + bg.double(), x.double() @ w[:, 1].double().T + bu.double()
    ref = a * torch.sigmoid(a) * b
    lib = _lib.load()
    assert lib.mui_tune_stream(rows, 0) == 0
    try:
        y = muillm_ext.mui_gateup_silu(None, 0.0, w[:, 0], w[:, 1], x, bg, bu)
    finally:
        lib.mui_tune_stream(0, 0)
    assert float((y.double() - ref).abs().max() / ref.abs().max()) <= REL[dtype]
