"""Products whose big tiles leave a last round of workgroups at most half full (it is a launch of its own, of smaller tiles): sizes on both sides of a quarter and
of half a round, with outputs and tokens that do not come out even, against float64 products and against one launch."""
import pytest
import torch

from muillm_amd import _lib, muillm_ext

pytestmark = pytest.mark.gpu
DEV = "cuda"
REL = {torch.bfloat16: 2 ** -7, torch.float16: 2 ** -10}  # as a share of the largest output: four times one rounding to 16 bits
K = 128
# (outputs, tokens); 256 CUs: a quarter of a round is 8 tiles of an XCD, half of it 16
GATEUP = [(14336, 2048), (14336, 1280), (14336, 3500), (14300, 3585), (8192, 1100), (8200, 1281), (4090, 2500)]
LINEAR = [(4096, 4352), (4096, 2304), (4100, 2305), (8192, 2300), (12290, 1700), (28672, 777), (6144, 2600), (4096, 8191)]


@pytest.mark.parametrize("weights", ["bf16", "fp16", "int8", "int8_group"])
@pytest.mark.parametrize("form,n,tokens", [("gateup", *s) for s in GATEUP] + [("linear", *s) for s in LINEAR])
def test_last_round(weights, form, n, tokens):
    dtype, g = torch.bfloat16 if weights == "bf16" else torch.float16, torch.Generator(device=DEV).manual_seed(n + tokens)
    gateup, rows = form == "gateup", 2 * n if form == "gateup" else n
    x = torch.randn(tokens, K, device=DEV, generator=g).to(dtype)
    bias, res = torch.randn(n, device=DEV, generator=g).to(dtype), torch.randn(tokens, n, device=DEV, generator=g).to(dtype)
    if "int8" in weights:
        q = torch.randint(-128, 128, (rows, K), device=DEV, generator=g, dtype=torch.int32)
        s = (torch.rand(rows, device=DEV, generator=g) * 2e-3 + 1e-3).to(dtype)
        w = q.float() * s.float()[:, None]
    else:
        w = (torch.randn(rows, K, device=DEV, generator=g) * 0.1).to(dtype)
    if weights == "int8":
        c = q.to(torch.int8)
        pair, sp = c.view(n, 2, K) if gateup else None, s.view(n, 2) if gateup else None
        call = (lambda: muillm_ext.mui_int8_channel_gateupsilu_forward(None, 0.0, pair[:, 0], pair[:, 1], sp[:, 0], sp[:, 1], x)) if gateup else \
            (lambda: muillm_ext.mui_int8_channel_linear_forward(x, c, s, add_bias=bias, residual=res))
    elif weights == "int8_group":  # one group of 128 per row: (scale, smallest value)
        c, low = (q + 128).to(torch.uint8), (s.float() * -128).to(dtype)
        pairs = torch.stack([s, low], 1)
        w = (q + 128).float() * s.float()[:, None] + low.float()[:, None]
        call = (lambda: muillm_ext.muillm_int8_gateupsilu_forward(None, 0.0, c.view(n, 2, K), pairs.view(n, 2, 1, 2), 7, x)) if gateup else \
            (lambda: muillm_ext.muillm_int8_linear_forward(x, c, pairs.contiguous(), 7, add_bias=bias, residual=res))
    else:
        pair = w.view(n, 2, K) if gateup else None
        call = (lambda: muillm_ext.mui_gateup_silu(None, 0.0, pair[:, 0], pair[:, 1], x)) if gateup else \
            (lambda: muillm_ext.muillm_linear_forward(None, x, w, add_bias=bias, residual=res))
    ref = x.double() @ w.double().T
    ref = ref[:, 0::2] * torch.sigmoid(ref[:, 0::2]) * ref[:, 1::2] if gateup else ref + bias.double() + res.double()
    lib = _lib.load()
    y = call()
    assert lib.mui_tune_prefill(3200, 0) == 0
    try:
        one = call()
    finally:
        lib.mui_tune_prefill(0, 0)
    for out in (y, one):
        assert float((out.double() - ref).abs().max() / ref.abs().max()) <= REL[dtype]
