"""int8 codes, 17 to 64 tokens, on streamed bands of weight rows (codes in LDS, converted as they are read): every width of a band at both numbers
of token tiles, one step and rings that go round, a last band of eight rows, several bands per workgroup; against float64 products of the weights."""
import pytest
import torch

from muillm_amd import _lib, muillm_ext

pytestmark = pytest.mark.gpu
DEV = "cuda"
REL = {torch.bfloat16: 2 ** -7, torch.float16: 2 ** -10}  # as a share of the largest output: four times one rounding to 16 bits
LINEAR, GATEUP = [0, 8, 16, 24, 32, 40, 48, 56, 64, 96], [0, 16, 32, 48, 64, 96, 112]  # rows of a band; 0: as the call chooses


def _check(form, dtype, tokens, rows, n, k, gateup, pad=0):
    g = torch.Generator(device=DEV).manual_seed(n + k + tokens)
    many = 2 * n if gateup else n
    q = torch.randint(-128, 128, (many, k), device=DEV, generator=g, dtype=torch.int32)
    x = torch.randn(tokens, k, device=DEV, generator=g).to(dtype)
    bias, res = torch.randn(n, device=DEV, generator=g).to(dtype), torch.randn(tokens, n, device=DEV, generator=g).to(dtype)
    if form == "channel":
        s = (torch.rand(many, device=DEV, generator=g) * 2e-3 + 1e-3).to(dtype)
        w = q.double() * s.double()[:, None]
        codes = torch.zeros(many, k + pad, device=DEV, dtype=torch.int8)
        codes[:, :k] = q
        if gateup:
            pair, sp = codes.view(n, 2, k + pad)[:, :, :k], s.view(n, 2)
            call = lambda: muillm_ext.mui_int8_channel_gateupsilu_forward(None, 0.0, pair[:, 0], pair[:, 1], sp[:, 0], sp[:, 1], x)
        else:
            call = lambda: muillm_ext.mui_int8_channel_linear_forward(x, codes[:, :k], s, add_bias=bias, residual=res)
    else:  # groups of 64, 128 or 256: (scale, smallest value) of each, the weight rounded once
        shift = int(form)
        groups = k >> shift
        s = (torch.rand(many, groups, device=DEV, generator=g) * 2e-3 + 1e-3).to(dtype)
        low = (s.float() * -128).to(dtype)
        spread = lambda t: t.double().repeat_interleave(1 << shift, 1)
        w = ((q + 128).double() * spread(s) + spread(low)).to(dtype).double()
        codes, pairs = (q + 128).to(torch.uint8), torch.stack([s, low], 2).contiguous()
        if gateup:
            call = lambda: muillm_ext.muillm_int8_gateupsilu_forward(None, 0.0, codes.view(n, 2, k), pairs.view(n, 2, groups, 2), shift, x)
        else:
            call = lambda: muillm_ext.muillm_int8_linear_forward(x, codes, pairs, shift, add_bias=bias, residual=res)
    ref = x.double() @ w.T
    ref = ref[:, 0::2] * torch.sigmoid(ref[:, 0::2]) * ref[:, 1::2] if gateup else ref + bias.double() + res.double()
    lib = _lib.load()
    assert lib.mui_tune_stream(rows, 0) == 0
    try:
        y = call()
    finally:
        lib.mui_tune_stream(0, 0)
    assert float((y.double() - ref).abs().max() / ref.abs().max()) <= REL[dtype], (n, k)


@pytest.mark.parametrize("form", ["channel", "6", "7", "8"])
@pytest.mark.parametrize("dtype", list(REL))
@pytest.mark.parametrize("tokens", [17, 32, 33, 64])
@pytest.mark.parametrize("rows", LINEAR)
def test_linear(form, dtype, tokens, rows):
    r = rows or 16
    for n, k, pad in [(8, 256, 0), (3 * r + 8, 3328, 16), (257 * r + 8, 512, 0)]:
        _check(form, dtype, tokens, rows, n, k, False, pad)


@pytest.mark.parametrize("form", ["channel", "6", "7", "8"])
@pytest.mark.parametrize("dtype", list(REL))
@pytest.mark.parametrize("tokens", [17, 32, 33, 64])
@pytest.mark.parametrize("rows", GATEUP)
def test_gateup(form, dtype, tokens, rows):
    r = rows or 16
    for n, k, pad in [(8, 256, 0), (r + 8, 3328, 16), (257 * r // 2 + 8, 512, 0)]:
        _check(form, dtype, tokens, rows, n, k, True, pad)
