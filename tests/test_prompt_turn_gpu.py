"""Prompts of a single token tile on the tiles whose waves split K: row tiles that start at different k-steps, with step counts and last steps that do not come
out even, against float64 products."""
import pytest
import torch

from muillm_amd import _lib, muillm_ext

pytestmark = pytest.mark.gpu
DEV = "cuda"
REL = {torch.bfloat16: 2 ** -7, torch.float16: 2 ** -10}  # as a share of the largest output: four times one rounding to 16 bits


@pytest.mark.parametrize("dtype", list(REL))
@pytest.mark.parametrize("which", [0, 5, 6, 9, 11, 12])  # the call's choice, 64 x 128, 32 x 64, 128 x 128, 128 x 64, 64 x 64
@pytest.mark.parametrize("k", [64, 264, 1000, 1536])
@pytest.mark.parametrize("n", [4000, 2056])
@pytest.mark.parametrize("form", ["linear", "gateup", "int8", "int8 gateup"])
def test_turned_steps(dtype, which, k, n, form):
    g, tokens = torch.Generator(device=DEV).manual_seed(n + k), 63 if which in (6, 11, 12) else 121
    int8, gateup = "int8" in form, "gateup" in form
    if int8:
        k = (k + 15) // 16 * 16
    x = torch.randn(tokens, k, device=DEV, generator=g).to(dtype)
    rows = 2 * n if gateup else n
    if int8:
        q = torch.randint(-128, 128, (rows, k), device=DEV, generator=g, dtype=torch.int32)
        s = (torch.rand(rows, device=DEV, generator=g) * 2e-3 + 1e-3).to(dtype)
        w, q = q.double() * s.double()[:, None], q.to(torch.int8)
        pair, sp = (q.view(n, 2, k), s.view(n, 2)) if gateup else (None, None)
        y = (lambda: muillm_ext.mui_int8_channel_gateupsilu_forward(None, 0.0, pair[:, 0], pair[:, 1], sp[:, 0], sp[:, 1], x)) if gateup else \
            (lambda: muillm_ext.mui_int8_channel_linear_forward(x, q, s))
    else:
        w = (torch.randn(rows, k, device=DEV, generator=g) * 0.1).to(dtype)
        pair = w.view(n, 2, k) if gateup else None
        y = (lambda: muillm_ext.mui_gateup_silu(None, 0.0, pair[:, 0], pair[:, 1], x)) if gateup else (lambda: muillm_ext.muillm_linear_forward(None, x, w))
    ref = x.double() @ w.double().T
    if gateup:
        ref = ref[:, 0::2] * torch.sigmoid(ref[:, 0::2]) * ref[:, 1::2]
    lib = _lib.load()
    assert lib.mui_tune_prefill(which, 0) == 0
    try:
        out = y()
    finally:
        lib.mui_tune_prefill(0, 0)
    assert float((out.double() - ref).abs().max() / ref.abs().max()) <= REL[dtype]
