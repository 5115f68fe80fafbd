"""What the built-in rules do with a prompt product, for tests that are about one route and have to take it, and such products."""
import ctypes

import torch

from muillm_amd import _lib, muillm_ext

WEIGHTS = {"fp16": (0, 0), "bf16": (1, 0), "int8": (0, 1), "int8_group": (0, 2), "int8_bf16": (1, 1)}  # dtype code, weight format


def prompt_plan(weights: str, form: str, n: int, k: int, tokens: int, shift: int = 7, scratch: bool = True):
    """(tokens in a launch of their own, tile of the others, what becomes of its last round: 0 as it is, 1 halves, 2 quarters); form "gateup" or "linear"."""
    (dtype, fmt), out = WEIGHTS[weights], [ctypes.c_int() for _ in range(3)]
    _lib.check(_lib.load().mui_probe_prefill_plan(dtype, fmt, int(form == "gateup"), n, k, tokens, shift if fmt == 2 else 0, int(scratch),
                                                  *[ctypes.byref(x) for x in out]), "mui_probe_prefill_plan")
    return tuple(x.value for x in out)


def prompt_product(weights: str, form: str, n: int, k: int, tokens: int):
    """(call, its result as a product of the same operands in 32 bits): gate/up plain, linears with bias and residual; int8 in groups of 128."""
    dev, dtype = "cuda", torch.bfloat16 if weights == "bf16" else torch.float16
    g, gateup, rows = torch.Generator(device=dev).manual_seed(n + k + tokens), form == "gateup", 2 * n if form == "gateup" else n
    x = torch.randn(tokens, k, device=dev, generator=g).to(dtype)
    bias, res = torch.randn(n, device=dev, generator=g).to(dtype), torch.randn(tokens, n, device=dev, generator=g).to(dtype)
    if "int8" in weights:
        q = torch.randint(-128, 128, (rows, k), device=dev, generator=g, dtype=torch.int16)
    if weights == "int8":
        s, c = (torch.rand(rows, device=dev, generator=g) * 2e-3 + 1e-3).to(dtype), q.to(torch.int8)
        w = q.float() * s.float()[:, None]
        if gateup:
            pair, sp = c.view(n, 2, k), s.view(n, 2)
            call = lambda: muillm_ext.mui_int8_channel_gateupsilu_forward(None, 0.0, pair[:, 0], pair[:, 1], sp[:, 0], sp[:, 1], x)
        else:
            call = lambda: muillm_ext.mui_int8_channel_linear_forward(x, c, s, add_bias=bias, residual=res)
    elif weights == "int8_group":  # (scale, smallest value); the weight is what rounds to 16 bits
        s, c = (torch.rand(rows, k // 128, device=dev, generator=g) * 2e-3 + 1e-3).to(dtype), (q + 128).to(torch.uint8)
        low = (s.float() * -128).to(dtype)
        pairs = torch.stack([s, low], 2)
        w = ((q + 128).float().view(rows, -1, 128) * s.float()[..., None] + low.float()[..., None]).to(dtype).float().view(rows, k)
        call = (lambda: muillm_ext.muillm_int8_gateupsilu_forward(None, 0.0, c.view(n, 2, k), pairs.view(n, 2, -1, 2), 7, x)) if gateup else \
            (lambda: muillm_ext.muillm_int8_linear_forward(x, c, pairs, 7, add_bias=bias, residual=res))
    else:
        v = (torch.randn(rows, k, device=dev, generator=g) * 0.1).to(dtype)
        w, pair = v.float(), v.view(n, 2, k) if gateup else None
        call = (lambda: muillm_ext.mui_gateup_silu(None, 0.0, pair[:, 0], pair[:, 1], x)) if gateup else \
            (lambda: muillm_ext.muillm_linear_forward(None, x, v, add_bias=bias, residual=res))
    ref = x.float() @ w.T
    return call, ref[:, 0::2] * torch.sigmoid(ref[:, 0::2]) * ref[:, 1::2] if gateup else ref + bias.float() + res.float()


def prompt_shares(weights: str, n: int, k: int, tokens: int, shift: int = 7):
    """(tile, shares) of a linear whose K is shared between workgroups; one share: it is not."""
    (dtype, fmt), out = WEIGHTS[weights], [ctypes.c_int() for _ in range(2)]
    _lib.check(_lib.load().mui_probe_prompt_shares(dtype, fmt, n, k, tokens, shift if fmt == 2 else 0, *[ctypes.byref(x) for x in out]), "mui_probe_prompt_shares")
    return tuple(x.value for x in out)
