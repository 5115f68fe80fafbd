"""fp16 results of a product or a multiply-add are rounded once, from the exact value: not to 32 bits first, which moves values next to the middle of two fp16 numbers."""
import numpy as np
import pytest
import torch

from muillm_amd import muillm_ext

pytestmark = pytest.mark.gpu
DEV = "cuda"


def test_dequantised_groups():
    """255 * s + m lies 2^-23 below the middle between m and the number above it; in 32 bits it is the middle, and m is odd."""
    n, k, shift = 16, 256, 5
    s, m = 257 * 2.0 ** -23, 16 + 2.0 ** -6
    codes = torch.full((n, k), 255, dtype=torch.uint8, device=DEV)
    pairs = torch.tensor([s, m], dtype=torch.float16, device=DEV).repeat(n * (k >> shift), 1)
    w = muillm_ext.muillm_int8_dequantize_forward(codes, pairs, shift)
    assert bool((w == m).all())
    # the kernels that convert codes themselves multiply the same weights: one value of x per token, tokens for every route
    for tokens in (20, 40, 300):
        for group in (5, 7):
            pairs = torch.tensor([s, m], dtype=torch.float16, device=DEV).repeat(n * (k >> group), 1)
            x = torch.zeros(tokens, k, dtype=torch.float16, device=DEV)
            x[torch.arange(tokens), torch.arange(tokens) % k] = 1
            assert bool((muillm_ext.muillm_int8_linear_forward(x, codes, pairs, group) == m).all()), (tokens, group)


def test_norm():
    """x of small whole numbers: the mean of squares is exact, and a row's factor is rsqrt of it, to a unit in the last place."""
    g = torch.Generator().manual_seed(0)
    x = torch.randint(-15, 16, (512, 4096), generator=g).half()
    gain = (1 + 0.3 * torch.randn(4096, generator=g)).half()
    got = muillm_ext.muillm_rmsnorm_forward(gain.to(DEV), x.to(DEV), 0.0).cpu().numpy()
    near = (1 / (x.numpy().astype(np.float64) ** 2).mean(-1, keepdims=True) ** 0.5).astype(np.float32)
    once, twice = np.zeros(len(x), dtype=bool), np.zeros(len(x), dtype=bool)
    for rs in (np.nextafter(near, np.float32(0)), near, np.nextafter(near, np.float32(2))):
        scaled = x.numpy().astype(np.float32) * rs  # (in 32 bits, as the kernel has it)
        once |= (got == (scaled.astype(np.float64) * gain.numpy().astype(np.float64)).astype(np.float16)).all(1)
        twice |= (got == (scaled * gain.numpy().astype(np.float32)).astype(np.float16)).all(1)
    assert once.all() and not twice.all()
