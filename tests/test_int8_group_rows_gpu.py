"""int8 in the group format at 1 to 16 tokens, rows of every length that the waves divide in ranges of their own (a range may begin inside a group),
against float64 products of the dequantised weights."""
import pytest
import torch

from muillm_amd import muillm_ext

pytestmark = pytest.mark.gpu
REL = {torch.float16: 2e-3, torch.bfloat16: 1e-2}  # of the 2-norm: outputs, and in bf16 and short groups the weights, are rounded to 16 bits


@pytest.mark.parametrize("dtype", list(REL))
@pytest.mark.parametrize("shift", [5, 6, 7, 8, 9])
@pytest.mark.parametrize("k", [256, 512, 768, 1024, 1280, 1536, 2048, 2560, 3072, 3840, 4096, 4608])
def test_rows_divided_inside_groups(dtype, shift, k):
    if k % (1 << shift):
        pytest.skip("no whole groups")
    n, g = 40, torch.Generator(device="cuda").manual_seed(k + shift)
    codes = torch.randint(0, 256, (2 * n, k), device="cuda", generator=g, dtype=torch.int32).to(torch.uint8)
    groups = k >> shift
    pairs = torch.stack([torch.rand(2 * n * groups, device="cuda", generator=g) * 2e-3 + 1e-3, -torch.rand(2 * n * groups, device="cuda", generator=g) * 0.3], 1).to(dtype)
    p = pairs.double().view(2 * n, groups, 1, 2)
    w = (codes.double().view(2 * n, groups, -1) * p[..., 0] + p[..., 1]).view(2 * n, k)
    for tokens in (1, 2, 3, 4, 5, 8, 9, 16):
        x = torch.randn(tokens, k, device="cuda", generator=g).to(dtype)
        want = x.double() @ w.T
        y = muillm_ext.muillm_int8_linear_forward(x, codes, pairs, shift)
        assert float((y.double() - want).norm() / want.norm()) <= REL[dtype], tokens
        a, b = want[:, 0::2], want[:, 1::2]
        want = a * torch.sigmoid(a) * b
        h = muillm_ext.muillm_int8_gateupsilu_forward(None, 0.0, codes.view(n, 2, k), pairs.view(n, 2, groups, 2), shift, x)
        assert float((h.double() - want).norm() / want.norm()) <= 2 * REL[dtype], tokens
