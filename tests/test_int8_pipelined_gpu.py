"""int8 prompts on the software-pipelined tiles (codes in LDS, converted between the matrix instructions): every tile shape at its edges, against
float64 products of the exact weights and against the kernels that convert the codes on their way to LDS."""
import pytest
import torch

from muillm_amd import _lib, muillm_ext

pytestmark = pytest.mark.gpu
DEV = "cuda"
# outputs are rounded once to 16 bits (half a unit: 2^-9 / 2^-12 of the value), sums are in 32 bits; fp16 in the group format rounds the weight
# itself once (2^-12 of each, an error of the sum that shrinks with sqrt(K)); as a share of the largest output, four times as much
REL = {torch.bfloat16: 2 ** -7, torch.float16: 2 ** -10}
SHAPES = [(64, 64, 257), (512, 64, 256), (520, 128, 300), (1000, 192, 513), (768, 1024, 700), (6144, 256, 1030), (256, 4160, 290)]  # outputs, K, tokens


def _codes(g, n, k):
    return torch.randint(-128, 128, (n, k), device=DEV, generator=g, dtype=torch.int32)


@pytest.fixture
def tile():
    lib = _lib.load()
    yield lambda t: lib.mui_tune_prefill(t, 0)
    lib.mui_tune_prefill(0, 0)


@pytest.mark.parametrize("dtype", list(REL))
@pytest.mark.parametrize("n,k,tokens", SHAPES)
@pytest.mark.parametrize("gateup", [False, True])
@pytest.mark.parametrize("which", [0, 4, 7, 8])  # built-in choice, 256 x 256, 128 x 256, 192 x 256
def test_per_channel(dtype, n, k, tokens, gateup, which, tile):
    g = torch.Generator(device=DEV).manual_seed(n + k)
    q = _codes(g, 2 * n if gateup else n, k)
    s = (torch.rand(len(q), device=DEV, generator=g) * 2e-3 + 1e-3).to(dtype)
    x = torch.randn(tokens, k, device=DEV, generator=g).to(dtype)
    w = q.double() * s.double()[:, None]
    q = q.to(torch.int8)
    if gateup:
        a, b = x.double() @ w[0::2].T, x.double() @ w[1::2].T
        ref = a * torch.sigmoid(a) * b
        call = lambda: muillm_ext.mui_int8_channel_gateupsilu_forward(None, 0.0, q.view(n, 2, k)[:, 0], q.view(n, 2, k)[:, 1], s.view(n, 2)[:, 0], s.view(n, 2)[:, 1], x)
    else:
        bias, res = torch.randn(n, device=DEV, generator=g).to(dtype), torch.randn(tokens, n, device=DEV, generator=g).to(dtype)
        ref = x.double() @ w.T + bias.double() + res.double()
        call = lambda: muillm_ext.mui_int8_channel_linear_forward(x, q, s, add_bias=bias, residual=res)
    assert tile(which) == 0
    y = call()
    assert float((y.double() - ref).abs().max() / ref.abs().max()) <= REL[dtype]
    if which in (4, 7):  # the same products in the same order
        older = {4: 13, 7: 200 + 7}[which]
        assert tile(older) == 0
        assert torch.equal(call(), y)


@pytest.mark.parametrize("n,k,tokens", [s for s in SHAPES if s[1] % 128 == 0])
@pytest.mark.parametrize("gateup", [False, True])
@pytest.mark.parametrize("which", [0, 4, 7, 8])
@pytest.mark.parametrize("shift", [6, 7])
def test_groups(n, k, tokens, gateup, which, shift, tile):
    dtype, g = torch.float16, torch.Generator(device=DEV).manual_seed(n + k + shift)
    rows = 2 * n if gateup else n
    q = (_codes(g, rows, k) + 128)
    pairs = torch.stack([torch.rand(rows * (k >> shift), device=DEV, generator=g) * 2e-3 + 1e-3, -torch.rand(rows * (k >> shift), device=DEV, generator=g) * 0.3], 1).to(dtype)
    p = pairs.double().view(rows, k >> shift, 1, 2)
    w = (q.double().view(rows, k >> shift, -1) * p[..., 0] + p[..., 1]).view(rows, k)
    x = torch.randn(tokens, k, device=DEV, generator=g).to(dtype)
    q = q.to(torch.uint8)
    assert tile(which) == 0
    if gateup:
        a, b = x.double() @ w[0::2].T, x.double() @ w[1::2].T
        ref = a * torch.sigmoid(a) * b
        y = muillm_ext.muillm_int8_gateupsilu_forward(None, 0.0, q.view(n, 2, k), pairs.view(n, 2, k >> shift, 2), shift, x)
    else:
        ref = x.double() @ w.T
        y = muillm_ext.muillm_int8_linear_forward(x, q, pairs, shift)
    assert float((y.double() - ref).abs().max() / ref.abs().max()) <= REL[dtype]


@pytest.mark.parametrize("tokens", [20, 40, 100, 300, 1100, 1600])
@pytest.mark.parametrize("gateup", [False, True])
@pytest.mark.parametrize("shift", [6, 7])
def test_pairs_off_the_four_byte_grid(tokens, gateup, shift):
    """(scale, min) pairs at an odd 2-byte address are taken by kernels that read them with ordinary loads, on every route by number of tokens."""
    dtype, n, k, g = torch.float16, 520, 256, torch.Generator(device=DEV).manual_seed(tokens + shift)
    rows = 2 * n if gateup else n
    q, x = _codes(g, rows, k) + 128, torch.randn(tokens, k, device=DEV, generator=g).to(dtype)
    room = torch.zeros(2 * rows * (k >> shift) + 1, dtype=dtype, device=DEV)
    pairs = room[1:].view(-1, 2)
    pairs[:, 0], pairs[:, 1] = torch.rand(len(pairs), device=DEV, generator=g) * 2e-3 + 1e-3, -torch.rand(len(pairs), device=DEV, generator=g) * 0.3
    assert pairs.data_ptr() % 4 == 2
    p = pairs.double().view(rows, k >> shift, 1, 2)
    w, q = (q.double().view(rows, k >> shift, -1) * p[..., 0] + p[..., 1]).view(rows, k), q.to(torch.uint8)
    if gateup:
        a, b = x.double() @ w[0::2].T, x.double() @ w[1::2].T
        ref = a * torch.sigmoid(a) * b
        y = muillm_ext.muillm_int8_gateupsilu_forward(None, 0.0, q.view(n, 2, k), pairs.view(n, 2, k >> shift, 2), shift, x)
    else:
        ref = x.double() @ w.T
        y = muillm_ext.muillm_int8_linear_forward(x, q, pairs, shift)
    assert float((y.double() - ref).abs().max() / ref.abs().max()) <= REL[dtype]


def test_where_matrices_are_dequantised():
    f, b, at = torch.float16, torch.bfloat16, muillm_ext.int8_dequantised_from
    assert at(f, 4096) == at(b, 14336) == 8192 and at(f, 4096 + 16) == at(b, 48) == 1280
    assert at(f, 4096, 7) == 1536 and at(f, 4096, 5) == at(b, 4096, 7) == 1024
    assert at(f, 4096, 7, 1 << 20) == 1536 and at(f, 4096, 7, (1 << 20) + 2) == 1024
