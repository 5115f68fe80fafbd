"""Linears of more than 128 tokens whose K is shared between workgroups, against the same in 64 bits at the edges of tiles, shares and rounds, and with the norm behind
taken along. Gate: fp32 accumulation is far below the roundings to 16 bits of the result."""
import pytest
import torch

from muillm_amd import _lib
from tests.prompt_util import prompt_shares
from tests.test_gemm_stream_gpu import CODE, DEV, HALF_ULP, _gen, _rand
from tests.test_linear_behind_gpu import EPS, _call, _close, _ptr, _rms

pytestmark = pytest.mark.gpu


@pytest.fixture
def tune():
    lib = _lib.load()
    yield lambda tile, shares: _lib.check(lib.mui_tune_prompt_shares(tile, shares), "mui_tune_prompt_shares")
    _lib.check(lib.mui_tune_prompt_shares(0, 0), "mui_tune_prompt_shares")


def _linear(x, w, mul, add, res, ws):
    (tokens, k), n = x.shape, w.shape[0]
    y = torch.full((tokens, n), float("nan"), dtype=x.dtype, device=DEV)
    _lib.check(_lib.load().mui_linear_ws(torch.cuda.current_stream().cuda_stream, CODE[x.dtype], w.data_ptr(), w.stride(0), x.data_ptr(), None, 0.0, _ptr(mul), _ptr(add),
                                         _ptr(res), y.data_ptr(), n, k, tokens, ws.data_ptr(), ws.numel()), "mui_linear_ws")
    return y


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tile,shares", [(7, 2), (7, 7), (8, 3), (8, 8), (4, 2), (4, 5)])
@pytest.mark.parametrize("n,k,tokens", [(4, 3072, 129), (260, 3136, 257), (1000, 3072, 300), (4104, 3200, 511), (2048, 3072, 256)])
def test_forced_shares(n, k, tokens, tile, shares, dtype, tune):
    """A share that gets a k-step less than another, tiles that end in the matrix or the tokens, rows that are not dense, several rounds of workgroups."""
    g = _gen(n + k + tokens)
    w, x = _rand((n, k + 8), dtype, g, k ** -0.5)[:, :k], _rand((tokens, k), dtype, g)
    res, mul, add = _rand((tokens, n), dtype, g), _rand((n,), dtype, g), _rand((n,), dtype, g)
    ws = torch.zeros(_lib.load().mui_linear_workspace_bytes(), dtype=torch.uint8, device=DEV)
    plain, rel = x.double() @ w.double().T, 2 * HALF_ULP[dtype]
    tune(tile, shares)
    _close(_linear(x, w, None, None, None, ws), plain, rel)
    assert bool(ws[4096:].any()) and not bool(ws[:4096].any())  # K was shared; the counters are left alone
    _close(_linear(x, w, mul, add, res, ws), plain * mul.double() + add.double() + res.double(), rel)
    tune(-1, 0)
    ws.zero_()
    _close(_linear(x, w, None, None, None, ws), plain, rel)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,k,tokens", [(4096, 14336, 129), (4096, 4096, 333), (2048, 8192, 700), (8192, 2048, 200), (8200, 4096, 200), (1000, 6144, 1300)])
def test_by_the_rule_and_with_the_norm_behind(n, k, tokens, dtype):
    """Boundaries taken along give the bits of two calls, whether K is shared or not (8200 outputs are two launches)."""
    lib, s, code = _lib.load(), torch.cuda.current_stream().cuda_stream, CODE[dtype]
    g = _gen(n + k + tokens)
    w, x, res = _rand((n, k), dtype, g, k ** -0.5), _rand((tokens, k), dtype, g), _rand((tokens, n), dtype, g)
    post, after = 1 + _rand((n,), dtype, g, 0.2), 1 + _rand((n,), dtype, g, 0.2)
    stream = torch.empty(tokens, n, device=DEV).normal_(generator=g)
    ws = torch.zeros(lib.mui_linear_workspace_bytes(), dtype=torch.uint8, device=DEV)
    y2, h2 = _linear(x, w, None, None, res, ws), torch.empty_like(res)
    assert bool(ws[4096:].any()) == (prompt_shares("fp16" if dtype == torch.float16 else "bf16", n, k, tokens)[1] > 1)
    _lib.check(lib.mui_rmsnorm(s, code, after.data_ptr(), y2.data_ptr(), EPS, h2.data_ptr(), tokens, n), "norm")
    y, h, out, out2 = torch.empty_like(res), torch.empty_like(res), torch.empty_like(stream), torch.empty_like(stream)
    _call("mui_linear_norm", x, w, k, None, (res.data_ptr(), after.data_ptr(), EPS, y.data_ptr(), h.data_ptr()), y, ws)
    assert torch.equal(y, y2) and torch.equal(h, h2)
    plain = x.double() @ w.double().T
    _close(y, plain + res.double(), 2 * HALF_ULP[dtype])
    _close(h, _rms(plain + res.double(), after.double()), 2 * HALF_ULP[dtype])
    y2 = _linear(x, w, None, None, None, ws)
    _lib.check(lib.mui_residual_norm(s, code, stream.data_ptr(), y2.data_ptr(), 1.0, post.data_ptr(), 0.5, after.data_ptr(), 2.0, EPS, out2.data_ptr(), h2.data_ptr(), tokens, n), "norm")
    _call("mui_linear_residual_norm", x, w, k, None, (stream.data_ptr(), post.data_ptr(), 0.5, after.data_ptr(), 2.0, EPS, y.data_ptr(), out.data_ptr(), h.data_ptr()), y, ws)
    assert torch.equal(y, y2) and torch.equal(out, out2) and torch.equal(h, h2)
