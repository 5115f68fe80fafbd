"""Linears of 16-bit weights at 17..128 tokens (csrc/gemm_stream.hip) at the sizes where its tiles, rounds and shares of K end,
against the same product in 64 bits. Gate: the output's own rounding (half a unit of its type) and fp32 accumulation,
k 2^-24 of the sum of the products' magnitudes."""

import pytest
import torch

from muillm_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"
HALF_ULP = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}
CODE = {torch.float16: _lib.MUI_DTYPE_F16, torch.bfloat16: _lib.MUI_DTYPE_BF16}


def _rand(shape, dtype, gen, std=1.0):
    return torch.empty(shape, dtype=dtype, device=DEV).normal_(0.0, std, generator=gen)


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _assert_within(y, ref, magnitude, k, dtype):
    assert bool(torch.isfinite(y).all())
    off = (y.double() - ref).abs()
    bound = HALF_ULP[dtype] * ref.abs() + 2.0 * k * 2.0 ** -24 * magnitude + 2.0 ** -24
    worst = float((off / bound).max())
    assert worst <= 1.0, f"{worst:.2f} times the bound"


def _linear(x, w, pitch, mul=None, add=None, res=None, ws=None):
    tokens, k = x.shape
    n = w.shape[0]
    y = torch.full((tokens, n), float("nan"), dtype=x.dtype, device=DEV)
    ptr = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    _lib.check(_lib.load().mui_linear_ws(torch.cuda.current_stream().cuda_stream, CODE[x.dtype], w.data_ptr(), pitch, x.data_ptr(), None, 0.0,
                                         ptr(mul), ptr(add), ptr(res), y.data_ptr(), n, k, tokens, ptr(ws), 0 if ws is None else ws.numel()),
               "mui_linear_ws")
    return y


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tokens", [17, 32, 33, 64, 65, 96, 97, 127, 128])
@pytest.mark.parametrize("n,k", [(8, 256), (24, 512), (2040, 768), (4096, 1024), (1000, 4096), (1024, 8192), (33000, 256), (17416, 512)])
def test_linear_against_64_bits(n, k, tokens, dtype):
    """With and without a workspace (shares of K on the long rows), pitched weights, every operand of the end."""
    g = _gen(n + k + tokens)
    pitch = k + 8
    w = _rand((n, pitch), dtype, g, k ** -0.5)[:, :k]
    x, res = _rand((tokens, k), dtype, g), _rand((tokens, n), dtype, g)
    mul, add = _rand((n,), dtype, g, 0.5), _rand((n,), dtype, g)
    ws = torch.zeros(_lib.load().mui_linear_workspace_bytes(), dtype=torch.uint8, device=DEV)
    plain = x.double() @ w.double().T
    size = x.double().abs() @ w.double().abs().T
    for scratch in (None, ws):
        _assert_within(_linear(x, w, pitch, ws=scratch), plain, size, k, dtype)
        got = _linear(x, w, pitch, mul, add, res, scratch)
        ref = plain * mul.double() + add.double() + res.double()
        _assert_within(got, ref, size * mul.double().abs() + add.double().abs() + res.double().abs(), k, dtype)
        assert torch.equal(got, _linear(x, w, pitch, mul, add, res, scratch)), "not the same twice"
    assert int(ws[:4096].sum()) == 0, "the counters of the workspace"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tokens", [17, 32, 33, 64, 65, 96])
@pytest.mark.parametrize("n", [32776, 65000])
def test_units_that_follow_each_other(n, tokens, dtype):
    """A workgroup takes several bands of up to 128 rows, each longer than the ring of stages and with more tiles than meet at a
    time (up to eight rounds): what one round or band leaves in LDS must not reach the next."""
    k = 2048
    g = _gen(n + tokens)
    w, x = _rand((n, k), dtype, g, k ** -0.5), _rand((tokens, k), dtype, g)
    y = _linear(x, w, k)
    _assert_within(y, x.double() @ w.double().T, x.double().abs() @ w.double().abs().T, k, dtype)
    for _ in range(3):
        assert torch.equal(y, _linear(x, w, k)), "not the same twice"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tokens", [17, 32, 33, 48, 64])
@pytest.mark.parametrize("n,k", [(8, 256), (56, 512), (1000, 1024), (16400, 256), (14336, 512)])
@pytest.mark.parametrize("packed,bias", [(True, False), (False, True)])
def test_gateup_against_64_bits(n, k, tokens, packed, bias, dtype):
    g = _gen(n + k + tokens)
    w = _rand((n, 2, k) if packed else (2, n, k), dtype, g, k ** -0.5)
    gate, up, pitch = (w[:, 0], w[:, 1], 2 * k) if packed else (w[0], w[1], k)
    x = _rand((tokens, k), dtype, g)
    bg, bu = (_rand((n,), dtype, g) for _ in range(2)) if bias else (None, None)
    h = torch.full((tokens, n), float("nan"), dtype=dtype, device=DEV)
    _lib.check(_lib.load().mui_gateup_silu_bias(torch.cuda.current_stream().cuda_stream, CODE[dtype], gate.data_ptr(), up.data_ptr(), pitch,
                                                x.data_ptr(), None, 0.0, bg.data_ptr() if bias else None, bu.data_ptr() if bias else None,
                                                h.data_ptr(), n, k, tokens), "mui_gateup_silu_bias")
    gv, uv = (x.double() @ m.double().T + (0.0 if b is None else b.double()) for m, b in ((gate, bg), (up, bu)))
    sg, su = (x.double().abs() @ m.double().abs().T + (0.0 if b is None else b.double().abs()) for m, b in ((gate, bg), (up, bu)))
    # |d silu| <= 1.1 |d g|; silu itself a few units of fp32 off
    size = 1.1 * sg * uv.abs() + gv.abs() * su + gv.abs() * uv.abs()
    _assert_within(h, gv * torch.sigmoid(gv) * uv, size, k, dtype)


LINEAR_ROWS = [8, 16, 24, 32, 40, 48, 56, 64, 96, 128]
GATEUP_ROWS = [16, 32, 48, 64, 96, 112]
TOKENS = [17, 32, 33, 64, 65, 96, 97, 128]  # the first and last of every number of token tiles


def _widest(tokens):
    tiles = 2 if tokens <= 32 else 4 if tokens <= 64 else 6 if tokens <= 96 else 8
    return min(128, 192 - 16 * tiles)


@pytest.fixture
def forced():
    lib = _lib.load()
    yield lambda rows, shares: _lib.check(lib.mui_tune_stream(rows, shares), "mui_tune_stream")
    _lib.check(lib.mui_tune_stream(0, 0), "mui_tune_stream")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,tokens", [(r, t) for r in LINEAR_ROWS for t in TOKENS if r <= _widest(t)])
def test_every_linear_unit(rows, tokens, dtype, forced):
    """Every width with every number of token tiles: one step, a ring of stages that goes round several times, a last unit of eight rows;
    several units per workgroup; shares of K of different lengths."""
    g = _gen(rows + tokens)
    ws = torch.zeros(_lib.load().mui_linear_workspace_bytes(), dtype=torch.uint8, device=DEV)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    for n, k, shares in [(rows + 8, 256, 1), (3 * rows + 8, 3328, 1), ((cus + 1) * rows + 8, 512, 1), (2 * rows + 8, 1792, 3), (5 * rows, 4352, 8)]:
        w, x, res = _rand((n, k), dtype, g, k ** -0.5), _rand((tokens, k), dtype, g), _rand((tokens, n), dtype, g)
        forced(rows, shares)
        got = _linear(x, w, k, res=res, ws=ws)
        _assert_within(got, x.double() @ w.double().T + res.double(), x.double().abs() @ w.double().abs().T + res.double().abs(), k, dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,tokens", [(r, t) for r in GATEUP_ROWS for t in TOKENS if t <= 64])
def test_every_gateup_unit(rows, tokens, dtype, forced):
    g = _gen(rows + tokens)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    for n, k in [(rows // 2 + 8, 256), (rows + 8, 3328), ((cus + 1) * rows // 2 + 8, 512)]:
        w, x = _rand((2, n, k), dtype, g, k ** -0.5), _rand((tokens, k), dtype, g)
        h = torch.full((tokens, n), float("nan"), dtype=dtype, device=DEV)
        forced(rows, 1)
        _lib.check(_lib.load().mui_gateup_silu(torch.cuda.current_stream().cuda_stream, CODE[dtype], w[0].data_ptr(), w[1].data_ptr(), k,
                                               x.data_ptr(), None, 0.0, h.data_ptr(), n, k, tokens), "mui_gateup_silu")
        gv, uv = (x.double() @ m.double().T for m in w)
        sg, su = (x.double().abs() @ m.double().abs().T for m in w)
        _assert_within(h, gv * torch.sigmoid(gv) * uv, 1.1 * sg * uv.abs() + gv.abs() * su + gv.abs() * uv.abs(), k, dtype)


def test_tokens_do_not_mix():
    """What one token holds, infinities and NaN among it, stays with it."""
    g = _gen(3)
    w, x = _rand((4096, 1024), torch.bfloat16, g, 0.03), _rand((33, 1024), torch.bfloat16, g)
    clean = _linear(x, w, 1024)
    x[32, 5], x[7, 9] = float("inf"), float("nan")
    dirty = _linear(x, w, 1024)
    rest = [t for t in range(33) if t not in (7, 32)]
    assert torch.equal(dirty[rest], clean[rest]) and bool(dirty[7].isnan().all()) and not bool(dirty[32].isfinite().any())


@pytest.mark.parametrize("n,k,tokens", [(4096, 14336, 128), (4096, 4096, 97), (2560, 8192, 96), (5120, 10240, 112), (28672, 512, 65), (128256, 256, 128)])
def test_calls_that_the_tiles_serve(n, k, tokens):
    """No workspace, or more rows than it can help with: where units of all of K take longer than the tiled GEMM, that
    runs (bit for bit what it gives by itself)."""
    g = _gen(n + k + tokens)
    w, x = _rand((n, k), torch.bfloat16, g, k ** -0.5), _rand((tokens, k), torch.bfloat16, g)
    got = _linear(x, w, k)
    lib = _lib.load()
    _lib.check(lib.mui_tune_prefill(0, -1), "mui_tune_prefill")
    try:
        tiles = _linear(x, w, k)
    finally:
        _lib.check(lib.mui_tune_prefill(0, 0), "mui_tune_prefill")
    assert torch.equal(got, tiles)
    if n == 4096:
        ws = torch.zeros(lib.mui_linear_workspace_bytes(), dtype=torch.uint8, device=DEV)
        _assert_within(_linear(x, w, k, ws=ws), x.double() @ w.double().T, x.double().abs() @ w.double().abs().T, k, torch.bfloat16)
        assert int(ws.count_nonzero()) > 0, "K is shared where there is a workspace"


@pytest.mark.parametrize("dtype", (torch.float16, torch.bfloat16))
@pytest.mark.parametrize("n,k,tokens,wide", [(296, 256, 17, True), (4096, 256, 40, True), (2048, 512, 32, True), (24, 512, 24, True),
                                             (4104, 256, 17, False), (512, 256, 41, False), (2056, 512, 32, False), (512, 512, 33, False), (512, 768, 17, False)])
def test_calls_of_one_or_two_steps(n, k, tokens, wide, dtype):
    """A K of one or two steps, few rows and tokens: 16 rows per workgroup without a ring of stages, bit for bit what that kernel gives by itself
    (it adds K in another order); on the other side of each line, units."""
    g = _gen(n + k + tokens)
    w, x, res = _rand((n, k), dtype, g, k ** -0.5), _rand((tokens, k), dtype, g), _rand((tokens, n), dtype, g)
    got = _linear(x, w, k, res=res)
    _assert_within(got, x.double() @ w.double().T + res.double(), x.double().abs() @ w.double().abs().T + res.double().abs(), k, dtype)
    if wide:
        lib = _lib.load()
        _lib.check(lib.mui_tune_prefill(0, 40), "mui_tune_prefill")
        try:
            by_itself = _linear(x, w, k, res=res)
        finally:
            _lib.check(lib.mui_tune_prefill(0, 0), "mui_tune_prefill")
        assert torch.equal(got, by_itself)


@pytest.mark.parametrize("n,k,tokens,tiles", [(14400, 768, 33, True), (16384, 768, 64, True), (28680, 1024, 48, True), (14336, 768, 64, False), (16392, 768, 33, False),
                                              (14400, 768, 32, False), (14400, 2048, 33, False), (14400, 512, 33, False)])
def test_gateup_calls_that_the_tiles_serve(n, k, tokens, tiles):
    """Units that need a round more than the tiled GEMM leave the call to it (256 CUs) unless K is two steps or rows are whole multiples of 4 KB apart, bit for bit."""
    g = _gen(n + k + tokens)
    gate, up = _rand((n, k), torch.bfloat16, g, k ** -0.5), _rand((n, k), torch.bfloat16, g, k ** -0.5)
    x, lib = _rand((tokens, k), torch.bfloat16, g), _lib.load()

    def run():
        h = torch.full((tokens, n), float("nan"), dtype=x.dtype, device=DEV)
        _lib.check(lib.mui_gateup_silu(torch.cuda.current_stream().cuda_stream, CODE[x.dtype], gate.data_ptr(), up.data_ptr(), k,
                                       x.data_ptr(), None, 0.0, h.data_ptr(), n, k, tokens), "mui_gateup_silu")
        return h

    got = run()
    a, b = x.double() @ gate.double().T, x.double() @ up.double().T
    ref = a * torch.sigmoid(a) * b
    assert float((got.double() - ref).abs().max() / ref.abs().max()) <= 2.0 ** -8
    if tiles:
        _lib.check(lib.mui_tune_prefill(0, -1), "mui_tune_prefill")
        try:
            assert torch.equal(got, run())
        finally:
            _lib.check(lib.mui_tune_prefill(0, 0), "mui_tune_prefill")
