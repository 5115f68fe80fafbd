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


@pytest.mark.parametrize("n,k,tokens", [(6144, 8192, 1281), (6144, 8192, 1500), (4096, 14336, 1345)])
def test_more_scratch_than_asked_for(n, k, tokens):
    """... changes neither whether K is shared nor the sums: shares that only a larger one would hold are not taken."""
    g, dtype = _gen(n + k + tokens), torch.float16
    w, x, res = _rand((n, k), dtype, g, k ** -0.5), _rand((tokens, k), dtype, g), _rand((tokens, n), dtype, g)
    size = _lib.load().mui_linear_workspace_bytes()
    assert torch.equal(*(_linear(x, w, None, None, res, torch.zeros(b, dtype=torch.uint8, device=DEV)) for b in (size, 4 * size)))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,k,tokens", [(4100, 14336, 333), (2052, 8192, 768), (1004, 6144, 1300)])
def test_rows_of_whole_fours_with_the_norm_behind(n, k, tokens, dtype):
    """K is shared for rows that are no multiple of eight, but the launch that takes the norm along moves eight values at a time: these are two calls, and nothing behind the
    outputs is written."""
    lib, s, code, guard = _lib.load(), torch.cuda.current_stream().cuda_stream, CODE[dtype], 64
    assert prompt_shares("fp16" if dtype == torch.float16 else "bf16", n, k, tokens)[1] > 1
    g = _gen(n + k + tokens)
    w, x, res = _rand((n, k), dtype, g, k ** -0.5), _rand((tokens, k), dtype, g), _rand((tokens, n), dtype, g)
    post, after = 1 + _rand((n,), dtype, g, 0.2), 1 + _rand((n,), dtype, g, 0.2)
    stream = torch.empty(tokens, n, device=DEV).normal_(generator=g)
    ws = torch.zeros(lib.mui_linear_workspace_bytes(), dtype=torch.uint8, device=DEV)

    def guarded(kind):
        buffer = torch.full((tokens * n + guard,), 7.0, dtype=kind, device=DEV)
        return buffer[:tokens * n].view(tokens, n), buffer[tokens * n:]

    (y, y_end), (h, h_end), (out, out_end) = guarded(dtype), guarded(dtype), guarded(torch.float32)
    y2, h2, out2 = _linear(x, w, None, None, res, ws), torch.empty_like(res), torch.empty_like(stream)
    _lib.check(lib.mui_rmsnorm(s, code, after.data_ptr(), y2.data_ptr(), EPS, h2.data_ptr(), tokens, n), "norm")
    _call("mui_linear_norm", x, w, k, None, (res.data_ptr(), after.data_ptr(), EPS, y.data_ptr(), h.data_ptr()), y, ws)
    assert torch.equal(y, y2) and torch.equal(h, h2)
    plain = x.double() @ w.double().T
    _close(h, _rms(plain + res.double(), after.double()), 2 * HALF_ULP[dtype])
    y2 = _linear(x, w, None, None, None, ws)
    _lib.check(lib.mui_residual_norm(s, code, stream.data_ptr(), y2.data_ptr(), 1.0, post.data_ptr(), 0.5, after.data_ptr(), 2.0, EPS, out2.data_ptr(), h2.data_ptr(), tokens, n), "norm")
    _call("mui_linear_residual_norm", x, w, k, None, (stream.data_ptr(), post.data_ptr(), 0.5, after.data_ptr(), 2.0, EPS, y.data_ptr(), out.data_ptr(), h.data_ptr()), y, ws)
    assert torch.equal(y, y2) and torch.equal(out, out2) and torch.equal(h, h2)
    for end in (y_end, h_end, out_end):
        assert bool((end == 7.0).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shift", [0, 6, 7])
@pytest.mark.parametrize("tile,shares", [(7, 7), (8, 3), (4, 5)])
@pytest.mark.parametrize("n,k,tokens", [(4, 3072, 65), (260, 3200, 257), (4104, 2816, 300)])
def test_codes(n, k, tokens, tile, shares, shift, dtype, tune):
    """int8 with a scale per row (shift 0) and in groups: forced shares, and the same without scratch. Groups in bf16 are left whole."""
    lib, s, g = _lib.load(), torch.cuda.current_stream().cuda_stream, _gen(n + k + tokens + shift)
    q = torch.randint(-128, 128, (n, k), device=DEV, generator=g, dtype=torch.int16)
    x, res, bias = _rand((tokens, k), dtype, g), _rand((tokens, n), dtype, g), _rand((n,), dtype, g)
    if shift:
        groups = k >> shift
        scale = (torch.rand(n, groups, device=DEV, generator=g) * 2e-3 + 1e-3).to(dtype)
        pairs = torch.stack([scale, (scale.float() * -128).to(dtype)], 2).contiguous()
        codes = (q + 128).to(torch.uint8)
        w = (codes.float().view(n, groups, -1) * pairs[..., :1].float() + pairs[..., 1:].float()).to(dtype).double().view(n, k)  # (what is multiplied is rounded)
    else:
        pairs, codes = (torch.rand(n, device=DEV, generator=g) * 2e-3 + 1e-3).to(dtype), q.to(torch.int8)
        w = codes.double() * pairs.double()[:, None]
    ref = x.double() @ w.T + bias.double() + res.double()
    ws = torch.zeros(lib.mui_linear_workspace_bytes(), dtype=torch.uint8, device=DEV)
    tune(tile, shares)
    for scratch in (ws, None):
        y = torch.full((tokens, n), float("nan"), dtype=dtype, device=DEV)
        end = (x.data_ptr(), None, 0.0, bias.data_ptr(), res.data_ptr(), y.data_ptr(), n, k, tokens, _ptr(scratch), 0 if scratch is None else scratch.numel())
        if shift:
            _lib.check(lib.mui_int8_group_linear_ws(s, CODE[dtype], codes.data_ptr(), k, pairs.data_ptr(), shift, *end), "groups")
        else:
            _lib.check(lib.mui_int8_linear_ws(s, CODE[dtype], codes.data_ptr(), k, pairs.data_ptr(), *end), "rows")
        _close(y, ref, 2 * HALF_ULP[dtype])
    assert bool(ws[4096:].any()) == (not shift or dtype == torch.float16)


@torch.no_grad()
@pytest.mark.parametrize("group", [0, 128])
def test_int8_prompts_in_one_call_and_layer_by_layer(group, monkeypatch):
    """The norms behind shared linears, taken along in the single call, give the bits of the layers' own calls."""
    from muillm_amd.engine import init_engine
    from muillm_amd.engineconfig import MuiEngineConfig
    from muillm_amd.modules.models.llama.model import MuiDecoderConfig, MuiLlamaForCausalLM
    from muillm_amd.quantization.quantizationmethod import Int8WeightOnlyQuantizationMethod

    torch.manual_seed(3)
    config = MuiDecoderConfig(hidden_size=2048, intermediate_size=8192, num_hidden_layers=2, num_attention_heads=16, num_key_value_heads=4, vocab_size=512)
    lm = MuiLlamaForCausalLM.from_config(MuiEngineConfig(), config, dtype=torch.float16, device=DEV, finalize=False)
    lm = init_engine(lm, device=DEV, engine_config=MuiEngineConfig(Int8WeightOnlyQuantizationMethod(group_size=group, modules=["qkv_proj", "o_proj", "mlp"])))
    assert prompt_shares("int8_group" if group else "int8", 2048, 8192, 150)[1] > 1
    ids = torch.randint(0, 512, (1, 150), generator=torch.Generator().manual_seed(4)).to(DEV)

    def logits():
        cache = lm.create_cache(1, 160)
        return lm(input_ids=ids, past_key_values=cache, use_cache=True, all_ones_mask=True).logits

    one = logits()
    handle = lm.model.norm.register_forward_pre_hook(lambda *a: None)
    hooks = [layer.self_attn.o_proj.register_forward_hook(lambda *a: None) for layer in lm.model.layers]
    apart = logits()
    for h in [handle] + hooks:
        h.remove()
    assert bool(torch.isfinite(one).all()) and torch.equal(one, apart)
