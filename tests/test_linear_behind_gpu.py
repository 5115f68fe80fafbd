"""A linear with the norm (and the residual stream) behind it in one call, against the same in 64 bits, at the sizes where its forms end: the shares of K, the
threads of a row, and what stays two launches. Gate: fp32 accumulation (k 2^-24 of the sum of the products' magnitudes) and the roundings to 16 bits
of y and h; a norm hands y's on, in proportion."""

import pytest
import torch

from muillm_amd import _lib, muillm_ext
from tests import zufadra_util
from tests.test_gemm_stream_gpu import CODE, DEV, HALF_ULP, _gen, _rand

pytestmark = pytest.mark.gpu
EPS = 1e-5


def _ptr(t):
    return None if t is None else t.data_ptr()


def _rms(x, gain):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * gain


def _call(name, x, w, pitch, bias, args, y, ws):
    (tokens, k), n = x.shape, w.shape[0]
    _lib.check(getattr(_lib.load(), name)(torch.cuda.current_stream().cuda_stream, CODE[x.dtype], w.data_ptr(), pitch, x.data_ptr(), _ptr(bias), *args, n, k, tokens,
                                          _ptr(ws), 0 if ws is None else ws.numel()), name)
    return y


def _close(got, ref, rel):
    """Root mean square of the difference over that of the result, and no single value far out."""
    assert bool(torch.isfinite(got).all())
    off, size = (got.double() - ref), ref.pow(2).mean().sqrt()
    assert float(off.pow(2).mean().sqrt() / size) <= rel
    assert float(off.abs().max() / torch.maximum(ref.abs(), size).max()) <= 4 * rel


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tokens", [1, 16, 17, 32, 33, 64, 65, 97, 128, 129])
@pytest.mark.parametrize("n,k", [(8, 1024), (1000, 2048), (2048, 512), (2056, 4096), (4096, 4096), (4104, 1280), (8192, 1024), (8200, 1024), (1024, 14336), (104, 520)])
def test_against_64_bits(n, k, tokens, dtype):
    g = _gen(n + k + tokens)
    pitch = k + 8
    w = _rand((n, pitch), dtype, g, k ** -0.5)[:, :k]
    x, res, bias = _rand((tokens, k), dtype, g), _rand((tokens, n), dtype, g), _rand((n,), dtype, g, 0.5)
    post, after = 1 + _rand((n,), dtype, g, 0.2), 1 + _rand((n,), dtype, g, 0.2)
    stream = torch.empty(tokens, n, device=DEV).normal_(0.0, 1.0, generator=g)
    ws = torch.zeros(_lib.load().mui_linear_workspace_bytes(), dtype=torch.uint8, device=DEV)
    plain = x.double() @ w.double().T
    # roundings: of y (once, in proportion) and of h; the sums' share is far below
    rel = 2 * HALF_ULP[dtype]
    for scratch in (ws, None):
        for add in (bias, None):
            ref = plain + res.double() + (0 if add is None else add.double())
            y, h = torch.empty_like(res), torch.empty_like(res)
            _call("mui_linear_norm", x, w, pitch, add, (res.data_ptr(), after.data_ptr(), EPS, y.data_ptr(), h.data_ptr()), y, scratch)
            _close(y, ref, rel)
            _close(h, _rms(ref, after.double()), rel)
            ref = plain + (0 if add is None else add.double())
            for p, a, old in ((post, after, stream), (post, None, stream), (None, after, None)):
                out, h = torch.empty_like(stream), torch.empty_like(res)
                _call("mui_linear_residual_norm", x, w, pitch, add, (_ptr(old), _ptr(p), 0.5, _ptr(a), 2.0, EPS, y.data_ptr(), out.data_ptr(), h.data_ptr()), y, scratch)
                want = (ref if p is None else 0.5 * _rms(ref, p.double())) + (0 if old is None else old.double())
                _close(y, ref, rel)
                _close(out, want, rel)
                _close(h, 2.0 * (want if a is None else _rms(want, a.double())), rel)
    assert not bool(ws[:4096].any())  # the counters


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tokens", [17, 20, 32, 48, 64, 65, 97, 128])
@pytest.mark.parametrize("n,k", [(1024, 14336), (2048, 2048), (2048, 8192), (4096, 4096), (4096, 14336), (8192, 1024)])
def test_same_bits_as_the_two_calls(n, k, tokens, dtype):
    """K divided (long K, few outputs) and undivided: what is taken along is what two calls give, bit for bit."""
    g = _gen(n + k + tokens)
    w, x, res = _rand((n, k), dtype, g, k ** -0.5), _rand((tokens, k), dtype, g), _rand((tokens, n), dtype, g)
    post, after = 1 + _rand((n,), dtype, g, 0.2), 1 + _rand((n,), dtype, g, 0.2)
    stream = torch.empty(tokens, n, device=DEV).normal_(0.0, 1.0, generator=g)
    ws = torch.zeros(_lib.load().mui_linear_workspace_bytes(), dtype=torch.uint8, device=DEV)
    lib, s, code = _lib.load(), torch.cuda.current_stream().cuda_stream, CODE[dtype]

    def linear(residual):
        y = torch.empty_like(res)
        _lib.check(lib.mui_linear_ws(s, code, w.data_ptr(), k, x.data_ptr(), None, 0.0, None, None, _ptr(residual), y.data_ptr(), n, k, tokens, ws.data_ptr(), ws.numel()), "linear")
        return y

    y, h, out = torch.empty_like(res), torch.empty_like(res), torch.empty_like(stream)
    y2, h2, out2 = linear(res), torch.empty_like(res), torch.empty_like(stream)
    _lib.check(lib.mui_rmsnorm(s, code, after.data_ptr(), y2.data_ptr(), EPS, h2.data_ptr(), tokens, n), "norm")
    _call("mui_linear_norm", x, w, k, None, (res.data_ptr(), after.data_ptr(), EPS, y.data_ptr(), h.data_ptr()), y, ws)
    assert torch.equal(y, y2) and torch.equal(h, h2)
    y2 = linear(None)
    _lib.check(lib.mui_residual_norm(s, code, stream.data_ptr(), y2.data_ptr(), 1.0, post.data_ptr(), 0.5, after.data_ptr(), 2.0, EPS, out2.data_ptr(), h2.data_ptr(), tokens, n), "norm")
    _call("mui_linear_residual_norm", x, w, k, None, (stream.data_ptr(), post.data_ptr(), 0.5, after.data_ptr(), 2.0, EPS, y.data_ptr(), out.data_ptr(), h.data_ptr()), y, ws)
    assert torch.equal(y, y2) and torch.equal(out, out2) and torch.equal(h, h2)


def test_in_place_and_empty_rows():
    """The stream may be updated in place; a row of zeros stays one."""
    g = _gen(1)
    x, w = _rand((20, 2048), torch.bfloat16, g), _rand((2048, 2048), torch.bfloat16, g, 2048 ** -0.5)
    x[3] = 0
    gain = torch.ones(2048, dtype=torch.bfloat16, device=DEV)
    ws = torch.zeros(_lib.load().mui_linear_workspace_bytes(), dtype=torch.uint8, device=DEV)
    stream = torch.empty(20, 2048, device=DEV).normal_(generator=g)
    stream[3] = 0
    apart, h, y = torch.empty_like(stream), torch.empty_like(x), torch.empty_like(x)
    _call("mui_linear_residual_norm", x, w, 2048, None, (stream.data_ptr(), gain.data_ptr(), 1.0, gain.data_ptr(), 1.0, EPS, y.data_ptr(), apart.data_ptr(), h.data_ptr()), y, ws)
    assert not bool(h[3].any()) and not bool(apart[3].any())
    first = h.clone()
    _call("mui_linear_residual_norm", x, w, 2048, None, (stream.data_ptr(), gain.data_ptr(), 1.0, gain.data_ptr(), 1.0, EPS, y.data_ptr(), stream.data_ptr(), h.data_ptr()), y, ws)
    assert torch.equal(stream, apart) and torch.equal(h, first)


@torch.no_grad()
def test_hybrid_layers_use_it_and_hooks_are_heard(monkeypatch):
    cfg = zufadra_util.default_config()
    lm = zufadra_util.build(cfg, zufadra_util.random_weights(cfg, seed=1), torch.bfloat16, DEV)
    ids = torch.randint(0, cfg["vocab"], (1, 60), generator=torch.Generator().manual_seed(2)).to(DEV)
    taken = []
    plain_take = muillm_ext.ResidualBehind.take
    monkeypatch.setattr(muillm_ext.ResidualBehind, "take", lambda self, y: taken.append(plain_take(self, y)) or taken[-1])
    fused = lm(input_ids=ids).logits.float()
    assert taken and all(r is not None for r in taken)
    monkeypatch.setattr(muillm_ext.ResidualBehind, "linear", lambda *a: False)
    taken.clear()
    apart = lm(input_ids=ids).logits.float()
    assert taken and all(r is None for r in taken)
    assert torch.equal(fused, apart)
    hook = lambda mod, args, out: out + 1.0  # noqa: E731
    handles = [layer.mixer.out_proj.register_forward_hook(hook) for layer in lm.model.layers]
    want = lm(input_ids=ids).logits.float()
    monkeypatch.undo()
    got = lm(input_ids=ids).logits.float()
    for h in handles:
        h.remove()
    assert float((got - want).norm() / want.norm()) < 0.03 and float((got - fused).norm() / fused.norm()) > 0.1


def test_hybrid_layers_give_the_same_bits_whoever_listens():
    """... and whether or not versions can be asked for (inference mode): the boundary is then joined behind the call. Writes without a version and forwards of an instance count."""
    cfg = zufadra_util.default_config()
    lm = zufadra_util.build(cfg, zufadra_util.random_weights(cfg, seed=1), torch.bfloat16, DEV)
    ids = torch.randint(0, cfg["vocab"], (1, 60), generator=torch.Generator().manual_seed(2)).to(DEV)
    outs = [m.mixer.out_proj for m in lm.model.layers]

    @torch.no_grad()
    def run():
        return lm(input_ids=ids).logits.float()

    plain = run()
    with torch.inference_mode():
        assert torch.equal(lm(input_ids=ids).logits.float(), plain)

    def hooked(hook):
        handles = [m.register_forward_hook(hook) for m in outs]
        try:
            return run()
        finally:
            for h in handles:
                h.remove()

    assert torch.equal(hooked(lambda mod, args, out: None), plain)
    shifted = hooked(lambda mod, args, out: out + 1.0)
    assert not torch.equal(shifted, plain)

    def unseen(mod, args, out):
        out.data.add_(1.0)

    assert torch.equal(hooked(unseen), shifted)
    for m in lm.model.layers:
        m.mixer.forward = lambda h, cache, cache_position, f=m.mixer.forward: f(h, cache, cache_position)
    assert torch.equal(run(), plain)
    for m in lm.model.layers:
        del m.mixer.forward
        m.mixer.out_proj.forward = lambda x, f=m.mixer.out_proj.forward: f(x)
    assert torch.equal(run(), plain)
