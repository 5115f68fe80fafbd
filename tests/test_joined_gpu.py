"""A boundary in front of the product of a single token in one launch: the bits of the two calls it stands for, at the ends of rows and chunks, and what runs as two calls
after all; in the hybrid models' layers, with hooks listening."""
import pytest
import torch

from muillm_amd import _lib, muillm_ext
from tests import salepel_util, zufadra_util
from tests.test_gemm_stream_gpu import CODE, DEV, _gen, _rand

pytestmark = pytest.mark.gpu
EPS = 1e-5


def _ptr(t):
    return None if t is None else t.data_ptr()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tokens,k", [(1, 8), (1, 1000), (1, 2048), (1, 2056), (1, 4096), (1, 4104), (3, 512), (17, 512)])
@pytest.mark.parametrize("n", [8, 72, 1000, 6400])
def test_same_bits_as_the_two_calls(n, k, tokens, dtype):
    lib, s, code, g = _lib.load(), torch.cuda.current_stream().cuda_stream, CODE[dtype], _gen(n + k)
    y, stream = _rand((tokens, k), dtype, g), torch.empty(tokens, k, device=DEV).normal_(generator=g)
    post, after, bias, up_bias = 1 + _rand((k,), dtype, g, 0.2), 1 + _rand((k,), dtype, g, 0.2), _rand((n,), dtype, g), _rand((n,), dtype, g)
    pitch = k + 8
    w, pair = _rand((n, pitch), dtype, g, k ** -0.5), _rand((n, 2, k), dtype, g, k ** -0.5)
    for p, a, old in ((post, None, stream), (post, after, stream), (None, after, stream), (None, None, stream), (post, after, None)):
        x1, h1, x2, h2 = (torch.full((tokens, k), float("nan"), dtype=t, device=DEV) for t in (torch.float32, dtype) * 2)
        one = (s, code, _ptr(old), y.data_ptr(), _ptr(p), 0.5, _ptr(a), 2.0, EPS, x1.data_ptr(), h1.data_ptr())
        _lib.check(lib.mui_residual_norm(s, code, _ptr(old), y.data_ptr(), 1.0, _ptr(p), 0.5, _ptr(a), 2.0, EPS, x2.data_ptr(), h2.data_ptr(), tokens, k), "norm")

        def same(name, o1, o2):
            assert torch.equal(x1, x2) and torch.equal(h1, h2) and torch.equal(o1, o2), name

        o1, o2 = (torch.full((tokens, n), float("nan"), dtype=dtype, device=DEV) for _ in range(2))
        _lib.check(lib.mui_joined_linear(*one, w.data_ptr(), pitch, bias.data_ptr(), o1.data_ptr(), n, k, tokens, None, 0), "linear")
        _lib.check(lib.mui_linear(s, code, w.data_ptr(), pitch, h2.data_ptr(), None, 0.0, None, bias.data_ptr(), None, o2.data_ptr(), n, k, tokens), "linear")
        same("linear", o1, o2)
        x1.fill_(float("nan"))
        _lib.check(lib.mui_joined_gateup_silu(*one, pair.data_ptr(), pair[:, 1].data_ptr(), 2 * k, bias.data_ptr(), up_bias.data_ptr(), o1.data_ptr(), n, k, tokens), "gateup")
        _lib.check(lib.mui_gateup_silu_bias(s, code, pair.data_ptr(), pair[:, 1].data_ptr(), 2 * k, h2.data_ptr(), None, 0.0, bias.data_ptr(), up_bias.data_ptr(), o2.data_ptr(), n, k,
                                            tokens), "gateup")
        same("gateup", o1, o2)
        x1.fill_(float("nan"))
        f1, f2, dense = torch.empty(tokens, n, device=DEV), torch.empty(tokens, n, device=DEV), w[:, :k].contiguous()
        _lib.check(lib.mui_joined_linear_f32(*one, dense.data_ptr(), bias.data_ptr(), f1.data_ptr(), n, k, tokens), "f32")
        _lib.check(lib.mui_linear_f32(s, code, dense.data_ptr(), h2.data_ptr(), bias.data_ptr(), f2.data_ptr(), n, k, tokens), "f32")
        same("f32", f1, f2)


def test_stream_in_place_and_refused_arguments():
    lib, s, g = _lib.load(), torch.cuda.current_stream().cuda_stream, _gen(1)
    y, w, post = _rand((1, 512), torch.bfloat16, g), _rand((64, 512), torch.bfloat16, g), _rand((512,), torch.bfloat16, g)
    stream = torch.empty(1, 512, device=DEV).normal_(generator=g)
    apart, h, out = torch.empty_like(stream), torch.empty_like(y), torch.empty(1, 64, dtype=torch.bfloat16, device=DEV)

    def call(x_in, x_out, y_ptr=y.data_ptr()):
        return lib.mui_joined_linear(s, 1, x_in.data_ptr(), y_ptr, post.data_ptr(), 1.0, None, 1.0, EPS, x_out.data_ptr(), h.data_ptr(), w.data_ptr(), 512, None, out.data_ptr(),
                                     64, 512, 1, None, 0)

    assert call(stream, apart) == 0
    first = out.clone()
    assert call(stream, stream) == 0  # (two launches)
    assert torch.equal(stream, apart) and torch.equal(out, first)
    assert call(stream, apart, None) == -1


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("where", ["y", "behind y", "stream", "gain", "h on the stream", "h on y"])
def test_outputs_on_inputs(where, dtype):
    """Where an output lies on what the boundary reads, the two calls follow each other: every workgroup would still be reading."""
    lib, s, code, g, k = _lib.load(), torch.cuda.current_stream().cuda_stream, CODE[dtype], _gen(2), 4096
    y, w, post = _rand((1, k), dtype, g), _rand((k, k), dtype, g, k ** -0.5), 1 + _rand((k,), dtype, g, 0.2)
    stream = torch.empty(1, k, device=DEV).normal_(generator=g)

    def run(name):
        pool = torch.zeros(8 * k, dtype=torch.int32, device=DEV)  # [stream | y, gain | stream behind | h, out], 4 k bytes each
        at = lambda part, n=0: pool.data_ptr() + 4 * k * part + 2 * n  # noqa: E731
        pool[:k].view(torch.float32).copy_(stream[0])
        pool[k:2 * k].view(dtype).copy_(torch.cat([y[0], post]))
        x_out, h, out = at(2), at(3), at(3, k)
        out = {"y": at(1), "behind y": at(1, k - 8), "stream": at(0, k), "gain": at(1, k)}.get(where, out)
        h = {"h on the stream": at(0, k), "h on y": at(1)}.get(where, h)
        if name:
            args = (s, code, at(0), at(1), at(1, k), 0.5, at(1, k), 2.0, EPS, x_out, h)
            if name == "mui_joined_linear":
                _lib.check(lib.mui_joined_linear(*args, w.data_ptr(), k, None, out, k, k, 1, None, 0), name)
            elif name == "mui_joined_gateup_silu":
                _lib.check(lib.mui_joined_gateup_silu(*args, w.data_ptr(), w[k // 2:].data_ptr(), k, None, None, out, k // 2, k, 1), name)
            else:
                _lib.check(lib.mui_joined_linear_f32(*args, w.data_ptr(), None, out, 256, k, 1), name)
            return pool
        return pool, (at(0), at(1), at(1, k), x_out, h, out)

    for name in ("mui_joined_linear", "mui_joined_gateup_silu", "mui_joined_linear_f32"):
        got = run(name)
        want, (x_in, y_at, gain, x_out, h, out) = run(None)
        _lib.check(lib.mui_residual_norm(s, code, x_in, y_at, 1.0, gain, 0.5, gain, 2.0, EPS, x_out, h, 1, k), "norm")
        if name == "mui_joined_linear":
            _lib.check(lib.mui_linear(s, code, w.data_ptr(), k, h, None, 0.0, None, None, None, out, k, k, 1), name)
        elif name == "mui_joined_gateup_silu":
            _lib.check(lib.mui_gateup_silu_bias(s, code, w.data_ptr(), w[k // 2:].data_ptr(), k, h, None, 0.0, None, None, out, k // 2, k, 1), name)
        else:
            _lib.check(lib.mui_linear_f32(s, code, w.data_ptr(), h, None, out, 256, k, 1), name)
        assert torch.equal(got, want), name


@torch.no_grad()
@pytest.mark.parametrize("util", [zufadra_util, salepel_util])
def test_hybrid_layers_use_it_and_hooks_are_heard(util, monkeypatch):
    cfg = util.default_config()
    lm = util.build(cfg, util.random_weights(cfg, seed=1), torch.bfloat16, DEV)
    ids = torch.randint(0, cfg["vocab"], (1, 9), generator=torch.Generator().manual_seed(2)).to(DEV)

    def steps():
        cache = lm.create_cache(1, 16)
        return torch.cat([lm(input_ids=ids[:, i:i + 1], past_key_values=cache, use_cache=True).logits.float() for i in range(ids.shape[1])], 1)

    used = []
    along = muillm_ext.ResidualFront.along
    monkeypatch.setattr(muillm_ext.ResidualFront, "along", lambda self, call: used.append(1) or along(self, call))
    fused = steps()
    assert used
    monkeypatch.setattr(muillm_ext.ResidualFront, "of", classmethod(lambda *a: None))
    apart = steps()
    assert torch.equal(fused, apart)
    monkeypatch.undo()
    # a hook on a sublayer sees, and changes, what it is documented to be given
    hook = lambda mod, args: (args[0] * 1.5,) + args[1:]  # noqa: E731
    handles = [layer.mlp.register_forward_pre_hook(hook) for layer in lm.model.layers if layer.mlp is not None]
    got = steps()
    monkeypatch.setattr(muillm_ext.ResidualFront, "of", classmethod(lambda *a: None))
    assert torch.equal(got, steps()) and not torch.equal(got, fused)
    for handle in handles:
        handle.remove()


@torch.no_grad()
@pytest.mark.parametrize("util", [zufadra_util, salepel_util])
def test_projections_that_stand_in_for_the_models_own(util):
    """A projection may be wrapped or replaced by a module that knows of no boundary in front (nor of a norm of the queries' latent): it is called as before."""
    class Around(torch.nn.Module):
        def __init__(self, linear):
            super().__init__()
            self.inner, self.weight = linear, linear.weight

        def forward(self, x):
            return self.inner(x)

    cfg = util.default_config() if util is zufadra_util else util.config([(util.latent(rot=16), util.moe()), (util.mlstm(), None), (util.latent(rot=16, window=5, kv_from=0), None)])
    lm = util.build(cfg, util.random_weights(cfg, seed=1), torch.bfloat16, DEV)
    ids = torch.randint(0, cfg["vocab"], (1, 9), generator=torch.Generator().manual_seed(2)).to(DEV)

    def steps():
        cache = lm.create_cache(1, 16)
        return torch.cat([lm(input_ids=ids[:, i:i + 1], past_key_values=cache, use_cache=True).logits.float() for i in range(ids.shape[1])], 1)

    heard = lambda m: m.register_forward_hook(lambda *a: None)  # noqa: E731
    handles = []
    for layer in lm.model.layers:
        mixer = layer.mixer
        handles += [heard(mixer.proj.linear)] if hasattr(mixer, "proj") else []
        handles += [heard(mixer.up_q)] if hasattr(mixer, "up_q") else []
    want = steps()  # with a hook that listens each of them is called by itself
    for handle in handles:
        handle.remove()
    for layer in lm.model.layers:
        mixer = layer.mixer
        if hasattr(mixer, "proj"):
            mixer.proj.linear = Around(mixer.proj.linear)
        if hasattr(mixer, "up_q"):
            mixer.up_q = Around(mixer.up_q)
    assert torch.equal(steps(), want)
