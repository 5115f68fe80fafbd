"""What the descriptors of the single-call layer stacks are made from, and when they no longer hold. Examined on the CPU with tensors that say they are on a GPU: nothing is launched."""
import ctypes

import pytest
import torch

from muillm_amd import _lib
from muillm_amd.engineconfig import MuiEngineConfig
from muillm_amd.modules.decoder.decoderstack import MuiDecoderStack, MuiPromptStack
from muillm_amd.modules.models.llama.model import MuiDecoderConfig, MuiLlamaForCausalLM


def _lm(**kw):
    cfg = MuiDecoderConfig(**{**dict(hidden_size=512, intermediate_size=1280, num_hidden_layers=2, num_attention_heads=4, num_key_value_heads=2, vocab_size=32,
                                     max_position_embeddings=128), **kw})
    return MuiLlamaForCausalLM.from_config(MuiEngineConfig(), cfg, dtype=torch.bfloat16, device="cpu", seed=0, init_std=0.05).eval()


@pytest.fixture
def lm(monkeypatch):
    lm = _lm()
    lm.cache = lm.create_cache(2, 64)
    monkeypatch.setattr(torch.Tensor, "is_cuda", property(lambda self: True))
    for rotary in [lm.model.rotary_emb] + [layer.self_attn.rotary_emb for layer in lm.model.layers]:
        rotary.dispatchable = True
    for layer in lm.model.layers:
        layer.mlp.dispatchable = True
    return lm


def _prompt_stack(lm):
    assert MuiPromptStack.eligible(lm.model.layers, lm.model.rotary_emb, lm.cache)
    return MuiPromptStack(lm.model.layers, lm.model.rotary_emb, lm.cache)


def _takes(stack, t=20, b=1):
    ids = torch.arange(t)
    with torch.no_grad():
        return stack.takes(torch.zeros(b, t, 512, dtype=torch.bfloat16), ids[None], ids, None)


def test_no_row_beyond_the_cache_is_read(lm):
    stack, at = _prompt_stack(lm), ctypes.c_void_p(256)
    for tokens, seq_len in ((20, 65), (64, 1 << 20), (1, 65)):
        status = _lib.load().mui_decoder_stack_prompt(None, ctypes.byref(stack.desc), 1, tokens, at, at, at, 0, at, seq_len, None, 0, 1, at, None, 0)
        assert status == -1  # MUI_ERR_INVALID_ARG, and nothing enqueued
    lm.cache.set_seen_tokens(44)
    assert _takes(stack, 20) and not _takes(stack, 21)


def _eligible(lm):
    found = [MuiDecoderStack.eligible(lm.model.layers, lm.model.rotary_emb, lm.cache, 1), MuiPromptStack.eligible(lm.model.layers, lm.model.rotary_emb, lm.cache)]
    assert found[0] == found[1]
    return found[0]


def test_layers_of_other_sizes(lm, monkeypatch):
    """One descriptor states the sizes of all layers: a narrower one would be read beyond its ends."""
    assert _eligible(lm)
    layer = lm.model.layers[1]
    with monkeypatch.context() as m:
        m.undo()
        narrow, more_heads = _lm(intermediate_size=640).model.layers[1], _lm(num_key_value_heads=4).model.layers[1]
    narrow.mlp.dispatchable = more_heads.self_attn.rotary_emb.dispatchable = True
    mlp, layer.mlp = layer.mlp, narrow.mlp
    assert not _eligible(lm)
    layer.mlp = mlp
    qkv, attn = layer.qkv_proj, layer.self_attn
    layer.qkv_proj, layer.self_attn = more_heads.qkv_proj, more_heads.self_attn
    assert not _eligible(lm)
    layer.qkv_proj, layer.self_attn = qkv, attn
    assert _eligible(lm)
    # tensors that are not of their modules' sizes
    for m, name in ((mlp.gate_proj, "weight"), (mlp.down_proj, "weight"), (attn.o_proj, "weight"), (qkv.linear, "weight"), (mlp, "norm_weights"), (qkv.linear, "norm_weights")):
        plain = getattr(m, name)
        setattr(m, name, torch.nn.Parameter(plain.detach()[:8], requires_grad=False))
        assert not _eligible(lm), (type(m), name)
        setattr(m, name, plain)
    assert _eligible(lm)


def test_layers_of_other_tables(lm, monkeypatch):
    """A layer rotates with its own module's tables, whatever the model's module holds."""
    steps, prompts = MuiDecoderStack(lm.model.layers, lm.model.rotary_emb, lm.cache, 1), _prompt_stack(lm)
    prompts.remember()
    asked = (lambda: steps.matches(lm.model.layers, lm.cache, 1), lambda: prompts.current(lm.model.layers))
    assert _eligible(lm) and all(a() for a in asked)
    with monkeypatch.context() as m:
        m.undo()
        other = _lm(rope_theta=1e4).model.rotary_emb
    other.dispatchable = True
    rotary = lm.model.layers[1].self_attn.rotary_emb
    assert other.cos32 is not rotary.cos32 and lm.model.rotary_emb.cos32 is rotary.cos32
    # a table built anew in place, in the module and (for prompts) in its handle; another module
    for owner, name in ((rotary, "cos32"), (rotary, "sin32"), (lm.model.layers[1].self_attn, "rotary_emb")):
        plain = getattr(owner, name)
        setattr(owner, name, getattr(other, name, other))
        assert not _eligible(lm) and not any(a() for a in asked), name
        setattr(owner, name, plain)
        assert _eligible(lm) and all(a() for a in asked)
    lm.model.layers[1].self_attn.rotary_emb = None
    assert not _eligible(lm) and not any(a() for a in asked)
    lm.model.layers[1].self_attn.rotary_emb = rotary
    rotary.cpp_module.sin32 = other.sin32
    assert not asked[1]() and not MuiPromptStack.eligible(lm.model.layers, lm.model.rotary_emb, lm.cache)
    rotary.cpp_module.sin32 = rotary.sin32
    # the model's own module rotates no layer
    lm.model.rotary_emb = other
    assert MuiDecoderStack(lm.model.layers, other, lm.cache, 1).cos32 is rotary.cos32 and _prompt_stack(lm).cos32 is rotary.cos32


def _watching(lm):
    stack = _prompt_stack(lm)
    stack.remember()
    assert stack.current(lm.model.layers) and stack.holds(lm.cache)
    return stack


def test_tensors_may_be_swapped(lm):
    """... as module.to() and load_state_dict() do it where they are told to, and it is noticed."""
    for m in (lm.model.layers[0].mlp.down_proj, lm.model.layers[1].qkv_proj.linear):
        stack = _watching(lm)
        torch.utils.swap_tensors(m.weight, torch.nn.Parameter(m.weight.detach().clone(), requires_grad=False))
        assert not stack.current(lm.model.layers)
    stack = _watching(lm)
    torch.utils.swap_tensors(lm.cache.key_cache[1], lm.cache.key_cache[1].clone())
    assert not stack.holds(lm.cache)


def test_the_same_address_read_otherwise(lm):
    layer = lm.model.layers[0]
    for m, name in ((layer.self_attn.o_proj, "weight"), (layer.mlp.down_proj, "weight"), (layer.qkv_proj.linear, "norm_weights")):
        t = getattr(m, name)
        plain = t.data
        for other in (plain.view(torch.float16), plain[:256], plain.reshape(-1, 256).T):
            stack = _watching(lm)
            t.data = other
            assert other.data_ptr() == plain.data_ptr() and not stack.current(lm.model.layers), (name, other.shape, other.dtype)
            t.data = plain
            assert stack.current(lm.model.layers)


def test_weights_that_are_plain_tensors(lm):
    """A parameter that was deleted and set again as a tensor, or as a buffer, is what the modules read."""
    mlp = lm.model.layers[0].mlp
    for m in (mlp.gate_proj, mlp.up_proj, mlp.down_proj):
        def another():
            return torch.empty(m.out_features, m.in_features, dtype=torch.bfloat16)

        del m.weight
        m.weight = another()
        if m is mlp.up_proj:
            mlp.gate_proj.weight = another()  # (the two have one pitch)
        if m is mlp.gate_proj:
            del mlp.up_proj.weight
            mlp.up_proj.weight = torch.nn.Parameter(another(), requires_grad=False)
        kept, stack = m.weight, _watching(lm)
        m.weight = another()
        assert not stack.current(lm.model.layers)
        m.weight = kept
        assert stack.current(lm.model.layers)
        del m.weight
        m.register_buffer("weight", another())
        stack = _watching(lm)
        m.weight = another()
        assert not stack.current(lm.model.layers)


def test_steps_notice_other_memory_and_modules(lm):
    layers, model = lm.model.layers, lm.model
    steps = MuiDecoderStack(layers, model.rotary_emb, lm.cache, 1)
    assert steps.matches(layers, lm.cache, 1)
    for m in (layers[1].mlp.gate_proj, layers[0].mlp.down_proj, layers[1].qkv_proj.linear, layers[0].self_attn.o_proj):
        plain = m.weight.data
        m.weight.data = plain.clone()
        assert not steps.matches(layers, lm.cache, 1)
        m.weight.data = plain
        assert steps.matches(layers, lm.cache, 1)
    for name in ("gate_proj", "up_proj", "down_proj"):
        plain = getattr(layers[1].mlp, name)
        setattr(layers[1].mlp, name, getattr(layers[0].mlp, name))
        assert not steps.matches(layers, lm.cache, 1)
        setattr(layers[1].mlp, name, plain)
    assert steps.matches(layers, lm.cache, 1)


def test_what_may_be_set_after_a_prompt(lm, monkeypatch):
    """The number of tokens from which prompts use torch's attention, on a module or on the class; attributes that appear where there were none, or go."""
    stack, layers = _watching(lm), lm.model.layers
    assert _takes(stack)
    attn = layers[1].self_attn
    attn.prefill_kernel_max_tokens = 19
    assert not _takes(stack) and _takes(stack, 19)
    del attn.prefill_kernel_max_tokens
    with monkeypatch.context() as m:
        m.setattr(type(attn), "prefill_kernel_max_tokens", 19)
        assert not _takes(stack)
    assert _takes(stack) and stack.current(layers)
    for m, name, value in ((layers[0].mlp.down_proj, "normalize", True), (layers[0].mlp, "method", None), (layers[0].mlp, "intermediate_size", 640), (attn, "training", True),
                           (layers[1].qkv_proj.linear, "variance_epsilon", 1e-3), (layers[1].qkv_proj, "slice_starts", [0, 512, 640]), (attn.o_proj, "cpp_module", None)):
        before = m.__dict__.get(name, m)
        setattr(m, name, value)
        assert not stack.current(layers), name
        delattr(m, name) if before is m else setattr(m, name, before)
        assert stack.current(layers), name
    # what has gone does not pass for what never was
    attn.o_proj.cpp_module = None
    assert not stack.current(layers)
    attn.o_proj.finalize_init()
    stack = _watching(lm)
    layers[0].mlp = None
    assert not stack.current(layers)
    unread = MuiPromptStack.__new__(MuiPromptStack)  # what could not be read is not the same as before
    unread.__dict__.update(stack.__dict__, _watched=None)
    unread.remember()
    assert unread._watched[0] is None and not unread.current(layers)


def test_tensors_of_another_type(lm):
    """The modules refuse them; one descriptor has one type."""
    mlp, qkv, o = lm.model.layers[1].mlp, lm.model.layers[1].qkv_proj.linear, lm.model.layers[1].self_attn.o_proj
    for m, name in ((mlp.gate_proj, "weight"), (mlp.up_proj, "weight"), (mlp.down_proj, "weight"), (mlp, "norm_weights"), (qkv, "weight"), (qkv, "norm_weights"), (o, "weight")):
        for dtype in (torch.float32, torch.float16):
            t = getattr(m, name)
            plain = t.data
            t.data = plain.to(dtype).as_strided(plain.shape, plain.stride()) if plain.is_contiguous() else torch.empty_strided(plain.shape, plain.stride(), dtype=dtype)
            assert not _eligible(lm), (type(m), name)
            t.data = plain
    assert _eligible(lm)


def test_handles_that_name_other_tensors(lm):
    """A projection's module computes by its handle, which names the tensors of the last finalize_init()."""
    qkv, o = lm.model.layers[1].qkv_proj.linear, lm.model.layers[0].self_attn.o_proj
    for m, name, value in ((qkv, "norm_weights", torch.nn.Parameter(2 * qkv.norm_weights.detach(), requires_grad=False)), (qkv, "variance_epsilon", 1e-5),
                           (o, "weight", torch.nn.Parameter(2 * o.weight.detach(), requires_grad=False))):
        stack, before = _watching(lm), getattr(m, name)
        lm_eps = [(x.qkv_proj.linear, x.mlp) for x in lm.model.layers]
        if name == "variance_epsilon":  # (of all layers: one descriptor has one)
            value = 2 * before
            for x, y in lm_eps:
                x.variance_epsilon = y.variance_epsilon = value
        else:
            setattr(m, name, value)
        assert not stack.current(lm.model.layers) and not MuiPromptStack.eligible(lm.model.layers, lm.model.rotary_emb, lm.cache), name
        for x, _ in lm_eps:
            x.finalize_init()
        o.finalize_init()
        assert MuiPromptStack.eligible(lm.model.layers, lm.model.rotary_emb, lm.cache), name
