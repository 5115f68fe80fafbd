"""Prompts, and steps of more rows than the decode kernels take, through one library call against the same layers called one by one: plain and int8 weights, several
turns, padding, captured steps; and what has to stay with the single layers. The two run the same products and sums: the same bits."""

import ctypes

import pytest
import torch

from muillm_amd import _lib, muillm_ext
from muillm_amd.engine import init_engine
from muillm_amd.engineconfig import MuiEngineConfig
from muillm_amd.modules.decoder.decoderstack import MuiPromptStack
from muillm_amd.modules.models.graphdecoder import MuiGraphDecoder
from muillm_amd.modules.models.llama.model import MuiDecoderConfig, MuiLlamaForCausalLM
from muillm_amd.quantization.quantizationmethod import Int8WeightOnlyQuantizationMethod

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _lm(dtype=torch.bfloat16, group=None, **kw):
    cfg = MuiDecoderConfig(**{**dict(hidden_size=512, intermediate_size=1280, num_hidden_layers=3, num_attention_heads=4, num_key_value_heads=2, vocab_size=512,
                                     max_position_embeddings=2048), **kw})
    lm = MuiLlamaForCausalLM.from_config(MuiEngineConfig(), cfg, dtype=dtype, device=DEV, seed=0, init_std=0.05, finalize=group is None)
    if group is None:
        return lm
    method = Int8WeightOnlyQuantizationMethod(group_size=group, modules=["qkv_proj", "o_proj", "mlp"])
    return init_engine(lm, device=DEV, engine_config=MuiEngineConfig(method))


def _ids(b, t, seed=3):
    return torch.randint(0, 512, (b, t), generator=torch.Generator().manual_seed(seed)).to(DEV)


def _run(lm, one_call, turns, capacity, batch, mask=None):
    """Logits of every turn and the cache, and whether the stack has run."""
    calls = []
    plain = MuiPromptStack.run

    def counted(self, *a):
        calls.append(a[0].shape)
        return plain(self, *a)

    lm.model.use_decoder_stack = one_call
    MuiPromptStack.run = counted
    try:
        cache = lm.create_cache(batch, capacity)
        out = [lm(input_ids=ids, past_key_values=cache, attention_mask=mask if i == 0 else None, all_ones_mask=mask is None).logits.float()
               for i, ids in enumerate(turns)]
        seen = cache.get_seq_length()
        return torch.cat(out, 1), torch.stack(cache.tensors())[..., :seen, :].float(), len(calls), seen
    finally:
        MuiPromptStack.run = plain
        lm.model.use_decoder_stack = True


def _off(a, b):
    return float((a - b).norm() / b.norm())


@torch.no_grad()
@pytest.mark.parametrize("kind", ["bf16", "fp16", "int8", "int8_group"])
@pytest.mark.parametrize("batch,lengths", [(1, [5]), (1, [16]), (1, [17]), (3, [6]), (1, [101, 2, 40]), (2, [64, 65]), (1, [300]), (20, [1, 1]), (17, [3, 1])])
def test_same_as_layer_by_layer(kind, batch, lengths):
    lm = _lm(torch.bfloat16 if kind == "bf16" else torch.float16, {"int8": 0, "int8_group": 128}.get(kind))
    turns = [_ids(batch, t, seed=t + i) for i, t in enumerate(lengths)]
    got, cache, calls, seen = _run(lm, True, turns, 512, batch)
    want, cache_want, none, seen_want = _run(lm, False, turns, 512, batch)
    assert calls == len(turns) and none == 0 and seen == seen_want == sum(lengths)
    assert torch.equal(got, want) and torch.equal(cache, cache_want)


@torch.no_grad()
@pytest.mark.parametrize("t", [40, 150])
def test_padded_prompts(t):
    lm, batch = _lm(), 4
    ids = _ids(batch, t)
    mask = torch.ones(batch, t, dtype=torch.int64, device=DEV)
    mask[0, :t // 2] = 0
    mask[2, :3] = 0
    got, _, calls, _ = _run(lm, True, [ids * mask], 512, batch, mask)
    want, _, _, _ = _run(lm, False, [ids * mask], 512, batch, mask)
    assert calls == 1
    live = mask.bool()
    assert torch.equal(got[live], want[live])


@torch.no_grad()
@pytest.mark.parametrize("padded", [False, True])
def test_captured_steps_of_many_rows(padded):
    lm, batch, t = _lm(), 20, 7
    ids = _ids(batch, t)
    mask = None
    if padded:
        mask = torch.ones(batch, t, dtype=torch.int64, device=DEV)
        mask[::2, :3] = 0
        ids = ids * mask
    shapes, plain = [], MuiPromptStack.run

    def counted(self, *a):
        shapes.append(tuple(a[0].shape[:2]))
        return plain(self, *a)

    MuiPromptStack.run = counted
    found = []
    try:
        for one_call in (True, False):
            lm.model.use_decoder_stack = one_call
            for graph in (True, False):
                decoder = MuiGraphDecoder(lm, use_graph=graph)
                for _ in range(2):
                    del shapes[:]
                    cache = lm.create_cache(batch, 64)
                    decoder.prefill(ids, 12, cache, attention_mask=mask)
                    decoder.decode(11)
                    found.append((decoder.out_tokens.clone(), decoder.logits.clone()))
                    # the prompt, and every step that is not a replay, by the call that is asked for
                    assert (shapes.count((batch, t)), (batch, 1) in shapes or graph) == (1, True) if one_call else not shapes
    finally:
        MuiPromptStack.run = plain
        lm.model.use_decoder_stack = True
    assert all(torch.equal(found[0][0], x) and torch.equal(found[0][1], y) for x, y in found[1:])


@torch.no_grad()
@pytest.mark.parametrize("batch,t", [(1, 20), (1, 101), (2, 64), (20, 1)])
def test_same_bits_where_k_is_divided(batch, t):
    """Long rows, few outputs: the linears share K between workgroups, and the launch that adds the shares takes the norm along."""
    lm = _lm(hidden_size=2048, intermediate_size=8192, num_hidden_layers=2, num_attention_heads=16, num_key_value_heads=4)
    turns = [_ids(batch, t), _ids(batch, t, seed=4)]
    got, cache, calls, _ = _run(lm, True, turns, 256, batch)
    want, cache_want, none, _ = _run(lm, False, turns, 256, batch)
    assert calls == 2 and none == 0 and torch.equal(got, want) and torch.equal(cache, cache_want)


@torch.no_grad()
def test_what_stays_layer_by_layer():
    lm = _lm()
    ids = _ids(1, 30)
    want = _run(lm, True, [ids], 64, 1)[0]
    heard = []
    for m in (lm.model.layers[1], lm.model.layers[0].self_attn.o_proj, lm.model.layers[2].qkv_proj.linear, lm.model.layers[2].mlp):
        handle = m.register_forward_hook(lambda mod, args, out: heard.append(mod))
        got, _, calls, _ = _run(lm, True, [ids], 64, 1)
        handle.remove()
        assert calls == 0 and heard.pop() is m and torch.equal(got, want)
    lm.model.layers[0].mlp.forward = lm.model.layers[0].mlp.forward
    assert _run(lm, True, [ids], 64, 1)[2] == 0
    del lm.model.layers[0].mlp.forward
    assert _run(lm, True, [ids], 64, 1)[2] == 1
    # another cache, a larger one: bound to it without a look at the layers
    stack = lm.model._prompt_layers
    for capacity, batch in ((64, 1), (512, 3)):
        got, cache, calls, _ = _run(lm, True, [_ids(batch, 30)], capacity, batch)
        other = _run(lm, False, [_ids(batch, 30)], capacity, batch)
        assert calls == 1 and lm.model._prompt_layers._watched is stack._watched and torch.equal(got, other[0]) and torch.equal(cache, other[1])
    # hidden states are asked for, no cache, gradients are on
    assert len(lm(input_ids=ids, output_hidden_states=True).hidden_states) == 4
    with torch.enable_grad():
        assert _run(lm, True, [ids], 64, 1)[2] == 0
    # weights replaced behind the stack's back: the parameter, its storage
    lm.model.layers[0].mlp.down_proj.weight.data = lm.model.layers[0].mlp.down_proj.weight.data * 1.5
    got, _, calls, _ = _run(lm, True, [ids], 64, 1)
    assert calls == 1 and torch.equal(got, _run(lm, False, [ids], 64, 1)[0]) and _off(got, want) > 0.02
    want = got
    layer = lm.model.layers[1].self_attn.o_proj
    layer.weight = torch.nn.Parameter(layer.weight * 2, requires_grad=False)
    layer.finalize_init()
    got, _, calls, _ = _run(lm, True, [ids], 64, 1)
    assert calls == 1 and torch.equal(got, _run(lm, False, [ids], 64, 1)[0]) and _off(got, want) > 0.02


@torch.no_grad()
def test_hook_on_the_models_positions():
    lm, ids, heard = _lm(), _ids(1, 30), []
    want = _run(lm, True, [ids], 64, 1)[0]
    handle = lm.model.rotary_emb.register_forward_hook(lambda mod, args, out: heard.append(out[0].shape))
    got, _, calls, _ = _run(lm, True, [ids], 64, 1)
    handle.remove()
    assert heard == [(1, 30, 128)] and calls == 0 and torch.equal(got, want)
    assert _run(lm, True, [ids], 64, 1)[2] == 1


@torch.no_grad()
def test_layers_that_differ():
    lm, other = _lm(), _lm(intermediate_size=640)
    lm.model.layers[1].mlp = other.model.layers[1].mlp
    got, cache, calls, _ = _run(lm, True, [_ids(1, 30)], 64, 1)
    want, cache_want, _, _ = _run(lm, False, [_ids(1, 30)], 64, 1)
    assert calls == 0 and torch.equal(got, want) and torch.equal(cache, cache_want)


@torch.no_grad()
def test_layers_rotate_with_their_own_tables():
    """... also where they were given others after a first prompt: all, one, the model's own module."""
    lm, other = _lm(), _lm(rope_theta=1e4)
    first = _run(lm, True, [_ids(1, 30), _ids(1, 1)], 64, 1)[0]
    for change in (lambda: [setattr(x.self_attn, "rotary_emb", y.self_attn.rotary_emb) for x, y in zip(lm.model.layers, other.model.layers)],
                   lambda: setattr(lm.model, "rotary_emb", other.model.rotary_emb),
                   lambda: setattr(lm.model.layers[1].self_attn, "rotary_emb", _lm().model.layers[1].self_attn.rotary_emb)):
        change()
        got = _run(lm, True, [_ids(1, 30), _ids(1, 1)], 64, 1)
        want = _run(lm, False, [_ids(1, 30), _ids(1, 1)], 64, 1)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]) and _off(got[0], first) > 0.01


@torch.no_grad()
def test_forward_mode_is_refused_as_by_the_modules():
    """The linears have no forward-mode rule: a tangent on the way in is an error, never lost."""
    lm = _lm()
    embeds = lm.model.embed_tokens(_ids(1, 30))
    for one_call in (True, False):
        lm.model.use_decoder_stack = one_call
        with torch.autograd.forward_ad.dual_level():
            dual = torch.autograd.forward_ad.make_dual(embeds, torch.ones_like(embeds))
            with pytest.raises(NotImplementedError):
                lm.model(inputs_embeds=dual, past_key_values=lm.create_cache(1, 64), use_cache=True, all_ones_mask=True)


@torch.no_grad()
def test_forward_mode_of_a_weight_is_refused_as_by_the_modules():
    """... of gate, up and down, which the MLP's node takes as arguments. A call without a tangent is an ordinary one."""
    lm, ids = _lm(), _ids(1, 30)
    want = lm(input_ids=ids).logits
    mlp = lm.model.layers[1].mlp
    for m in (mlp.gate_proj, mlp.up_proj, mlp.down_proj):
        plain = m.weight
        for one_call in (True, False):
            lm.model.use_decoder_stack = one_call
            with torch.autograd.forward_ad.dual_level():
                assert torch.equal(lm(input_ids=ids).logits, want)
                del m.weight
                m.weight = torch.autograd.forward_ad.make_dual(plain.detach(), torch.ones_like(plain))
                with pytest.raises(NotImplementedError):
                    lm(input_ids=ids)
                del m.weight
                m.weight = plain


@torch.no_grad()
def test_layers_are_examined_once_where_calls_are_refused():
    lm, built = _lm(), []
    handle = lm.model.layers[1].register_forward_hook(lambda *a: None)
    examine = MuiPromptStack.eligible
    MuiPromptStack.eligible = staticmethod(lambda *a: built.append(1) or examine(*a))
    try:
        assert [_run(lm, True, [_ids(1, 30)], 64, 1)[2] for _ in range(3)] == [0, 0, 0] and len(built) == 1
        handle.remove()
        assert _run(lm, True, [_ids(1, 30)], 64, 1)[2] == 1 and len(built) == 1
    finally:
        MuiPromptStack.eligible = staticmethod(examine)


@torch.no_grad()
def test_first_long_prompt_runs_on_the_modules(monkeypatch):
    """... and has the layers examined behind it: the second one goes by the single call, with the same bits."""
    from muillm_amd.modules.models.llama import model as llama

    rows, per_row = 150, 512 * (3 * 1280 + 2 * 512)
    for most, calls_first in ((rows * per_row, 1), (rows * per_row - 1, 0)):
        monkeypatch.setattr(llama, "_BUSY_PRODUCTS", most)
        lm, ids = _lm(), _ids(1, rows)
        first, second = _run(lm, True, [ids], 256, 1), _run(lm, True, [ids], 256, 1)
        assert first[2] == calls_first and second[2] == 1
        assert torch.equal(first[0], second[0]) and torch.equal(first[1], second[1])


@torch.no_grad()
@pytest.mark.parametrize("group,layer,field,value,status", [
    (128, 0, "int8_group_size_shift", 8, -2),  # o has a K of three groups and a half (all other products have whole ones)
    (128, 0, "int8_group_size_shift", 40, -2),
    (128, 0, "o_weight", None, -1), (0, 0, "o_weight", None, -1), (0, 0, "down_weight", None, -1),
    (0, 0, "o_pitch", 880, -1), (0, 0, "down_pitch", 1008, -1), (0, 0, "o_pitch", 904, -2)])
def test_int8_operands_are_refused_where_k_is_shared_too(group, layer, field, value, status):
    """As by mui_int8_linear and mui_int8_group_linear: nothing is read through a descriptor that those refuse."""
    lm = _lm(torch.float16, group, hidden_size=1024, intermediate_size=1024, num_attention_heads=8, num_key_value_heads=1)
    cache, lib, t = lm.create_cache(1, 128), _lib.load(), 80
    stack = MuiPromptStack(lm.model.layers, lm.model.rotary_emb, cache)
    stack.desc.n_q_heads = 7  # (the first 896 columns of o)
    x = torch.randn(1, t, 1024, device=DEV).half()
    pos, out = torch.arange(t, device=DEV), torch.empty_like(x)
    ws, scratch = torch.empty(lib.mui_decoder_stack_prompt_bytes(ctypes.byref(stack.desc), 1, t, 1), dtype=torch.uint8, device=DEV), muillm_ext.new_linear_workspace(DEV)

    def run():
        return lib.mui_decoder_stack_prompt(torch.cuda.current_stream().cuda_stream, ctypes.byref(stack.desc), 1, t, x.data_ptr(), out.data_ptr(), pos.data_ptr(), 0,
                                            pos.data_ptr(), t, None, 0, 1, ws.data_ptr(), scratch.data_ptr(), scratch.numel())

    try:
        _lib.check(lib.mui_tune_prompt_shares(7, 2), "mui_tune_prompt_shares")
        assert run() == 0 and bool(scratch[4096:].any())  # K is shared
        setattr(stack.desc.layers[layer], field, value)
        assert run() == status
    finally:
        _lib.check(lib.mui_tune_prompt_shares(0, 0), "mui_tune_prompt_shares")
