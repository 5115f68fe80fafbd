"""Prompts of a padded batch with the padding left out of what works on one token at a time, against the same prompts with it and
against every row alone."""
import pytest
import torch

from muillm_amd import _lib, muillm_ext
from muillm_amd.modules.models.graphdecoder import MuiGraphDecoder
from muillm_amd.modules import realrows
from muillm_amd.modules.decoder.decoderstack import MuiPromptStack
from muillm_amd.modules.models.llama import model as llama_model
from muillm_amd.modules.realrows import RealRows
from muillm_amd.modules.models.salepel.model import MuiSalepelForCausalLM
from tests import salepel_util, zufadra_util
from tests.test_prompt_stack_gpu import _lm

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(autouse=True)
def _however_little(monkeypatch):
    monkeypatch.setattr(realrows, "worth_it", lambda *a: True)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16, torch.int64])
@pytest.mark.parametrize("n,w", [(1, 8), (5, 16), (7, 24), (300, 4096), (3, 51), (4, 1)])
def test_rows_by_number(dtype, n, w):
    """Rows of whole 16-byte chunks by the kernel, others by torch; numbers outside give zeros."""
    g = torch.Generator().manual_seed(n)
    x = torch.randint(-50, 50, (n, w), generator=g).to(dtype)
    index = torch.randint(-2, n + 2, (2 * n + 3,), generator=g)
    want = torch.stack([x[i] if 0 <= i < n else torch.zeros(w, dtype=dtype) for i in index.tolist()])
    assert torch.equal(muillm_ext.take_rows(x.to(DEV), index.to(DEV)).cpu(), want)
    off = torch.zeros(n * w + 1, dtype=dtype, device=DEV)[1:].view(n, w).copy_(x)
    assert torch.equal(muillm_ext.take_rows(off, index.to(DEV)).cpu(), want)
    assert muillm_ext.take_rows(x.to(DEV), index[:0].to(DEV)).shape == (0, w)


def test_refused_arguments():
    lib, x = _lib.load(), torch.zeros(4, 8, device=DEV)
    at = torch.zeros(4, dtype=torch.int64, device=DEV)
    alignment = next(c for c in range(-1, -10, -1) if "align" in _lib.status_string(c))
    call = lambda bytes_, src=x.data_ptr(), rows=4, n=4: lib.mui_take_rows(0, src, n, bytes_, at.data_ptr(), x.data_ptr(), rows)
    assert call(24) == call(16, x.data_ptr() + 4) == alignment and call(0) == call(16, None) == call(16, rows=-1) == call(16, n=-1) == -1
    assert call(16, rows=0) == 0


def test_numbers_of_a_mask():
    mask = torch.tensor([[0, 0, 1, 1], [1, 1, 1, 1], [0, 0, 0, 1]], dtype=torch.bool)
    real = RealRows(mask, "cpu")
    assert real.n == 7 and real.rows.tolist() == [2, 3, 4, 5, 6, 7, 11] and real.last.tolist() == [1, 5, 6]
    assert real.slots.tolist() == [-1, -1, 0, 1, 2, 3, 4, 5, -1, -1, -1, 6]
    x = torch.arange(24.).view(3, 4, 2)
    assert torch.equal(real.spread(real.take(x)), x * mask[..., None]) and torch.equal(real.last_of(real.take(x)), x[:, -1:])


def _batch(lengths, vocab, seed=1):
    t = max(lengths)
    ids = torch.randint(0, vocab, (len(lengths), t), generator=torch.Generator().manual_seed(seed))
    mask = (torch.arange(t)[None] >= t - torch.tensor(lengths)[:, None]).to(torch.int64)
    return (ids * mask).to(DEV), mask.to(DEV)


def _prompt(lm, ids, mask, new, without=False):
    """(last position's logits, tokens, cache, calls that left the padding out)"""
    calls, plain = [], RealRows.last_of
    RealRows.last_of = lambda self, x: calls.append(x.shape) or plain(self, x)
    of = RealRows.of
    if without:
        RealRows.of = staticmethod(lambda *a: None)
    try:
        decoder = MuiGraphDecoder(lm, use_graph=False)
        cache = lm.create_cache(ids.shape[0], ids.shape[1] + new)
        logits = decoder.prefill(ids, new, cache, attention_mask=mask).float()
        decoder.decode(new - 1)
        return logits, decoder.out_tokens.clone(), cache, len(calls)
    finally:
        RealRows.last_of, RealRows.of = plain, of


def _off(a, b):
    return float((a - b).abs().max() / b.abs().max())


# one 16-bit rounding more or less per product, in a few layers: a few units in the last place of the largest logit
LIMIT = {torch.float32: 2e-5, torch.bfloat16: 3e-2, torch.float16: 4e-3}


@torch.no_grad()
@pytest.mark.parametrize("kind", ["bf16", "fp16", "int8", "int8_group"])
@pytest.mark.parametrize("lengths", [(2, 1), (5, 9, 3), (40, 13, 40, 1), (150, 50, 101), (7,) * 20 + (20,), (300, 299)])
def test_llama(kind, lengths):
    """Real rows that the decode kernels, the streaming ones and the tiles take, among them rows of a single token."""
    dtype = torch.bfloat16 if kind == "bf16" else torch.float16
    lm = _lm(dtype, {"int8": 0, "int8_group": 128}.get(kind))
    ids, mask = _batch(lengths, 512)
    got, tokens, cache, calls = _prompt(lm, ids, mask, 3)
    want, tokens_want, cache_want, none = _prompt(lm, ids, mask, 3, without=True)
    assert calls == 1 and none == 0 and cache.get_seq_length() == cache_want.get_seq_length() == max(lengths) + 2
    assert _off(got, want) <= LIMIT[dtype]
    t = max(lengths)
    for x, y in zip(cache.tensors(), cache_want.tensors()):
        for b, n in enumerate(lengths):
            assert not x[b, :, :t - n].any()  # padding's slots
            assert _off(x[b, :, t - n:t].float(), y[b, :, t - n:t].float()) <= LIMIT[dtype]
    for b, n in enumerate(lengths):
        alone = lm(input_ids=ids[b:b + 1, t - n:], num_logits_to_keep=1).logits[0, -1].float()
        assert _off(got[b], alone) <= LIMIT[dtype]


@torch.no_grad()
def test_layers_are_examined_once(monkeypatch):
    """For several padded prompts in a row, of more rows than the decode kernels take or fewer, and caches of their own; again once a weight has been replaced."""
    lm, built, examine = _lm(), [], MuiPromptStack.eligible
    monkeypatch.setattr(MuiPromptStack, "eligible", staticmethod(lambda *a: built.append(1) or examine(*a)))
    ids, mask = _batch((9, 4), 512)
    for _ in range(3):
        assert _prompt(lm, ids, mask, 1)[3] == 1 and len(built) == 1
    monkeypatch.setattr(llama_model, "_BUSY_PRODUCTS", 0)  # (a long prompt, as far as the model knows: only a first one is left to the modules)
    assert _prompt(lm, *_batch((30, 12, 7), 512), 1)[3] == 1 and len(built) == 1
    down = lm.model.layers[1].mlp.down_proj
    down.weight = torch.nn.Parameter(down.weight.detach().clone(), requires_grad=False)
    down.finalize_init()
    assert _prompt(lm, ids, mask, 1)[3] == 0 and len(built) == 2 and _prompt(lm, ids, mask, 1)[3] == 1 and len(built) == 2


@torch.no_grad()
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("util,name", [(salepel_util, "default"), (zufadra_util, "default")])
@pytest.mark.parametrize("lengths", [(5, 9, 3), (40, 13, 40, 1), (150, 50, 101)])
def test_native(dtype, util, name, lengths):
    cfg = util.default_config()
    w = util.random_weights(cfg, seed=4, **({"close_calls": dtype == torch.float32} if util is salepel_util else {}))
    lm = salepel_util.build(cfg, w, dtype) if util is salepel_util else _zufadra(cfg, w, dtype)
    ids, mask = _batch(lengths, cfg["vocab"])
    t, outs = max(lengths), []
    for real in (RealRows.of(lm, mask.cpu() != 0, DEV), None):
        cache = lm.create_cache(len(lengths), t + 2)
        logits = [lm(input_ids=ids, attention_mask=mask, past_key_values=cache, num_logits_to_keep=1, real=real).logits[:, -1]]
        for _ in range(2):
            logits.append(lm(input_ids=logits[0].argmax(-1)[:, None], past_key_values=cache).logits[:, -1])
        assert cache.real is None and cache.get_seq_length() == t + 2
        # (of the convolutions' last inputs those in front of a row's first token are left as they came; they count as zeros)
        outs.append((torch.stack(logits), [x.double() for x in cache.step_state() if util is salepel_util or x.dim() == 4]))
    for a, b in zip(*outs):
        for x, y in zip(a, b):
            assert _off(x, y) <= LIMIT[dtype]
    for b, n in enumerate(lengths):
        alone = lm(input_ids=ids[b:b + 1, t - n:], num_logits_to_keep=1).logits[0, -1].float()
        assert _off(outs[0][0][0, b], alone) <= LIMIT[dtype]
    if dtype == torch.bfloat16:  # as the decode loop calls it
        logits, _, _, calls = _prompt(lm, ids, mask, 3)
        assert calls == 1 and _off(logits, outs[0][0][0]) <= LIMIT[dtype]


def _zufadra(cfg, w, dtype):
    return zufadra_util.build(cfg, w, dtype)


@torch.no_grad()
@pytest.mark.parametrize("util", [salepel_util, zufadra_util])
def test_a_mask_of_another_shape_stays_refused(util):
    """One row of a mask for two of tokens: the layers refuse it, and the real rows of its one row are not taken for the batch."""
    cfg = util.default_config()
    lm = util.build(cfg, util.random_weights(cfg, seed=4), torch.bfloat16)
    ids = torch.randint(0, cfg["vocab"], (2, 9), device=DEV)
    mask = torch.ones(1, 9, dtype=torch.int64, device=DEV)
    mask[0, :4] = 0
    for real in (None, RealRows.of(lm, mask.cpu() != 0, DEV)):
        with pytest.raises(RuntimeError, match="row_start"):
            lm(input_ids=ids, attention_mask=mask, past_key_values=lm.create_cache(2, 12), num_logits_to_keep=1, real=real)


@torch.no_grad()
def test_what_is_run_with_the_padding():
    lm = _lm()
    ids, mask = _batch((9, 4), 512)
    assert _prompt(lm, ids, mask, 2)[3] == 1
    assert _prompt(lm, ids, torch.ones_like(mask), 2)[3] == 0
    heard = []
    for m in (lm, lm.model, lm.model.embed_tokens, lm.model.norm, lm.model.layers[1].mlp):
        hook = m.register_forward_hook(lambda m, a, out: heard.append(type(m)))
        assert _prompt(lm, ids, mask, 2)[3] == 0
        hook.remove()
    assert len(set(heard)) == 5
    with pytest.raises(ValueError):
        _prompt(lm, ids, mask.flip(1), 2)
    # whoever asks for every position gets every position
    out = lm(input_ids=ids, attention_mask=mask)
    assert out.logits.shape[:2] == ids.shape


def test_a_class_of_its_own_is_not_asked():
    lm = _lm()
    mask = torch.tensor([[0, 1], [1, 1]], dtype=torch.bool)
    assert RealRows.of(lm, mask, DEV) is not None
    lm.__class__ = type("Derived", (type(lm),), {})  # may have a forward of its own
    assert RealRows.of(lm, mask, DEV) is None


@pytest.mark.parametrize("tokens,padding,hidden,worth", [
    (128, 100, 4096, False), (192, 64, 4096, True), (192, 63, 4096, False), (319, 120, 2048, True), (319, 100, 2048, True), (319, 99, 2048, False), (256, 100, 4096, False), (300, 44, 4096, True),
    (300, 43, 4096, False), (192, 66, 2048, False), (4000, 300, 2048, True)])
def test_where_it_is_worth_it(monkeypatch, tokens, padding, hidden, worth):
    """Llama: padding of 1e10 operations a layer, with which a tile of 256 tokens falls away or the rest are no more than 128."""
    monkeypatch.undo()
    lm = _lm()
    lm.config.hidden_size = hidden
    mask = torch.ones(1, tokens, dtype=torch.bool)
    mask[0, :padding] = False
    assert (RealRows.of(lm, mask, DEV) is not None) == worth
    # mixtures of experts: whatever tiles there are, but not a few of many tokens
    least = 8e9 / (24 * hidden ** 2) + tokens * 3800 / (24 * hidden)
    assert realrows.worth_it(MuiSalepelForCausalLM.padding_worth, hidden, tokens, padding) == (tokens > 128 and padding >= least)
