"""The scratch of linears beyond MUI_MAX_TOKENS rows in captured decode steps: a step of 17 to 32 rows shares K between workgroups like an eager
one, through scratch that is its decoder's own."""
import pytest
import torch

from muillm_amd import muillm_ext
from muillm_amd.engineconfig import MuiEngineConfig
from muillm_amd.modules.models.graphdecoder import MuiGraphDecoder
from muillm_amd.modules.models.llama.model import MuiDecoderConfig, MuiLlamaForCausalLM

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def lm():
    """Width 2048 with 8192 in between: the down projection divides K at 17 to 32 rows."""
    cfg = MuiDecoderConfig(hidden_size=2048, intermediate_size=8192, num_hidden_layers=2, num_attention_heads=16, num_key_value_heads=4,
                           vocab_size=4096, max_position_embeddings=512)
    return MuiLlamaForCausalLM.from_config(MuiEngineConfig(), cfg, dtype=torch.float16, device=DEV, seed=3, init_std=0.03)


def _prompt(lm, batch, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(0, lm.config.vocab_size, (batch, 9), generator=g).to(DEV)


@pytest.mark.parametrize("batch", [17, 20, 32])
def test_captured_step_equals_the_eager_one(lm, batch):
    """Bit for bit over replays of one and of several steps, with eager work in between; the step wrote partial sums into its
    decoder's scratch."""
    ids, new = _prompt(lm, batch, batch), 14
    eager, eager_logits = MuiGraphDecoder(lm, use_graph=False).generate(ids, new, return_logits=True)
    dec = MuiGraphDecoder(lm, use_graph=True)
    tokens, logits = dec.generate(ids, new, return_logits=True)
    assert torch.equal(tokens, eager) and torch.equal(logits, eager_logits)
    assert int(dec._linear_ws.count_nonzero()) > 0, "the captured step ran without scratch"
    _ = lm(input_ids=ids[:, :5])
    torch.cuda.synchronize()
    dec.cache.reset()
    assert torch.equal(dec.generate(ids, new, cache=dec.cache), eager)  # (several steps per replay)
    assert dec._linear_ws.data_ptr() not in [w.data_ptr() for w in muillm_ext._PROMPT_WORKSPACES.values()]


def test_decoders_on_two_streams(lm):
    """Replays that overlap on the device leave each other's sums alone."""
    new, alone, decs = 40, [], []
    for i in range(2):
        dec = MuiGraphDecoder(lm, use_graph=True)
        alone.append(dec.generate(_prompt(lm, 32, i), new))
        decs.append(dec)
    assert decs[0]._linear_ws.data_ptr() != decs[1]._linear_ws.data_ptr()
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    for i, (dec, s) in enumerate(zip(decs, streams)):
        with torch.cuda.stream(s):
            dec.cache.reset()
            dec.prefill(_prompt(lm, 32, i), new, cache=dec.cache)
    torch.cuda.synchronize()
    for _ in range(new - 1):
        for dec, s in zip(decs, streams):
            with torch.cuda.stream(s):
                dec.decode(1)
    torch.cuda.synchronize()
    for dec, want in zip(decs, alone):
        assert torch.equal(dec.out_tokens[:, :new], want[:, -new:])
