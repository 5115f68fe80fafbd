"""The work a user of this framework has it do, as cases to be timed: requests served by the decode loop.

A pass is one request (or one batch of them) through MuiGraphDecoder, which generate() and generate_greedy() are thin
wrappers of: the prompt into an emptied cache, then `new` - 1 further tokens, in whatever launch mode the loop chooses.
It returns the logits behind the prompt, the tokens, the last step's logits and the cache.

Models are the three kinds the framework has, at the widths of its benchmark: the Llama-shaped decoder (16-bit, int8 per
channel, int8 in groups of 128), the Salepel decoder (latent attention, matrix memory, mixture of experts) and the Zufadra decoder (channel-wise
delta rule, windowed attention with sinks). Weights are random with the fan-in scale of trained ones. Two things are as in a trained
model and not as in plain noise, because results could not be compared otherwise: the head knows the next token (its rows are the
embedding's, shifted), so greedy tokens do not hang on rounding; and a token's experts are written in its embedding, so
neither does the choice of experts. A token's experts are drawn uniformly, so the load is a balanced one."""
import zlib

import torch

DEVICE = "cuda"
EPS = 1e-5
VOCAB = {"llama": 128256, "salepel": 32768, "zufadra": 32768}
SIZES = {
    ("llama", 4096): dict(heads=32, kv_heads=8, ff=14336),
    ("llama", 2048): dict(heads=16, kv_heads=4, ff=8192),
    ("salepel", 4096): dict(heads=32, q_rank=1536, window=4096, mem_heads=8, experts=64, identity=8, top=8, ff=1792),
    ("salepel", 2048): dict(heads=16, q_rank=768, window=1024, mem_heads=4, experts=64, identity=8, top=6, ff=1408),
    ("zufadra", 4096): dict(heads=32, kv_heads=8, window=4096, keep=64, ff=14336),
    ("zufadra", 2048): dict(heads=16, kv_heads=4, window=1024, keep=64, ff=8192),
}
HEAD = 128                               # query, key and value size of a head (and both sizes of the delta rule's memory)
ROT, KV_RANK, CAP = 64, 512, 15.0        # Salepel: rotated part, latent rank, gate cap; memory 256 x 512 a head
MEM_K, MEM_V = 256, 512
RANK, TAPS, SOFTCAP = 128, 4, 30.0       # Zufadra: ranks of the low-rank maps, convolution taps, score cap
BIGRAM = dict(buckets=32003, mul_prev=1009, mul_cur=31)
SALEPEL = ("latent", 0, "latent", "mem", "latent", 4, "latent", "mem")  # a number: over that layer's latent rows
SHIFT = 7919                             # the token after t is t + SHIFT
MARK = 8.0                               # what marks a token's experts in its embedding
BRANCH = 0.3                             # gain of a sublayer's contribution to the residual stream


# --------------------------------------------------------------------------------------
# cases
# --------------------------------------------------------------------------------------
def _case(name, model, width, batch, prompt, new, dtype="bf16", weights="16", layers=8, padded=False):
    c = dict(model=model, width=width, layers=layers, dtype=dtype, weights=weights, batch=batch, prompt=prompt, new=new, padded=padded)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the headline: one user's chat turn on the whole 8B-shaped model, a short prompt and its answer
        _case("llama_chat", "llama", 4096, 1, 32, 16, dtype="fp16", layers=32),
        # a server's batch: prompts of different lengths, padded on the left, answered together
        _case("llama_batch", "llama", 4096, 32, 24, 12, dtype="fp16", padded=True),
        # time to first token of an ordinary question, and of a long document
        _case("llama_prompt_short", "llama", 4096, 1, 101, 1),
        _case("llama_prompt_long", "llama", 4096, 1, 3500, 1, dtype="fp16"),
        # int8 weights, a few users
        _case("llama_int8", "llama", 4096, 4, 200, 12, dtype="fp16", weights="int8"),
        # the smallest: a small model answers a few words with a few words; launches and latency
        _case("llama_small", "llama", 2048, 1, 17, 8),
        # Salepel: one user, a batch of ragged prompts on the small model, a long prompt
        _case("salepel_chat", "salepel", 4096, 1, 50, 12),
        _case("salepel_batch", "salepel", 2048, 8, 150, 8, padded=True),
        _case("salepel_prompt", "salepel", 4096, 1, 2000, 1),
        # Zufadra: one user, a batch on the small model, a long prompt
        _case("zufadra_chat", "zufadra", 4096, 1, 333, 12),
        _case("zufadra_batch", "zufadra", 2048, 20, 64, 8),
        _case("zufadra_prompt", "zufadra", 4096, 1, 4000, 1),
    ]


def _cost(case):
    w = work(case)
    return w["bytes"] / 6e12 + w["flops"] / 1e15


def draw(rng):
    """Any model, width, type and option; batches of 1 to 32, prompts of 5 to 4096 tokens and up to 8192 in a batch, prompts alone
    or with 2 to 24 new tokens."""
    most = _cost(listed()[0])
    while True:
        model = rng.choice(("llama", "llama", "salepel", "zufadra"))
        batch = min(32, int(2 ** rng.uniform(0.0, 5.1)))
        prompt = min(4096, int(5 * 2 ** rng.uniform(0.0, 9.7)))
        if batch * prompt > 8192:
            continue
        case = _case(None, model, rng.choice((2048, 4096)), batch, prompt, 1 if rng.random() < 0.4 else rng.randint(2, 24),
                     dtype=rng.choice(("bf16", "fp16")) if model == "llama" else "bf16",
                     weights=rng.choice(("16", "16", "int8", "int8_group")) if model == "llama" else "16",
                     padded=batch > 1 and rng.random() < 0.5)
        if _cost(case) <= 0.9 * most:
            return case


def work(case):
    """One forward pass per prompt and per further token; each reads the weights it touches (of a mixture: the experts that
    its tokens are expected to choose) and the keys, values or memories that its tokens see once."""
    z, n, b = SIZES[case["model"], case["width"]], case["width"], case["batch"]
    vocab, layers = VOCAB[case["model"]], case["layers"]
    unit = {"16": 2.0, "int8": 1.0, "int8_group": 1.0 + 4.0 / 128}[case["weights"]]
    nbytes = flops = 0.0
    for step in range(case["new"]):
        t = case["prompt"] if step == 0 else 1
        tokens, ctx = b * t, case["prompt"] + step
        seen = ctx * (0.5 if step == 0 else 1.0)  # keys a token sees on average
        for i in range(layers):
            if case["model"] == "llama":
                dense, moe = n * HEAD * (2 * z["heads"] + 2 * z["kv_heads"]) + 3 * n * z["ff"], 0
                state, per = 4.0 * b * ctx * HEAD * z["kv_heads"], 4.0 * HEAD * z["heads"] * seen
            elif case["model"] == "zufadra":
                if i % 2:
                    dense = n * HEAD * (3 * z["heads"] + 2 * z["kv_heads"])
                    state, per = 4.0 * b * min(ctx, z["window"]) * HEAD * z["kv_heads"], 4.0 * HEAD * z["heads"] * min(seen, z["window"])
                else:
                    dense = 4 * n * n + n * (2 * RANK + z["heads"]) + 2 * n * RANK
                    state, per = 8.0 * b * z["heads"] * HEAD * HEAD, 8.0 * z["heads"] * HEAD * HEAD
                dense, moe = dense + 3 * n * z["ff"], 0
            else:
                if SALEPEL[i] == "mem":
                    dense = n * z["mem_heads"] * (2 * MEM_K + 3 * MEM_V)
                    state, per = 8.0 * b * z["mem_heads"] * MEM_K * MEM_V, 6.0 * z["mem_heads"] * MEM_K * MEM_V
                else:
                    own = SALEPEL[i] == "latent"
                    dense = z["q_rank"] * (n + z["heads"] * (HEAD + ROT)) + (KV_RANK + ROT) * n * own + 2 * KV_RANK * z["heads"] * HEAD + n * n
                    state, per = 2.0 * b * min(ctx, z["window"]) * (KV_RANK + ROT), 2.0 * z["heads"] * (2 * HEAD + ROT) * min(seen, z["window"])
                moe = 3 * n * z["ff"]
                outputs = z["experts"] + z["identity"]
                nbytes += 2.0 * moe * z["experts"] * (1.0 - (1.0 - z["top"] / outputs) ** tokens)
                flops += 2.0 * moe * tokens * z["top"] * z["experts"] / outputs
            nbytes += unit * dense + state + 4.0 * n * tokens
            flops += (2.0 * dense + per) * tokens
        nbytes += 2.0 * n * vocab + 2.0 * b * vocab
        flops += 2.0 * n * vocab * b
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # four times what lies between run() and exact(): logits and caches of 16-bit models are 0.008 (bf16) and 0.002 (fp16) off in the
    # 2-norm, single values of a memory up to 0.11 and of an fp16 cache 0.01 of the rest's root mean square
    return {"rel": 0.03, "max": 0.45} if case["dtype"] == "bf16" else {"rel": 0.008, "max": 0.04}


# --------------------------------------------------------------------------------------
# weights and inputs
# --------------------------------------------------------------------------------------
def _dtype(case):
    return {"fp16": torch.float16, "bf16": torch.bfloat16}[case["dtype"]]


def _normal(case, seed, name, shape, std=1.0, mean=0.0):
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed((zlib.crc32(name.encode()) << 20) ^ int(seed))
    return torch.empty(shape, dtype=_dtype(case), device=DEVICE).normal_(mean, std, generator=gen)


def _embedding(case, seed):
    z, vocab, n = SIZES[case["model"], case["width"]], VOCAB[case["model"]], case["width"]
    table = _normal(case, seed, "embed", (vocab, n))
    if case["model"] == "salepel":
        gen = torch.Generator(device=DEVICE)
        gen.manual_seed(int(seed))
        outputs = z["experts"] + z["identity"]
        for i in range(case["layers"]):
            marks = table[:, i * outputs:(i + 1) * outputs]
            marks.mul_(0.1)
            chosen = torch.rand(vocab, outputs, device=DEVICE, generator=gen).topk(z["top"], dim=-1).indices
            marks.scatter_(1, chosen, MARK)
    return table


def _weight(case, seed, name, shape):
    """The tensor called `name` in a checkpoint (Llama: in the lists of _llama_places)."""
    z, n = SIZES[case["model"], case["width"]], case["width"]
    last = name.split(".")[-1]
    if name == "embed":
        return _embedding(case, seed)
    if name == "head":
        return _embedding(case, seed).roll(SHIFT, 0).mul_(n ** -0.5)
    if name == "bigram":
        return _normal(case, seed, name, shape, 0.5)
    if last in ("norm1b", "norm2b") or (case["model"] == "zufadra" and last in ("norm1", "norm2")):
        return _normal(case, seed, name, shape, 0.1 * BRANCH, BRANCH)
    if last == "norm" or last in ("norm1", "norm2"):
        return _normal(case, seed, name, shape, 0.1, 1.0)
    if last == "router":  # reads the marks of its layer
        w = _normal(case, seed, name, shape, 0.02 * n ** -0.5)
        i = int(name[1:].split(".")[0])
        w[:, i * shape[0]:(i + 1) * shape[0]].fill_diagonal_(0.7)
        return w
    if last == "correction":
        return _normal(case, seed, name, shape, 0.002)
    if last == "b" and ".mlp." in name:
        return _normal(case, seed, name, shape, 0.1)
    if name.endswith(".i.b"):
        return _normal(case, seed, name, shape, 0.2)
    if name.endswith(".f.b"):
        return _normal(case, seed, name, shape, 1.0, 3.0)
    if last == "dt_bias":
        return _normal(case, seed, name, shape, 1.0, -4.0)
    if last == "A_log":
        return _normal(case, seed, name, shape, 0.5, 1.0)
    if last == "conv":
        return _normal(case, seed, name, shape, 0.5)
    branch = BRANCH if case["model"] == "llama" and last in ("o", "down") else 1.0
    return _normal(case, seed, name, shape, branch * shape[-1] ** -0.5)


def _prompts(case, seed):
    """(ids [B, prompt], 0 / 1 mask or None): padded batches hold prompts from a third of the longest on."""
    gen = torch.Generator().manual_seed(int(seed))
    b, t = case["batch"], case["prompt"]
    ids = torch.randint(0, VOCAB[case["model"]], (b, t), generator=gen)
    if not case["padded"]:
        return ids, None
    lengths = torch.randint(max(1, t // 3), t + 1, (b,), generator=gen)
    lengths[0], lengths[-1] = t, max(1, t // 3)
    mask = (torch.arange(t)[None, :] >= t - lengths[:, None]).to(torch.int64)
    return ids * mask, mask


def _llama_places(lm):
    m = lm.model
    yield "embed", m.embed_tokens.weight
    for i, layer in enumerate(m.layers):
        p = "l%d." % i
        yield p + "norm1", layer.qkv_proj.linear.norm_weights
        yield p + "qkv", layer.qkv_proj.linear.weight
        yield p + "o", layer.self_attn.o_proj.weight
        yield p + "norm2", layer.mlp.norm_weights
        for part in ("gate", "up", "down"):
            yield p + part, getattr(layer.mlp, part + "_proj").weight
    yield "final.norm", m.norm.weight
    yield "head", lm.lm_head.weight


def _llama(case, seed):
    from muillm_amd.engine import init_engine
    from muillm_amd.engineconfig import MuiEngineConfig
    from muillm_amd.modules.models.llama.model import MuiDecoderConfig, MuiLlamaForCausalLM
    from muillm_amd.quantization.quantizationmethod import Int8WeightOnlyQuantizationMethod

    z = SIZES[case["model"], case["width"]]
    config = MuiDecoderConfig(hidden_size=case["width"], intermediate_size=z["ff"], num_hidden_layers=case["layers"],
                              num_attention_heads=z["heads"], num_key_value_heads=z["kv_heads"], vocab_size=VOCAB["llama"])
    lm = MuiLlamaForCausalLM.from_config(MuiEngineConfig(), config, dtype=_dtype(case), device=DEVICE, finalize=False)
    with torch.no_grad():
        for name, p in _llama_places(lm):
            p.copy_(_weight(case, seed, name, tuple(p.shape)))
    method = None
    if case["weights"] != "16":
        method = Int8WeightOnlyQuantizationMethod(group_size=0 if case["weights"] == "int8" else 128, modules=["qkv_proj", "o_proj", "mlp"])
    return init_engine(lm, device=DEVICE, engine_config=MuiEngineConfig(method))


def _salepel_config(case):
    z = SIZES[case["model"], case["width"]]
    mem = {"type": "mlstm", "mixer": {"heads": z["mem_heads"], "dim": MEM_K, "vdim": MEM_V, "gate_cap": CAP}}
    ff = {"kind": "moe", "expert": {"ff": z["ff"], "limit": 7.0}, "router": {"experts": z["experts"], "identity": z["identity"], "top": z["top"]}}
    layers = []
    for kind in SALEPEL:
        layer = mem
        if kind != "mem":
            layer = {"type": "latent_attention", "mixer": {
                "heads": z["heads"], "dim": HEAD, "rot_dim": ROT, "vdim": HEAD, "q_rank": z["q_rank"], "kv_rank": KV_RANK,
                "mask": {"size": z["window"]}, "rot": {"base": 10000.0, "dims": ROT}, "scale": (HEAD + ROT) ** -0.5}}
            if kind != "latent":
                layer["mixer"]["kv_from"] = kind
        layers.append(dict(layer, mlp=ff))
    return {"architecture": "Salepel", "embedding": {"scale": 1.0}, "norm": {"eps": EPS}, "vocab": VOCAB["salepel"], "width": case["width"],
            "layers": layers}


def _zufadra_config(case):
    z = SIZES[case["model"], case["width"]]
    mem = {"type": "channel_delta", "mixer": {"conv": TAPS, "dim": HEAD, "vdim": HEAD, "heads": z["heads"], "kv_heads": z["heads"]}}
    att = {"type": "attention", "mixer": {"heads": z["heads"], "kv_heads": z["kv_heads"], "dim": HEAD, "vdim": HEAD, "scale": HEAD ** -0.5,
                                          "rot": {"base": 10000.0, "dims": ROT}, "softcap": SOFTCAP,
                                          "mask": {"size": z["window"], "keep_first": z["keep"]}}}
    layers = [dict(att if i % 2 else mem, mlp={"kind": "dense", "ff": z["ff"]}) for i in range(case["layers"])]
    return {"architecture": "Zufadra", "embedding": {"scale": 1.0, "bigram": dict(BIGRAM)}, "norm": {"eps": EPS}, "vocab": VOCAB["zufadra"],
            "width": case["width"], "residual_mult": 1.0, "logit_scale": 1.0, "layers": layers}


def _native(case, seed):
    from muillm_amd.modules.models.salepel.config import MuiSalepelConfig
    from muillm_amd.modules.models.salepel.model import MuiSalepelForCausalLM
    from muillm_amd.modules.models.zufadra.config import MuiZufadraConfig
    from muillm_amd.modules.models.zufadra.model import MuiZufadraForCausalLM

    if case["model"] == "salepel":
        cls, config = MuiSalepelForCausalLM, MuiSalepelConfig.from_dict(_salepel_config(case))
    else:
        cls, config = MuiZufadraForCausalLM, MuiZufadraConfig.from_dict(_zufadra_config(case))
    lm = cls.from_config(None, config, dtype=_dtype(case), device=DEVICE)
    shapes = {name: tuple(t.shape) for name, t in lm.checkpoint_tensors()}
    lm.load_tensors(list(shapes), lambda name: _weight(case, seed, name, shapes[name]))
    return lm


def prepare(case, seed):
    from muillm_amd.modules.models.graphdecoder import MuiGraphDecoder

    lm = (_llama if case["model"] == "llama" else _native)(case, seed)
    ids, mask = _prompts(case, seed)
    return {"lm": lm, "decoder": MuiGraphDecoder(lm, use_graph=None),
            "cache": lm.create_cache(case["batch"], case["prompt"] + case["new"]), "new": case["new"],
            "ids": ids.to(DEVICE), "mask": None if mask is None else mask.to(DEVICE)}


def run(state):
    decoder, cache, new = state["decoder"], state["cache"], state["new"]
    cache.reset()
    out = {"first_logits": decoder.prefill(state["ids"], new, cache, attention_mask=state["mask"])}
    if new > 1:
        decoder.decode(new - 1)
        out["last_logits"] = decoder.logits
    out["tokens"] = decoder.out_tokens
    if state["mask"] is None:  # (slots in front of a padded row hold nothing that anyone reads)
        out["cache"] = cache.tensors()[:56]
    return out


# --------------------------------------------------------------------------------------
# the same in 64 bits
# --------------------------------------------------------------------------------------
HI = torch.float64


def _rms(x, gain=1.0):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * gain


def _rotate(x, pos, freq, pairs):
    """Rotary positions on the first 2 len(freq) of x [T, heads, d]; pairs (2 i, 2 i + 1) or (i, i + len(freq))."""
    n = len(freq)
    a, b = (slice(0, 2 * n, 2), slice(1, 2 * n, 2)) if pairs else (slice(0, n), slice(n, 2 * n))
    angle = pos.to(HI)[:, None, None] * freq
    y = x.clone()
    y[..., a] = x[..., a] * angle.cos() - x[..., b] * angle.sin()
    y[..., b] = x[..., b] * angle.cos() + x[..., a] * angle.sin()
    return y


def _freq(base, dims):
    return float(base) ** (-torch.arange(0, dims, 2, dtype=HI, device=DEVICE) / dims)


def _attend(q, k, v, scale, window=0, keep=0, cap=0.0):
    """Causal attention of one sequence: q [T, H, d], k [T, G, d], v [T, G, dv]."""
    t, heads, share = q.shape[0], q.shape[1], q.shape[1] // k.shape[1]
    at = torch.arange(t, device=DEVICE)
    seen = at[:, None] >= at
    if window:
        seen &= (at[:, None] - at < window) | (at < keep)
    out = torch.empty(t, heads, v.shape[2], dtype=HI, device=DEVICE)
    for h in range(heads):
        score = (q[:, h] @ k[:, h // share].T) * scale
        if cap:
            score = cap * torch.tanh(score / cap)
        out[:, h] = torch.softmax(score.masked_fill_(~seen, -float("inf")), -1) @ v[:, h // share]
    return out.reshape(t, -1)


class _Exact:
    """One case in 64 bits: all tokens of all rows side by side, row after row, a row's sequence in self.rows[b]."""

    def __init__(self, case, seed):
        self.case, self.seed, self.z = case, seed, SIZES[case["model"], case["width"]]
        ids, mask = _prompts(case, seed)
        vocab, tokens, self.rows = VOCAB[case["model"]], [], []
        for b in range(case["batch"]):
            row = ids[b] if mask is None else ids[b, mask[b] == 1]
            more = [int(row[-1] + SHIFT * (i + 1)) % vocab for i in range(case["new"] - 1)]
            at = sum(len(r) for r in tokens)
            tokens.append(torch.cat([row, torch.tensor(more, dtype=torch.int64)]))
            self.rows.append(slice(at, at + len(tokens[-1])))
        self.tokens = torch.cat(tokens).to(DEVICE)
        self.pos = torch.cat([torch.arange(len(r)) for r in tokens]).to(DEVICE)
        self.state = []
        slots = 1
        while slots < case["prompt"] + case["new"]:
            slots *= 2
        self.slots = slots

    def w(self, name, *shape):
        return _weight(self.case, self.seed, name, shape).to(HI)

    def linear(self, x, name, n):
        return x @ self.w(name, n, x.shape[1]).T

    def per_row(self, f, *xs):
        return torch.cat([f(*(x[r] for x in xs)) for r in self.rows])

    def kept(self, x):
        """Rows [T, ...] of every sequence in a cache's slots."""
        y = torch.zeros((len(self.rows), self.slots) + x.shape[1:], dtype=HI, device=DEVICE)
        for b, r in enumerate(self.rows):
            y[b, :r.stop - r.start] = x[r]
        return y

    def quantised(self, name, *shape):
        """A matrix as its int8 codes stand for it."""
        w = _weight(self.case, self.seed, name, shape)
        f = w.float()
        if self.case["weights"] == "int8":
            s = (f.abs().amax(1, keepdim=True) / 127.0).to(w.dtype)
            return (f / s.float()).round().clamp(-127, 127).to(HI) * s.to(HI)
        if self.case["weights"] == "int8_group":
            f = f.reshape(-1, 128)
            lo, hi = f.amin(1, keepdim=True), f.amax(1, keepdim=True)
            span = (hi - lo).clamp(min=1e-6)
            lo = (lo + hi) * 0.5 - span * 0.5
            codes = ((f - lo) / (span / 255)).clamp(0, 255).round()
            return (codes.to(HI) * (span / 255).to(w.dtype).to(HI) + lo.to(w.dtype).to(HI)).reshape(shape)
        return w.to(HI)

    def llama(self):
        z, n = self.z, self.case["width"]
        hq, hkv, t = z["heads"], z["kv_heads"], len(self.tokens)
        x, freq, keys, values = self.w("embed")[self.tokens], _freq(500000.0, HEAD), [], []
        for i in range(self.case["layers"]):
            p = "l%d." % i
            qkv = _rms(x, self.w(p + "norm1", n)) @ self.quantised(p + "qkv", (hq + 2 * hkv) * HEAD, n).T
            q, k, v = (y.reshape(t, -1, HEAD) for y in qkv.split([hq * HEAD, hkv * HEAD, hkv * HEAD], 1))
            q, k = (_rotate(y, self.pos, freq, False) for y in (q, k))
            keys.append(self.kept(k).transpose(1, 2))
            values.append(self.kept(v).transpose(1, 2))
            o = self.per_row(lambda q, k, v: _attend(q, k, v, HEAD ** -0.5), q, k, v)
            x = x + o @ self.quantised(p + "o", n, hq * HEAD).T
            h = _rms(x, self.w(p + "norm2", n))
            g = h @ self.quantised(p + "gate", z["ff"], n).T
            h = g * torch.sigmoid(g) * (h @ self.quantised(p + "up", z["ff"], n).T)
            x = x + h @ self.quantised(p + "down", n, z["ff"]).T
        self.state = keys + values
        return _rms(x, self.w("final.norm", n))

    def latent(self, h, i, rows):
        z, t = self.z, h.shape[0]
        heads, p, freq = z["heads"], "l%d.mix." % i, _freq(10000.0, ROT)
        q = _rms(self.linear(h, p + "dq", z["q_rank"]), self.w(p + "dq.norm", z["q_rank"]))
        q = self.linear(q, p + "uq", heads * (HEAD + ROT)).reshape(t, heads, HEAD + ROT)
        q = torch.cat([q[..., :HEAD], _rotate(q[..., HEAD:], self.pos, freq, False)], -1)
        if SALEPEL[i] == "latent":
            y = self.linear(h, p + "dkv", KV_RANK + ROT)
            rows[i] = (_rms(y[:, :KV_RANK], self.w(p + "dkv.norm", KV_RANK)), _rotate(y[:, None, KV_RANK:], self.pos, freq, False))
            self.state += [self.kept(rows[i][0]), self.kept(rows[i][1][:, 0])]
        c, r = rows[i if SALEPEL[i] == "latent" else SALEPEL[i]]
        k = torch.cat([self.linear(c, p + "uk", heads * HEAD).reshape(t, heads, HEAD), r.expand(t, heads, ROT)], -1)
        v = self.linear(c, p + "uv", heads * HEAD).reshape(t, heads, HEAD)
        return self.per_row(lambda q, k, v: _attend(q, k, v, (HEAD + ROT) ** -0.5, z["window"]), q, k, v)

    def memory(self, h, i):
        heads, p, t = self.z["mem_heads"], "l%d.mix." % i, h.shape[0]
        q = self.linear(h, p + "q", heads * MEM_K).reshape(t, heads, MEM_K) * MEM_K ** -0.5
        k = self.linear(h, p + "k", heads * MEM_K).reshape(t, heads, MEM_K)
        v = self.linear(h, p + "v", heads * MEM_V).reshape(t, heads, MEM_V)
        gi, gf = (CAP * torch.tanh((self.linear(h, p + g, heads) + self.w(p + g + ".b", heads)) / CAP) for g in "if")
        gf = torch.nn.functional.logsigmoid(gf)
        o, states = torch.empty_like(v), []
        for r in self.rows:
            s = torch.zeros(heads, MEM_K, MEM_V, dtype=HI, device=DEVICE)
            n, m = torch.zeros(heads, MEM_K, dtype=HI, device=DEVICE), torch.zeros(heads, dtype=HI, device=DEVICE)
            for j in range(r.start, r.stop):
                top = torch.maximum(gf[j] + m, gi[j])
                keep, add = torch.exp(gf[j] + m - top), torch.exp(gi[j] - top)
                s = torch.baddbmm(keep[:, None, None] * s, (add[:, None] * k[j])[:, :, None], v[j][:, None, :])
                n, m = keep[:, None] * n + add[:, None] * k[j], top
                den = torch.maximum((n * q[j]).sum(-1).abs(), torch.exp(-m)) + 1e-6
                o[j] = (q[j][:, None, :] @ s)[:, 0] / den[:, None]
            states.append((s, n, m))
        self.state += [torch.stack([s for s, _, _ in states]), None, None]  # (n and m: copies by the framework's own slices)
        return _rms(o).reshape(t, -1) * self.w(p + "norm", heads * MEM_V) * torch.sigmoid(self.linear(h, p + "g", heads * MEM_V))

    def experts(self, h, i):
        z, p, n = self.z, "l%d.mlp." % i, self.case["width"]
        outputs = z["experts"] + z["identity"]
        score = torch.softmax(self.linear(h, p + "router", outputs), -1)
        chosen = (score + self.w(p + "correction", outputs)).topk(z["top"], -1).indices
        share = torch.zeros_like(score).scatter_(1, chosen, score.gather(1, chosen))
        y = share[:, z["experts"]:].sum(1, keepdim=True) * h
        for e in range(z["experts"]):
            at = (chosen == e).any(1).nonzero().flatten()
            if not len(at):
                continue
            g = self.linear(h[at], "%se%d.gate" % (p, e), z["ff"]).clamp(max=7.0)
            u = self.linear(h[at], "%se%d.up" % (p, e), z["ff"]).clamp(-7.0, 7.0)
            y[at] += share[at, e, None] * self.linear(g * torch.sigmoid(1.702 * g) * (u + 1), "%se%d.down" % (p, e), n)
        return y

    def salepel(self):
        n, rows = self.case["width"], {}
        x = self.w("embed")[self.tokens]
        for i in range(self.case["layers"]):
            p = "l%d." % i
            h = _rms(x, self.w(p + "norm1", n))
            y = self.memory(h, i) if SALEPEL[i] == "mem" else self.latent(h, i, rows)
            x = x + _rms(self.linear(y, p + "mix.o", n), self.w(p + "norm1b", n))
            x = x + _rms(self.experts(_rms(x, self.w(p + "norm2", n)), i), self.w(p + "norm2b", n))
        return _rms(x, self.w("final.norm", n))

    def windowed(self, h, i):
        z, p, t = self.z, "l%d.mix." % i, h.shape[0]
        hq, hkv, freq = z["heads"], z["kv_heads"], _freq(10000.0, ROT)
        q = _rms(self.linear(h, p + "q", hq * HEAD), self.w(p + "q.norm", hq * HEAD)).reshape(t, hq, HEAD)
        k = _rms(self.linear(h, p + "k", hkv * HEAD), self.w(p + "k.norm", hkv * HEAD)).reshape(t, hkv, HEAD)
        v = self.linear(h, p + "v", hkv * HEAD).reshape(t, hkv, HEAD)
        q, k = (_rotate(y, self.pos, freq, True) for y in (q, k))
        self.state += [self.kept(k.reshape(t, -1)), self.kept(v.reshape(t, -1))]
        o = self.per_row(lambda q, k, v: _attend(q, k, v, HEAD ** -0.5, z["window"], z["keep"], SOFTCAP), q, k, v)
        return o * torch.sigmoid(self.linear(h, p + "g", hq * HEAD))

    def delta(self, h, i):
        p, t, heads = "l%d.mix." % i, h.shape[0], self.z["heads"]

        def conv(name):
            taps = self.w(p + name + ".conv", heads * HEAD, TAPS)

            def one(x):
                x = torch.cat([x.new_zeros(TAPS - 1, x.shape[1]), x])
                y = sum(x[j:x.shape[0] - TAPS + 1 + j] * taps[:, j] for j in range(TAPS))
                return y * torch.sigmoid(y)

            return self.per_row(one, self.linear(h, p + name, heads * HEAD)).reshape(t, heads, HEAD)

        q, k, v = conv("q"), conv("k"), conv("v")
        q, k = (y * torch.rsqrt((y * y).sum(-1, keepdim=True) + 1e-6) for y in (q, k))
        q = q * HEAD ** -0.5
        beta = torch.sigmoid(self.linear(h, p + "b", heads))
        step = self.linear(self.linear(h, p + "a1", RANK), p + "a2", heads * HEAD) + self.w(p + "dt_bias", heads * HEAD)
        step = torch.nn.functional.softplus(step, threshold=1e9).reshape(t, heads, HEAD)
        decay = torch.exp(-torch.exp(self.w(p + "A_log", heads))[:, None] * step)
        o, states = torch.empty_like(v), []
        for r in self.rows:
            s = torch.zeros(heads, HEAD, HEAD, dtype=HI, device=DEVICE)
            for j in range(r.start, r.stop):
                s = decay[j][:, :, None] * s
                u = beta[j][:, None] * (v[j] - (k[j][:, None, :] @ s)[:, 0])
                s = torch.baddbmm(s, k[j][:, :, None], u[:, None, :])
                o[j] = (q[j][:, None, :] @ s)[:, 0]
            states.append(s)
        self.state += [torch.stack(states), None]  # (the ring of the convolutions' inputs: the framework's own layout)
        gate = torch.sigmoid(self.linear(self.linear(h, p + "g1", RANK), p + "g2", heads * HEAD))
        return (_rms(o) * self.w(p + "norm", HEAD)).reshape(t, -1) * gate

    def zufadra(self):
        n, ff, x = self.case["width"], self.z["ff"], self.w("embed")[self.tokens]
        prev = torch.cat([self.tokens[:1], self.tokens[:-1]])
        pair = (prev * BIGRAM["mul_prev"] + self.tokens * BIGRAM["mul_cur"]) % BIGRAM["buckets"]
        pair[self.pos == 0] = BIGRAM["buckets"]
        x = x + self.w("bigram", BIGRAM["buckets"] + 1, n)[pair]
        for i in range(self.case["layers"]):
            p = "l%d." % i
            y = self.linear(self.windowed(x, i) if i % 2 else self.delta(x, i), p + "mix.o", n)
            x = x + _rms(y, self.w(p + "norm1", n))
            g = self.linear(x, p + "mlp.gate", ff) + self.w(p + "mlp.gate.b", ff)
            y = g * torch.sigmoid(g) * (self.linear(x, p + "mlp.up", ff) + self.w(p + "mlp.up.b", ff))
            x = x + _rms(self.linear(y, p + "mlp.down", n) + self.w(p + "mlp.down.b", n), self.w(p + "norm2", n))
        self.state.append(None)  # the tokens in front
        return _rms(x, self.w("final.norm", n))


@torch.no_grad()
def exact(case, seed):
    e = _Exact(case, seed)
    h = getattr(e, case["model"])()
    new = case["new"]
    at = torch.tensor([[r.stop - new + j for j in range(new)] for r in e.rows], device=DEVICE)
    logits = h[at] @ e.w("head").T
    out = {"first_logits": logits[:, 0], "tokens": logits.argmax(-1)}
    if new > 1:
        out["last_logits"] = logits[:, -1]
    if not case["padded"]:
        out["cache"] = e.state[:56]
    return out
