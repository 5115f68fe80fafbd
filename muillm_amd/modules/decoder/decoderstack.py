"""All decoder layers of a decode step through one library call.

The reference walks its layers from C++ only under tensor parallelism
(muillm/modules/models/llama/model.py:331-358 -> csrc/modules/parallel_decoder_stack.cpp); on
one GPU it calls its Python layer modules one by one (muillm/modules/decoder/decoder.py:130-165).
Here `mui_decoder_stack_step` enqueues the same per-layer sequence for every layer, so a step
that is not replayed from a HIP graph pays the host cost of one call instead of ~160.
`mui_decoder_stack_prompt` does the same for prompts and for steps of more batch rows than
the decode kernels take (~180 us of host time per layer otherwise, more than a prompt of 100 tokens keeps the GPU busy).
"""
import copy
import ctypes
import weakref
from typing import Optional

import torch
import torch.nn as nn
from torch.autograd import forward_ad

from ... import _lib, muillm_ext
from ..attention.baseattention import MuiBaseAttention
from ..attention.sdpaattention import MuiSdpaAttention
from ..gateupdownmlp import MuiGateUpDownMLP, _MuiGateUpSiLUMethod
from ..kvcache.cache_utils import MuiStaticCache
from ..linear import MuiLinear
from ..multilinear import MuiMultiLinear
from ..quantized.int8gateupdownmlp import MuiInt8GateUpDownMLP
from ..quantized.int8linear import MuiInt8Linear
from ..realrows import RealRows
from .decoder import MuiDecoderLayer


def _at(m, name: str):
    """m.name, from where nn.Module keeps it; None where it has none. (A layer has some sixty to read, in front of an idle GPU; nn.Module's own lookup takes several times as long.)"""
    d = m.__dict__
    v = d.get(name)
    if v is None:
        v = d["_parameters"].get(name)
        if v is None:
            v = d["_modules"].get(name)
            if v is None:
                v = d["_buffers"].get(name)
    return v


def _group_shift(m) -> int:
    """0 for a 16-bit or per-channel int8 module, the group size's log2 for the group format."""
    if type(m) is MuiInt8Linear and not m.per_channel:
        return int(m.quantizer.group_size_shift)
    if type(m) is MuiInt8GateUpDownMLP and not m.per_channel:
        return int(m.group_size_shift)
    return 0


def _plain_linear(m, normalize: Optional[bool] = None) -> bool:
    """A bias-free MuiLinear, or a bias-free MuiInt8Linear (per-channel, or the group format with
    groups of at least 16 that divide the rows)."""
    if type(m) is MuiInt8Linear:
        if _at(m, "bias") is not None or not m.dispatchable or (normalize is not None and bool(m.normalize) != normalize):
            return False
        if m.per_channel:
            return _at(m, "weights_int8").is_contiguous() and _at(m, "scales").is_contiguous()
        return (m.quantizer.group_size_shift >= 4 and m.in_features % 16 == 0 and _at(m, "weights_uint8").is_contiguous()
                and _at(m, "scales_min_vals").is_contiguous())
    if type(m) is not MuiLinear or _at(m, "bias") is not None:
        return False
    w = _at(m, "weight")
    return w.is_cuda and w.stride(1) == 1 and (normalize is None or bool(m.normalize) == normalize)


def _linear_fields(m):
    """(weight tensor, row pitch, scales tensor or None, [(owner, attribute, object)]) of a projection;
    "scales" are per-channel scales or, in the group format, the (scale, min) pairs."""
    if type(m) is MuiInt8Linear:
        names = ("weights_int8", "scales") if m.per_channel else ("weights_uint8", "scales_min_vals")
        w, sc = _at(m, names[0]), _at(m, names[1])
        return w, w.stride(0), sc, [(m, names[0], w), (m, names[1], sc)]
    w = _at(m, "weight")
    return w, w.stride(0), None, [(m, "weight", w)]


def _scales_of(mlp) -> str:
    """What an int8 MLP calls its gate and up scales: [inter, 2], or [inter, 2, G, 2] (scale, min) pairs."""
    return "gate_up_scales" if mlp.per_channel else "gate_up_scales_min_vals"


def _layer_sizes(layer) -> Optional[tuple]:
    """(hidden, query heads, key / value heads, intermediate) of a layer, or None where its tensors are of other sizes: kernels go by the sizes that a descriptor states."""
    multi, attn, mlp = _at(layer, "qkv_proj"), _at(layer, "self_attn"), _at(layer, "mlp")
    qkv = _at(multi, "linear")
    hidden, inter = qkv.in_features, mlp.intermediate_size
    q, kv = attn.num_heads * attn.head_dim, attn.num_key_value_heads * attn.head_dim

    def fits(m, n: int, k: int) -> bool:
        if type(m) is not MuiInt8Linear:
            return _at(m, "weight").shape == (n, k)
        if m.per_channel:
            return _at(m, "weights_int8").shape == (n, k) and _at(m, "scales").shape == (n,)
        return _at(m, "weights_uint8").shape == (n, k) and _at(m, "scales_min_vals").numel() == 2 * n * (k >> m.quantizer.group_size_shift)

    if not (fits(qkv, q + 2 * kv, hidden) and fits(_at(attn, "o_proj"), hidden, q) and fits(_at(mlp, "down_proj"), hidden, inter)):
        return None
    if multi.slice_starts != [0, q, q + kv] or _at(qkv, "norm_weights").shape != (hidden,) or _at(mlp, "norm_weights").shape != (hidden,):
        return None
    if type(mlp) is MuiGateUpDownMLP:
        if not (fits(_at(mlp, "gate_proj"), inter, hidden) and fits(_at(mlp, "up_proj"), inter, hidden)):
            return None
    else:
        sc = _at(mlp, _scales_of(mlp))
        if _at(mlp, "gate_up_weights").shape != (inter, 2, hidden) or (
                sc.shape != (inter, 2) if mlp.per_channel else sc.numel() != 4 * inter * (hidden >> mlp.group_size_shift)):
            return None
    return hidden, attn.num_heads, attn.num_key_value_heads, inter


def _rotate_with(attentions, cos, sin) -> bool:
    """Whether all of them still rotate with these tables (looked up past nn.Module's slow attribute access: asked before every call)."""
    for attn in attentions:
        rotary = attn.__dict__["_modules"].get("rotary_emb")
        if rotary is None:
            return False
        d = rotary.__dict__
        if d.get("cos32") is not cos or d.get("sin32") is not sin:
            return False
    return True


def _held(t) -> Optional[tuple]:
    """What a descriptor takes from a tensor. As long as the module's tensor gives the same, the memory is the module's and the descriptor holds: the tensor itself is neither
    kept alive nor referred to (torch.utils.swap_tensors refuses tensors with weak references)."""
    return None if t is None else (t.data_ptr(), t.dtype, t.shape, t.stride())


def _tensor(d: dict, name: str):
    """A module's tensor, from its __dict__: an attribute (a parameter that was deleted and set again is a plain one), a parameter, a buffer."""
    t = d.get(name)
    if t is None:
        t = d["_parameters"].get(name)
        if t is None:
            t = d["_buffers"].get(name)
    return t


def _handle_agrees(m, weight, gain) -> bool:
    """Whether a MuiLinear's handle, by which its module computes, names what the module names (a tensor that was replaced is the module's alone until finalize_init())."""
    handle = m.__dict__["cpp_module"]
    return (handle is not None and handle.weights is weight and handle.norm_weights is gain and handle.epsilon == m.__dict__["variance_epsilon"]
            and handle.mul_bias is None and handle.add_bias is None)


def _linear_reads(m) -> tuple:
    """What a descriptor, or the choice to use one, goes by in a projection."""
    d, kind = m.__dict__, type(m)
    norm = _tensor(d, "norm_weights")
    gain = None if norm is None else (norm.data_ptr(), norm.dtype, norm.shape, norm.stride())
    if kind is MuiLinear:
        w = _tensor(d, "weight")
        return (kind, w.data_ptr(), w.dtype, w.shape, w.stride(), gain, _tensor(d, "bias") is None, d["normalize"], d["variance_epsilon"], d["in_features"],
                _handle_agrees(m, w, norm))
    codes, scales = ("weights_int8", "scales") if d["per_channel"] else ("weights_uint8", "scales_min_vals")
    return (kind, _held(_tensor(d, codes)), _held(_tensor(d, scales)), gain, _tensor(d, "bias") is None, d["normalize"], d["variance_epsilon"], d["in_features"],
            d["per_channel"], d["dispatchable"], None if d["per_channel"] else d["quantizer"].group_size_shift)


def _layer_reads(layer) -> Optional[tuple]:
    """The same of a whole layer. Modules are gone through by what they hold and not by which they are; None where they are not as expected."""
    try:
        parts = layer.__dict__["_modules"]
        multi, attn, mlp = parts["qkv_proj"], parts["self_attn"], parts["mlp"]
        attn_parts, mlp_parts = attn.__dict__["_modules"], mlp.__dict__["_modules"]
        a, f, rotary = attn.__dict__, mlp.__dict__, attn_parts["rotary_emb"].__dict__
        cos, sin, handle = rotary["cos32"], rotary["sin32"], rotary["cpp_module"]
        reads = (type(layer), type(multi), tuple(multi.__dict__["slice_starts"]), _linear_reads(multi.__dict__["_modules"]["linear"]),
                 type(attn), a["training"], a["layer_idx"], a["num_heads"], a["num_key_value_heads"], a["head_dim"], _linear_reads(attn_parts["o_proj"]),
                 id(cos), id(sin), rotary["dispatchable"], handle is not None and handle.cos32 is cos and handle.sin32 is sin and handle.layer_idx,
                 type(mlp), _held(_tensor(f, "norm_weights")), f["normalize"], f["variance_epsilon"], f["intermediate_size"], f["dispatchable"],
                 type(mlp_parts["activation_function"]), _linear_reads(mlp_parts["down_proj"]))
        if type(mlp) is MuiGateUpDownMLP:
            return reads + (f["method"], _linear_reads(mlp_parts["gate_proj"]), _linear_reads(mlp_parts["up_proj"]))
        return reads + (f["per_channel"], f.get("group_size_shift"), _held(_tensor(f, "gate_up_weights")), _held(_tensor(f, _scales_of(mlp))))
    except (AttributeError, KeyError):
        return None


def _ptr(t) -> Optional[int]:
    return None if t is None else t.data_ptr()


class MuiDecoderStack:
    """Descriptor + workspace of `mui_decoder_stack_step` for one model, cache and batch size.

    Holds plain pointers: it has to be rebuilt when the cache is re-allocated (`matches`)."""

    def __init__(self, layers, rotary_emb, cache: MuiStaticCache, batch: int):
        self.lib = _lib.load()
        first = layers[0]
        attn0: MuiBaseAttention = first.self_attn
        self.dtype, self.device = first.qkv_proj.linear.norm_weights.dtype, first.qkv_proj.linear.norm_weights.device
        self.batch = batch
        self.hidden = first.qkv_proj.linear.in_features
        self.hq, self.hkv, self.d = attn0.num_heads, attn0.num_key_value_heads, attn0.head_dim
        self.cos32, self.sin32 = attn0.rotary_emb.cos32, attn0.rotary_emb.sin32
        kc0 = cache.key_cache[0]
        cb, chs, cts = kc0.stride(0), kc0.stride(1), kc0.stride(2)
        self.max_cache_len = kc0.shape[2]
        self._layer_list, self._attentions = layers, [layer.self_attn for layer in layers]
        self._cache_ptrs = tuple(t.data_ptr() for t in cache.key_cache) + tuple(t.data_ptr() for t in cache.value_cache)
        self._keep, self._owners = [], []  # tensors the descriptor points into; what matches() compares
        arr = (_lib.MuiDecoderLayerDesc * len(layers))()
        for i, layer in enumerate(layers):
            multi, attn, mlp = _at(layer, "qkv_proj"), _at(layer, "self_attn"), _at(layer, "mlp")
            qkv, o, down = _at(multi, "linear"), _at(attn, "o_proj"), _at(mlp, "down_proj")
            kc, vc = cache.key_cache[attn.layer_idx], cache.value_cache[attn.layer_idx]
            if (kc.stride(), vc.stride()) != (kc0.stride(), kc0.stride()):
                raise ValueError("cache layers must share one layout")
            qw, qp, qs, q_own = _linear_fields(qkv)
            ow, op, osc, o_own = _linear_fields(o)
            dw, dp, ds, d_own = _linear_fields(down)
            shift = max(_group_shift(m) for m in (qkv, o, mlp, down))
            if type(mlp) is MuiInt8GateUpDownMLP:
                gu = _at(mlp, "gate_up_weights")  # [inter, 2, hidden] codes
                g_ptr, u_ptr, g_pitch = gu.data_ptr(), gu.data_ptr() + gu.stride(1), gu.stride(0)
                gs_name = _scales_of(mlp)
                gs = _at(mlp, gs_name)
                gs_ptr, us_ptr = gs.data_ptr(), gs.data_ptr() + gs.stride(1) * gs.element_size()
                gs_stride = gs.stride(0)
                gu_own = [(mlp, "gate_up_weights", gu), (mlp, gs_name, gs)]
            else:
                gate, up = _at(mlp, "gate_proj"), _at(mlp, "up_proj")
                g, u = _at(gate, "weight"), _at(up, "weight")
                g_ptr, u_ptr, g_pitch = g.data_ptr(), u.data_ptr(), g.stride(0)
                gs_ptr, us_ptr, gs_stride = None, None, 0
                gu_own = [(mlp, "gate_proj", gate), (mlp, "up_proj", up), (gate, "weight", g), (up, "weight", u)]
            qn, mn = _at(qkv, "norm_weights"), _at(mlp, "norm_weights")
            arr[i] = _lib.MuiDecoderLayerDesc(
                qn.data_ptr(), qw.data_ptr(), qp, ow.data_ptr(), op,
                mn.data_ptr(), g_ptr, u_ptr, g_pitch, dw.data_ptr(), dp, kc.data_ptr(), vc.data_ptr(),
                _ptr(qs), _ptr(osc), gs_ptr, us_ptr, gs_stride, _ptr(ds), shift)
            self._built_from([(layer, "qkv_proj", multi), (layer, "self_attn", attn), (layer, "mlp", mlp), (multi, "linear", qkv),
                              (qkv, "norm_weights", qn), (attn, "o_proj", o), (mlp, "norm_weights", mn), (mlp, "down_proj", down)]
                             + q_own + o_own + d_own + gu_own, (kc, vc))
        self._layers = arr
        self.desc = _lib.MuiDecoderStackDesc(
            muillm_ext._dtype_code(first.qkv_proj.linear.norm_weights), len(layers), self.hidden, self.hq, self.hkv,
            self.d, first.mlp.intermediate_size, float(first.qkv_proj.linear.variance_epsilon),
            ctypes.cast(arr, ctypes.POINTER(_lib.MuiDecoderLayerDesc)), self.cos32.data_ptr(), self.sin32.data_ptr(),
            self.cos32.stride(0), self.cos32.shape[0], cb, chs, cts, self.max_cache_len)
        self._ws = None
        self._ws_splits = 0

    def _built_from(self, owners, cache_tensors) -> None:
        """owners: [(module, attribute name, object)] of a layer. The objects are kept, tensors with what they hold."""
        self._keep += [v for _, _, v in owners if isinstance(v, torch.Tensor)] + list(cache_tensors)
        self._owners += [(m, name, v, _held(v) if isinstance(v, torch.Tensor) else None) for m, name, v in owners]

    @staticmethod
    def eligible(layers, rotary_emb, cache, batch: int) -> bool:
        """fp16 / bf16 Llama-shaped layers of one size without biases on a static cache, head_dim 128;
        every projection 16-bit or int8 (per-channel, or the reference's group format)."""
        if not isinstance(cache, MuiStaticCache) or len(layers) == 0 or batch > _lib.MUI_MAX_TOKENS:
            return False
        if not getattr(rotary_emb, "dispatchable", False):
            return False
        eps, dtype, sizes, tables = None, None, None, None
        for layer in layers:
            multi, attn, mlp = _at(layer, "qkv_proj"), _at(layer, "self_attn"), _at(layer, "mlp")
            if type(multi) is not MuiMultiLinear or not isinstance(attn, MuiBaseAttention) or type(mlp) not in (MuiGateUpDownMLP, MuiInt8GateUpDownMLP):
                return False
            qkv, o, down = _at(multi, "linear"), _at(attn, "o_proj"), _at(mlp, "down_proj")
            if not (_plain_linear(qkv, True) and _plain_linear(o, False) and _plain_linear(down, False)):
                return False
            if attn.head_dim != 128:
                return False
            # a layer rotates with its own module's tables: they have to be the same for all
            rotary = _at(attn, "rotary_emb")
            if not getattr(rotary, "dispatchable", False) or (tables is not None and (rotary.cos32 is not tables[0] or rotary.sin32 is not tables[1])):
                return False
            tables = (rotary.cos32, rotary.sin32)
            if type(mlp) is MuiGateUpDownMLP:
                gate, up = _at(mlp, "gate_proj"), _at(mlp, "up_proj")
                if type(gate) is not MuiLinear or type(up) is not MuiLinear or not (_plain_linear(gate, False) and _plain_linear(up, False)):
                    return False
                gate, up = _at(gate, "weight"), _at(up, "weight")
                if gate.stride(0) != up.stride(0):
                    return False
                held = [gate, up]
            else:
                if not (mlp.dispatchable and _at(mlp, "gate_up_weights").is_contiguous()):
                    return False
                sc = _at(mlp, _scales_of(mlp))
                if not sc.is_contiguous() or (not mlp.per_channel and mlp.group_size_shift < 4):
                    return False
                held = [sc]
            if not mlp.normalize or not isinstance(_at(mlp, "activation_function"), nn.SiLU):
                return False
            w, mw = _at(qkv, "norm_weights"), _at(mlp, "norm_weights")
            if w is None or mw is None or w.dtype not in (torch.float16, torch.bfloat16):
                return False
            if cache.key_cache[attn.layer_idx].dtype != w.dtype or (dtype is not None and w.dtype != dtype):
                return False
            dtype = w.dtype
            of = _layer_sizes(layer)
            if of is None or (sizes is not None and of != sizes):
                return False
            sizes = of
            # one type throughout, as the kernels read it (the modules refuse others)
            held += [_at(m, "weight") if type(m) is MuiLinear else _at(m, "scales") if m.per_channel else _at(m, "scales_min_vals") for m in (qkv, o, down)] + [mw]
            if any(t.dtype != dtype for t in held):
                return False
            # the int8 projections of a layer share one format: all per-channel, or all in the group
            # format with one group size (the layer descriptor carries a single shift)
            if len({_group_shift(m) for m in (qkv, o, mlp, down) if type(m) in (MuiInt8Linear, MuiInt8GateUpDownMLP)}) > 1:
                return False
            e = (float(qkv.variance_epsilon), float(mlp.variance_epsilon))
            if e[0] != e[1] or (eps is not None and e != eps):
                return False
            eps = e
        return True

    def matches(self, layers, cache: MuiStaticCache, batch: int) -> bool:
        """Still valid for this step? The cache tensors are where they were, and every module and
        tensor the descriptor was built from is still the object in place, with the memory it had (a
        later quantize_layers / .to() / weight swap replaces them, `.data = ` its memory)."""
        if batch != self.batch or layers is not self._layer_list:
            return False
        for owner, name, obj, held in self._owners:
            d = owner.__dict__
            if held is None:
                if d["_modules"].get(name) is not obj:
                    return False
            elif _tensor(d, name) is not obj or _held(obj) != held:
                return False
        if not _rotate_with(self._attentions, self.cos32, self.sin32):
            return False
        ptrs = tuple(t.data_ptr() for t in cache.key_cache) + tuple(t.data_ptr() for t in cache.value_cache)
        return ptrs == self._cache_ptrs

    def step(self, hidden_in: torch.Tensor, position_ids: torch.Tensor, cache_position: torch.Tensor,
             seq_len: Optional[int], mask: Optional[torch.Tensor]) -> torch.Tensor:
        """hidden_in [B, 1, hidden] -> output of the last layer [B, 1, hidden]."""
        lib, b = self.lib, self.batch
        x = hidden_in.reshape(b, self.hidden)
        if not x.is_contiguous():
            x = x.contiguous()
        hint = seq_len if seq_len is not None else self.max_cache_len
        n_splits = lib.mui_flash_decode_splits(b, self.hq, self.hkv, int(hint))
        if self._ws is None or n_splits > self._ws_splits:
            nbytes = lib.mui_decoder_stack_workspace_bytes(ctypes.byref(self.desc), b, n_splits)
            self._ws = torch.empty(nbytes + 256, dtype=torch.uint8, device=self.device)
            self._ws_splits = n_splits
        ws_ptr = (self._ws.data_ptr() + 255) & ~255
        pos = position_ids.reshape(-1)
        if pos.dtype != torch.int64 or cache_position.dtype != torch.int64:
            raise RuntimeError("position_ids and cache_position must be int64")
        mask_ptr, mask_bs = None, 0
        if mask is not None:
            mask = muillm_ext._mask_rows(mask, b, x.dtype)
            mask_ptr, mask_bs = mask.data_ptr(), mask.stride(0)
        out = torch.empty((b, 1, self.hidden), dtype=x.dtype, device=x.device)
        muillm_ext.check(
            lib.mui_decoder_stack_step(muillm_ext._stream(x), ctypes.byref(self.desc), b, x.data_ptr(), out.data_ptr(),
                                       pos.data_ptr(), 1 if pos.numel() > 1 else 0, cache_position.data_ptr(),
                                       -1 if seq_len is None else int(seq_len), mask_ptr, mask_bs, n_splits, ws_ptr),
            "mui_decoder_stack_step")
        return out


class MuiPromptStack(MuiDecoderStack):
    """The same for `mui_decoder_stack_prompt`: prompts, and steps of more batch rows than the decode kernels take. Layers called one by one run the same
    kernels; here nobody can listen in between, so a model with hooks stays with its modules.

    Before every call the layers are read again and compared with what they were (current(), a few us per layer, where examining them and building the descriptor takes
    ~20 with an idle GPU waiting). Tensors are compared by what they hold: nothing is kept alive beyond a call."""

    def __init__(self, layers, rotary_emb, cache: MuiStaticCache):
        super().__init__(layers, rotary_emb, cache, 1)
        self._watched, self._layer_refs = None, [weakref.ref(layer) for layer in layers]
        self._cache_layers = [attn.layer_idx for attn in self._attentions]
        self._layer_list = self._attentions = self._cache_ptrs = None  # (nothing is held but weakly)
        self._bound(cache)
        # (the library's call converts codes, the modules dequantise long prompts' matrices)
        ks = (self.hidden, self.hq * self.d, layers[0].mlp.intermediate_size)
        codes = {(x.int8_group_size_shift, (x.qkv_scales or 0) | (x.o_scales or 0) | (x.gate_scales or 0) | (x.up_scales or 0) | (x.down_scales or 0))
                 for x in self._layers if x.qkv_scales or x.o_scales or x.gate_scales or x.down_scales}
        self._most_rows = min([muillm_ext.int8_dequantised_from(self.dtype, k, *of) - 1 for k in ks for of in codes], default=1 << 30)

    def _built_from(self, owners, cache_tensors) -> None:
        pass  # see remember()

    def remember(self) -> None:
        """What current() compares with. (Made behind the first call, while the GPU is at work.)"""
        if self._watched is None:
            self._watched = [_layer_reads(r()) for r in self._layer_refs]

    @staticmethod
    def eligible(layers, rotary_emb, cache) -> bool:
        """Whether the layers, called one by one, would run the kernels that mui_decoder_stack_prompt runs."""
        if not MuiDecoderStack.eligible(layers, rotary_emb, cache, 1):
            return False
        if not MuiPromptStack._cache_serves(cache):
            return False
        for layer in layers:
            attn, mlp = _at(layer, "self_attn"), _at(layer, "mlp")
            qkv, o, down = _at(_at(layer, "qkv_proj"), "linear"), _at(attn, "o_proj"), _at(mlp, "down_proj")
            if type(layer) is not MuiDecoderLayer or type(attn) is not MuiSdpaAttention or attn.training:
                return False
            rotary = _at(attn, "rotary_emb")
            handle = rotary.cpp_module  # (prompts rotate by what the handle names)
            if handle is None or handle.cos32 is not rotary.cos32 or handle.sin32 is not rotary.sin32 or handle.layer_idx != attn.layer_idx:
                return False
            if type(mlp) is MuiGateUpDownMLP and (not mlp.dispatchable or mlp.method == _MuiGateUpSiLUMethod.GATEUPSILU_UNFUSED):
                return False
            for m in (qkv, o) + ((down,) if type(mlp) is MuiInt8GateUpDownMLP else ()):
                if type(m) is MuiLinear and not _handle_agrees(m, _at(m, "weight"), _at(m, "norm_weights")):
                    return False
            hidden, inter = qkv.in_features, mlp.intermediate_size
            if hidden % 8 or inter % 8 or hidden > 16384:
                return False
            int8 = any(type(m) in (MuiInt8Linear, MuiInt8GateUpDownMLP) for m in (qkv, o, mlp, down))
            if int8 and (hidden % 16 or inter % 16 or (inter > 16384 and _at(qkv, "norm_weights").dtype != torch.float16)):
                return False
        return True

    @staticmethod
    def _cache_serves(cache: MuiStaticCache) -> bool:
        kc = cache.key_cache[0]
        return (kc.stride(3) == 1 and not any(x % 8 for x in kc.stride()[:3])
                and all(x.stride() == kc.stride() and x.dtype == kc.dtype and x.device == kc.device and x.data_ptr() % 16 == 0 for x in cache.tensors()))

    def _bound(self, cache: MuiStaticCache) -> None:
        self._cache = weakref.ref(cache)
        self._cache_tensors = [_held(t) for t in cache.tensors()]

    def bound_to(self, cache: MuiStaticCache) -> Optional["MuiPromptStack"]:
        """The same for another cache (a request brings its own), or None. A descriptor of its own: another thread may be in a call with this one."""
        kc = cache.key_cache[0]
        if (len(cache.key_cache) <= max(self._cache_layers) or kc.dtype != self.dtype or kc.device != self.device or kc.shape[1] != self.hkv
                or kc.shape[3] != self.d or not self._cache_serves(cache)):
            return None
        new = copy.copy(self)
        new._layers = type(self._layers).from_buffer_copy(self._layers)
        for i, at in enumerate(self._cache_layers):
            new._layers[i].k_cache, new._layers[i].v_cache = cache.key_cache[at].data_ptr(), cache.value_cache[at].data_ptr()
        new.desc = type(self.desc).from_buffer_copy(self.desc)
        new.desc.layers = ctypes.cast(new._layers, ctypes.POINTER(_lib.MuiDecoderLayerDesc))
        new.desc.cache_batch_stride, new.desc.cache_head_stride, new.desc.cache_token_stride = kc.stride()[:3]
        new.desc.max_cache_len = new.max_cache_len = kc.shape[2]
        new._bound(cache)
        return new

    def current(self, layers) -> bool:
        """Whether everything is as it was when the descriptor was built."""
        if len(layers) != len(self._layer_refs):
            return False
        for layer, r in zip(layers, self._layer_refs):
            if layer is not r():
                return False
        if self._watched is None:
            return False  # the first call did not come about
        for layer, reads in zip(layers, self._watched):
            if reads is None or _layer_reads(layer) != reads:
                return False
        return True

    def holds(self, cache: MuiStaticCache) -> bool:
        return cache is self._cache() and [_held(t) for t in cache.tensors()] == self._cache_tensors

    def takes(self, hidden_states: torch.Tensor, position_ids: torch.Tensor, cache_position: torch.Tensor, key_mask: Optional[torch.Tensor]) -> bool:
        """Whether this call can be made: its sizes, and nobody who listens to the modules."""
        b, t = hidden_states.shape[0], hidden_states.shape[1]
        if hidden_states.dtype != self.dtype or hidden_states.device != self.device or hidden_states.shape[2] != self.hidden:
            return False
        if forward_ad._current_level >= 0:
            return False  # forward mode: the linears' modules refuse tangents, of inputs and of weights; here they would be lost
        cache = self._cache()
        if b > cache.max_batch_size or b > 65535 or t > 65535 or not 1 <= b * t <= self._most_rows:
            return False
        if cache.get_seq_length() + t > self.max_cache_len:
            return False  # the modules refuse to read a cache beyond its rows
        if position_ids.dtype != torch.int64 or cache_position.dtype != torch.int64 or not (position_ids.is_cuda and cache_position.is_cuda):
            return False
        if tuple(position_ids.shape) not in ((1, t), (b, t)) or tuple(cache_position.shape) != (t,) or not cache_position.is_contiguous():
            return False
        if key_mask is not None and (key_mask.dtype != self.dtype or key_mask.dim() != 2 or key_mask.shape[0] != b or key_mask.stride(1) != 1
                                     or key_mask.shape[1] < (cache.get_seq_length() + t + 3) // 4 * 4 or not key_mask.is_cuda):
            return False
        g = nn.modules.module
        if g._global_forward_hooks or g._global_forward_pre_hooks:
            return False
        for r in self._layer_refs:
            layer = r()
            parts = layer.__dict__["_modules"]
            multi, attn, mlp = parts["qkv_proj"], parts["self_attn"], parts["mlp"]
            inside = mlp.__dict__["_modules"]
            for m in (layer, multi, multi.__dict__["_modules"]["linear"], attn, attn.__dict__["_modules"]["o_proj"], mlp, inside["down_proj"], inside.get("gate_proj", mlp),
                      inside.get("up_proj", mlp)):
                d = m.__dict__
                if d["_forward_hooks"] or d["_forward_pre_hooks"] or "forward" in d:
                    return False
            most = attn.prefill_kernel_max_tokens  # (set at any time, on a module or for all of them)
            if most is not None and t > most:
                return False
        return True

    def run_real(self, hidden_in: torch.Tensor, real: RealRows, position_ids: torch.Tensor, cache_position: torch.Tensor, seq_len: int,
                 mask: torch.Tensor) -> torch.Tensor:
        """hidden_in [1, real rows, hidden] of a padded batch of prompts -> output of the last layer, likewise. mask: the key mask that hides the padding."""
        lib, x, stream = self.lib, hidden_in.contiguous(), muillm_ext._stream(hidden_in)
        b, t, n = real.batch, real.tokens, real.n
        ws = torch.empty(lib.mui_decoder_stack_prompt_rows_bytes(ctypes.byref(self.desc), b, t, n) + 256, dtype=torch.uint8, device=x.device)
        linear_ws = muillm_ext._prompt_workspace(x, stream) if n > _lib.MUI_MAX_TOKENS else None
        pos, out = position_ids.contiguous(), torch.empty_like(x)
        muillm_ext.check(
            lib.mui_decoder_stack_prompt_rows(stream, ctypes.byref(self.desc), b, t, n, real.rows.data_ptr(), real.slots.data_ptr(), x.data_ptr(),
                                              out.data_ptr(), pos.data_ptr(), t if pos.shape[0] > 1 else 0, cache_position.data_ptr(), seq_len,
                                              mask.data_ptr(), mask.stride(0), (ws.data_ptr() + 255) & ~255, _ptr(linear_ws),
                                              0 if linear_ws is None else linear_ws.numel()), "mui_decoder_stack_prompt_rows")
        self.remember()
        return out

    def run(self, hidden_in: torch.Tensor, position_ids: torch.Tensor, cache_position: torch.Tensor, seq_len: Optional[int],
            mask: Optional[torch.Tensor]) -> torch.Tensor:
        """hidden_in [B, T, hidden] -> output of the last layer [B, T, hidden]. mask: T > 1 a key mask (see mui_prefill_attention), T 1 additive."""
        lib = self.lib
        x = hidden_in.contiguous()
        b, t = x.shape[0], x.shape[1]
        stream = muillm_ext._stream(x)
        n_splits = 1
        if t == 1:
            n_splits = lib.mui_flash_decode_splits(b, self.hq, self.hkv, int(seq_len if seq_len is not None else self.max_cache_len))
            mask = None if mask is None else muillm_ext._mask_rows(mask, b, x.dtype)
        ws = torch.empty(lib.mui_decoder_stack_prompt_bytes(ctypes.byref(self.desc), b, t, n_splits) + 256, dtype=torch.uint8, device=x.device)
        linear_ws = muillm_ext._prompt_workspace(x, stream) if b * t > _lib.MUI_MAX_TOKENS else None
        pos = position_ids.contiguous()
        out = torch.empty_like(x)
        muillm_ext.check(
            lib.mui_decoder_stack_prompt(stream, ctypes.byref(self.desc), b, t, x.data_ptr(), out.data_ptr(), pos.data_ptr(),
                                         t if pos.shape[0] > 1 else 0, cache_position.data_ptr(), -1 if seq_len is None else int(seq_len),
                                         _ptr(mask), 0 if mask is None else mask.stride(0), n_splits, (ws.data_ptr() + 255) & ~255,
                                         _ptr(linear_ws), 0 if linear_ws is None else linear_ws.numel()),
            "mui_decoder_stack_prompt")
        self.remember()
        return out
