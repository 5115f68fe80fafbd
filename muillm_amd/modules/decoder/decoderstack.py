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
from .decoder import MuiDecoderLayer


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
        if m.bias is not None or not m.dispatchable or (normalize is not None and bool(m.normalize) != normalize):
            return False
        if m.per_channel:
            return m.weights_int8.is_contiguous() and m.scales.is_contiguous()
        return (m.quantizer.group_size_shift >= 4 and m.in_features % 16 == 0 and m.weights_uint8.is_contiguous()
                and m.scales_min_vals.is_contiguous())
    return (type(m) is MuiLinear and m.bias is None and m.weight.is_cuda and m.weight.stride(1) == 1
            and (normalize is None or bool(m.normalize) == normalize))


def _linear_fields(m):
    """(weight tensor, row pitch, scales tensor or None, [(owner, attribute, object)]) of a projection;
    "scales" are per-channel scales or, in the group format, the (scale, min) pairs."""
    if type(m) is MuiInt8Linear:
        if m.per_channel:
            return m.weights_int8, m.weights_int8.stride(0), m.scales, [(m, "weights_int8", m.weights_int8),
                                                                         (m, "scales", m.scales)]
        return m.weights_uint8, m.weights_uint8.stride(0), m.scales_min_vals, [
            (m, "weights_uint8", m.weights_uint8), (m, "scales_min_vals", m.scales_min_vals)]
    return m.weight, m.weight.stride(0), None, [(m, "weight", m.weight)]


def _layer_sizes(layer) -> Optional[tuple]:
    """(hidden, query heads, key / value heads, intermediate) of a layer, or None where its tensors are of other sizes: kernels go by the sizes that a descriptor states."""
    qkv, attn, mlp = layer.qkv_proj.linear, layer.self_attn, layer.mlp
    hidden, inter = qkv.in_features, mlp.intermediate_size
    q, kv = attn.num_heads * attn.head_dim, attn.num_key_value_heads * attn.head_dim

    def fits(m, n: int, k: int) -> bool:
        if type(m) is not MuiInt8Linear:
            return m.weight.shape == (n, k)
        if m.per_channel:
            return m.weights_int8.shape == (n, k) and m.scales.shape == (n,)
        return m.weights_uint8.shape == (n, k) and m.scales_min_vals.numel() == 2 * n * (k >> m.quantizer.group_size_shift)

    if not (fits(qkv, q + 2 * kv, hidden) and fits(attn.o_proj, hidden, q) and fits(mlp.down_proj, hidden, inter)):
        return None
    if layer.qkv_proj.slice_starts != [0, q, q + kv] or qkv.norm_weights.shape != (hidden,) or mlp.norm_weights.shape != (hidden,):
        return None
    if type(mlp) is MuiGateUpDownMLP:
        if not (fits(mlp.gate_proj, inter, hidden) and fits(mlp.up_proj, inter, hidden)):
            return None
    elif mlp.gate_up_weights.shape != (inter, 2, hidden) or (
            mlp.gate_up_scales.shape != (inter, 2) if mlp.per_channel
            else mlp.gate_up_scales_min_vals.numel() != 4 * inter * (hidden >> mlp.group_size_shift)):
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


_TENSORS = {MuiLinear: ("weight", "bias", "norm_weights"),
            MuiInt8Linear: ("weights_int8", "scales", "weights_uint8", "scales_min_vals", "bias", "norm_weights"),
            MuiGateUpDownMLP: ("norm_weights",),
            MuiInt8GateUpDownMLP: ("norm_weights", "gate_up_weights", "gate_up_scales", "gate_up_scales_min_vals")}


# what else a descriptor, or the choice to use one, goes by (a name may be missing: its default stands in the class then)
_LINEAR = ("variance_epsilon", "normalize", "in_features", "out_features", "dispatchable", "per_channel", "quantizer")
_MLP = ("variance_epsilon", "normalize", "intermediate_size", "dispatchable", "method", "per_channel", "group_size_shift")
_VALUES = {MuiLinear: _LINEAR, MuiInt8Linear: _LINEAR, MuiGateUpDownMLP: _MLP, MuiInt8GateUpDownMLP: _MLP, MuiMultiLinear: ("slice_starts", "slice_ends"),
           MuiSdpaAttention: ("training", "layer_idx", "num_heads", "num_key_value_heads", "head_dim")}
_ABSENT = object()


def _nothing():  # in the place of a weak reference
    return None


def _same(v, ref) -> bool:
    """Whether v is what ref was made of. (What has gone is nobody's.)"""
    return v is ref() and (v is not None or ref is _nothing)


def _tensor(d: dict, name: str):
    """A module's tensor, from its __dict__: an attribute (a parameter that was deleted and set again is a plain one), a parameter, a buffer."""
    t = d.get(name)
    if t is None:
        t = d["_parameters"].get(name)
        if t is None:
            t = d["_buffers"].get(name)
    return t


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
        self._attentions = [layer.self_attn for layer in layers]
        kc0 = cache.key_cache[0]
        cb, chs, cts = kc0.stride(0), kc0.stride(1), kc0.stride(2)
        self.max_cache_len = kc0.shape[2]
        self._cache_ptrs = tuple(t.data_ptr() for t in cache.key_cache) + tuple(t.data_ptr() for t in cache.value_cache)
        self._keep = []  # tensors the descriptor points into
        self._layer_list = layers
        self._owners = []  # (module, attribute name, object) the descriptor was built from, tensors with what they hold
        arr = (_lib.MuiDecoderLayerDesc * len(layers))()
        for i, layer in enumerate(layers):
            qkv, attn, mlp = layer.qkv_proj.linear, layer.self_attn, layer.mlp
            kc, vc = cache.key_cache[attn.layer_idx], cache.value_cache[attn.layer_idx]
            if (kc.stride(), vc.stride()) != (kc0.stride(), kc0.stride()):
                raise ValueError("cache layers must share one layout")
            qw, qp, qs, q_own = _linear_fields(qkv)
            ow, op, osc, o_own = _linear_fields(attn.o_proj)
            dw, dp, ds, d_own = _linear_fields(mlp.down_proj)
            shift = max(_group_shift(m) for m in (qkv, attn.o_proj, mlp, mlp.down_proj))
            if type(mlp) is MuiInt8GateUpDownMLP:
                gu = mlp.gate_up_weights  # [inter, 2, hidden] codes
                g_ptr, u_ptr, g_pitch = gu.data_ptr(), gu.data_ptr() + gu.stride(1), gu.stride(0)
                if mlp.per_channel:
                    gs, gs_name = mlp.gate_up_scales, "gate_up_scales"  # [inter, 2] scales
                else:
                    gs, gs_name = mlp.gate_up_scales_min_vals, "gate_up_scales_min_vals"  # [inter, 2, G, 2] pairs
                gs_ptr, us_ptr = gs.data_ptr(), gs.data_ptr() + gs.stride(1) * gs.element_size()
                gs_stride = gs.stride(0)
                gu_keep = [gu, gs]
                gu_own = [(mlp, "gate_up_weights", gu), (mlp, gs_name, gs)]
            else:
                g, u = mlp.gate_proj.weight, mlp.up_proj.weight
                g_ptr, u_ptr, g_pitch = g.data_ptr(), u.data_ptr(), g.stride(0)
                gs_ptr, us_ptr, gs_stride = None, None, 0
                gu_keep = [g, u]
                gu_own = [(mlp, "gate_proj", mlp.gate_proj), (mlp, "up_proj", mlp.up_proj), (mlp.gate_proj, "weight", g), (mlp.up_proj, "weight", u)]
            arr[i] = _lib.MuiDecoderLayerDesc(
                qkv.norm_weights.data_ptr(), qw.data_ptr(), qp, ow.data_ptr(), op,
                mlp.norm_weights.data_ptr(), g_ptr, u_ptr, g_pitch, dw.data_ptr(), dp, kc.data_ptr(), vc.data_ptr(),
                _ptr(qs), _ptr(osc), gs_ptr, us_ptr, gs_stride, _ptr(ds), shift)
            self._keep += [qkv.norm_weights, qw, qs, ow, osc, mlp.norm_weights, dw, ds, kc, vc] + gu_keep
            owners = [(layer, "qkv_proj", layer.qkv_proj), (layer, "self_attn", attn), (layer, "mlp", mlp),
                      (layer.qkv_proj, "linear", qkv), (qkv, "norm_weights", qkv.norm_weights),
                      (attn, "o_proj", attn.o_proj), (mlp, "norm_weights", mlp.norm_weights),
                      (mlp, "down_proj", mlp.down_proj)] + q_own + o_own + d_own + gu_own
            self._owners += [(m, name, v, _held(v) if isinstance(v, torch.Tensor) else None) for m, name, v in owners]
        self._layers = arr
        self.desc = _lib.MuiDecoderStackDesc(
            muillm_ext._dtype_code(first.qkv_proj.linear.norm_weights), len(layers), self.hidden, self.hq, self.hkv,
            self.d, first.mlp.intermediate_size, float(first.qkv_proj.linear.variance_epsilon),
            ctypes.cast(arr, ctypes.POINTER(_lib.MuiDecoderLayerDesc)), self.cos32.data_ptr(), self.sin32.data_ptr(),
            self.cos32.stride(0), self.cos32.shape[0], cb, chs, cts, self.max_cache_len)
        self._ws = None
        self._ws_splits = 0

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
            qkv, attn, mlp = getattr(layer, "qkv_proj", None), getattr(layer, "self_attn", None), getattr(layer, "mlp", None)
            if type(qkv) is not MuiMultiLinear or not _plain_linear(qkv.linear, True):
                return False
            if not isinstance(attn, MuiBaseAttention) or not _plain_linear(attn.o_proj, False):
                return False
            if attn.head_dim != 128:
                return False
            # a layer rotates with its own module's tables: they have to be the same for all
            rotary = attn.rotary_emb
            if not rotary.dispatchable or (tables is not None and (rotary.cos32 is not tables[0] or rotary.sin32 is not tables[1])):
                return False
            tables = (rotary.cos32, rotary.sin32)
            if type(mlp) is MuiGateUpDownMLP:
                if not all(_plain_linear(m, False) and type(m) is MuiLinear for m in (mlp.gate_proj, mlp.up_proj)):
                    return False
                if mlp.gate_proj.weight.stride(0) != mlp.up_proj.weight.stride(0):
                    return False
            elif type(mlp) is MuiInt8GateUpDownMLP:
                if not (mlp.dispatchable and mlp.gate_up_weights.is_contiguous()):
                    return False
                sc = mlp.gate_up_scales if mlp.per_channel else mlp.gate_up_scales_min_vals
                if not sc.is_contiguous() or (not mlp.per_channel and mlp.group_size_shift < 4):
                    return False
            else:
                return False
            if not mlp.normalize or not isinstance(mlp.activation_function, nn.SiLU):
                return False
            if not _plain_linear(mlp.down_proj, False):
                return False
            w = qkv.linear.norm_weights
            if w is None or mlp.norm_weights is None or w.dtype not in (torch.float16, torch.bfloat16):
                return False
            if cache.key_cache[attn.layer_idx].dtype != w.dtype or (dtype is not None and w.dtype != dtype):
                return False
            dtype = w.dtype
            of = _layer_sizes(layer)
            if of is None or (sizes is not None and of != sizes):
                return False
            sizes = of
            # one type throughout, as the kernels read it (the modules refuse others)
            held = [m.weight if type(m) is MuiLinear else m.scales if m.per_channel else m.scales_min_vals for m in (qkv.linear, attn.o_proj, mlp.down_proj)]
            held += [mlp.norm_weights] + ([mlp.gate_proj.weight, mlp.up_proj.weight] if type(mlp) is MuiGateUpDownMLP
                                          else [mlp.gate_up_scales if mlp.per_channel else mlp.gate_up_scales_min_vals])
            if any(t.dtype != dtype for t in held):
                return False
            # the int8 projections of a layer share one format: all per-channel, or all in the group
            # format with one group size (the layer descriptor carries a single shift)
            int8_mods = [m for m in (qkv.linear, attn.o_proj, mlp, mlp.down_proj)
                         if type(m) in (MuiInt8Linear, MuiInt8GateUpDownMLP)]
            if len({_group_shift(m) for m in int8_mods}) > 1:
                return False
            e = (float(qkv.linear.variance_epsilon), float(mlp.variance_epsilon))
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

    What the descriptor was built from is watched, modules by weak references and tensors by what they hold (current(), asked before every call, takes a few us per
    layer, where examining the layers anew takes ~35 with an idle GPU waiting): nothing is kept alive beyond a call."""

    def __init__(self, layers, rotary_emb, cache: MuiStaticCache):
        super().__init__(layers, rotary_emb, cache, 1)
        self._keep, self._owners, self._layer_list = [], [], None
        self._watched, self._layer_refs = None, [weakref.ref(layer) for layer in layers]
        self._cache_layers = [layer.self_attn.layer_idx for layer in layers]
        self._bound(cache)
        self._attentions = None  # (layers are held weakly here)
        int8 = any(type(m) in (MuiInt8Linear, MuiInt8GateUpDownMLP)
                   for layer in layers for m in (layer.qkv_proj.linear, layer.self_attn.o_proj, layer.mlp, layer.mlp.down_proj))
        self._most_rows = min(muillm_ext.INT8_DEQUANT_MIN_TOKENS, muillm_ext.INT8_GROUP_DEQUANT_MIN_TOKENS) - 1 if int8 else 1 << 30
        self._attention_refs = [weakref.ref(layer.self_attn) for layer in layers]

    def remember(self) -> None:
        """What current() compares with. (Made behind the first call, while the GPU is at work.)"""
        if self._watched is not None:
            return

        def ref(v):
            return _nothing if v is None else weakref.ref(v)

        watched = []  # per module: itself, its children, what its tensors hold, what else was read from it, its handle
        for layer in [r() for r in self._layer_refs]:
            qkv, attn, mlp = layer.qkv_proj, layer.self_attn, layer.mlp
            inside = [getattr(mlp, n) for n in ("gate_proj", "up_proj", "down_proj") if isinstance(getattr(mlp, n, None), nn.Module)]
            for m in [layer, qkv, qkv.linear, attn, attn.o_proj, mlp] + inside:
                d, kind = m.__dict__, type(m)
                watched.append((weakref.ref(m), [(k, ref(v)) for k, v in m._modules.items()],
                                [(k, _held(_tensor(d, k))) for k in _TENSORS.get(kind, ())],
                                [(k, d.get(k, _ABSENT)) for k in _VALUES.get(kind, ())], ref(d.get("cpp_module"))))
        self._watched = watched  # whole: another thread may ask meanwhile

    @staticmethod
    def eligible(layers, rotary_emb, cache) -> bool:
        """Whether the layers, called one by one, would run the kernels that mui_decoder_stack_prompt runs."""
        if not MuiDecoderStack.eligible(layers, rotary_emb, cache, 1):
            return False
        if not MuiPromptStack._cache_serves(cache):
            return False
        for layer in layers:
            qkv, attn, mlp = layer.qkv_proj.linear, layer.self_attn, layer.mlp
            if type(layer) is not MuiDecoderLayer or type(attn) is not MuiSdpaAttention or attn.training:
                return False
            rotary, handle = attn.rotary_emb, attn.rotary_emb.cpp_module  # (prompts rotate by what the handle names)
            if handle is None or handle.cos32 is not rotary.cos32 or handle.sin32 is not rotary.sin32 or handle.layer_idx != attn.layer_idx:
                return False
            if type(mlp) is MuiGateUpDownMLP and (not mlp.dispatchable or mlp.method == _MuiGateUpSiLUMethod.GATEUPSILU_UNFUSED):
                return False
            for m in (qkv, attn.o_proj) + ((mlp.down_proj,) if type(mlp) is MuiInt8GateUpDownMLP else ()):
                if type(m) is MuiLinear and (m.cpp_module is None or m.cpp_module.weights is not m.weight):
                    return False
            hidden, inter = qkv.in_features, mlp.intermediate_size
            if hidden % 8 or inter % 8 or hidden > 16384:
                return False
            int8 = any(type(m) in (MuiInt8Linear, MuiInt8GateUpDownMLP) for m in (qkv, attn.o_proj, mlp, mlp.down_proj))
            if int8 and (hidden % 16 or inter % 16 or (inter > 16384 and qkv.norm_weights.dtype != torch.float16)):
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
        attentions = [layer.__dict__["_modules"].get("self_attn") for layer in layers]
        if None in attentions or not _rotate_with(attentions, self.cos32, self.sin32):
            return False
        for attn in attentions:
            rotary = attn.__dict__["_modules"]["rotary_emb"].__dict__
            handle = rotary["cpp_module"]
            if handle is None or handle.cos32 is not self.cos32 or handle.sin32 is not self.sin32 or handle.layer_idx != attn.layer_idx or not rotary["dispatchable"]:
                return False
        for r, children, tensors, values, handle in self._watched:
            m = r()
            if m is None:
                return False
            d = m.__dict__
            mods = d["_modules"]
            if len(mods) != len(children):
                return False
            for k, v in children:
                if not _same(mods.get(k), v):
                    return False
            for k, v in tensors:
                if _held(_tensor(d, k)) != v:
                    return False
            for k, v in values:
                if d.get(k, _ABSENT) is not v:
                    return False
            if not _same(d.get("cpp_module"), handle):
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
        for r in self._attention_refs:  # (set at any time, on a module or for all of them)
            most = r().prefill_kernel_max_tokens
            if most is not None and t > most:
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
        modules = [r() for r, *_ in self._watched] if self._watched else [m for r in self._layer_refs for m in r().modules()]
        for m in modules:
            d = m.__dict__
            if d["_forward_hooks"] or d["_forward_pre_hooks"] or "forward" in d:
                return False
        return True

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
