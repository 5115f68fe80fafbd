"""Decoder layers with norms around each sublayer and an fp32 residual stream:
x <- x + m post_norm(mixer(pre_norm(x))), then the same with an optional feed-forward. The pre norms can be
left out: the sublayers then read x itself, rounded to the activations' type.

A sublayer's post norm, the residual sum and the next sublayer's input (its pre norm) are one kernel
(hybrid_ops.residual_norm), so a layer hands its last sublayer's output on unjoined: run_layers joins it
together with the input of whatever comes next."""
from typing import List, Optional

import torch
import torch.nn as nn

from ... import hybrid_ops
from ...engineconfig import MuiEngineConfig
from ...muillm_ext import ResidualBehind, ResidualFront
from ..module import MuiModule
from ..norm.rmsnorm import MuiRMSNorm


class MuiSandwichDecoderLayer(MuiModule):
    """mixer: a module with forward(h, cache, cache_position) and new_state(...); mlp: a module with
    forward(h), or None for a layer without feed-forward. Where the class of either has a takes_behind() that is true, its forward takes a
    `behind` for its last linear, and where it has a takes_front() that is, a `front` for its first. branch_scale: m."""

    def __init__(self, engine_config: MuiEngineConfig, hidden: int, mixer: MuiModule, mlp: Optional[MuiModule], eps: float,
                 device=None, dtype=None, pre_norms: bool = True, branch_scale: float = 1.0):
        super().__init__(engine_config=engine_config)

        def norm(there: bool):
            return MuiRMSNorm(engine_config, hidden, eps=eps, device=device, dtype=dtype) if there else None

        self.mixer, self.mlp, self.branch_scale = mixer, mlp, branch_scale
        self.pre_mixer_norm, self.post_mixer_norm = norm(pre_norms), norm(True)
        self.pre_mlp_norm, self.post_mlp_norm = norm(pre_norms and mlp is not None), norm(mlp is not None)


def run_layers(layers: List[MuiSandwichDecoderLayer], x: torch.Tensor, h: torch.Tensor, final_norm: MuiRMSNorm, eps: float,
               cache, cache_position: torch.Tensor, collect: Optional[list] = None, final_scale: float = 1.0) -> torch.Tensor:
    """x (fp32 residual stream) and h (the first sublayer's input) [B, T, hidden] through all layers; returns
    final_scale times the final norm's output. collect: a list that receives the residual stream after every layer."""
    shape = h.shape

    # (the functions in here carry no annotations: those are evaluated on every call)
    def join(x, y, post, m, following, scale=1.0):
        return hybrid_ops.residual_norm(x, y, post.weight, None if following is None else following.weight, eps,
                                        branch_scale=m, next_scale=scale, emit=True)

    # where it saves a launch the sublayer's last linear takes the join along, or, of a single row, the next sublayer's first product
    rows = h.numel() // h.shape[-1]
    along = ResidualBehind.worth_it(rows)
    ahead = rows == 1 and collect is None

    def sublayer(module, args, x, post, m, following, scale=1.0):
        if not (along and "takes_behind" in type(module).__dict__ and module.takes_behind()):
            return join(x, module(*args), post, m, following, scale)
        behind = ResidualBehind(x, post.weight, m, None if following is None else following.weight, scale, eps)
        y = module(*args, behind=behind)
        return behind.take(y) or join(x, y, post, m, following, scale)

    def single(module, args, state, post, m, following, scale=1.0):
        """(x, h) behind a sublayer of one row, or what the next one takes in front of itself."""
        front = isinstance(state, ResidualFront)
        if front and "takes_front" in type(module).__dict__ and module.takes_front():
            y = module(state.y.reshape(shape), *args, front=state)
            x = state.joined()[0]
        else:
            x, h = state.joined() if front else state
            y = module(h.reshape(shape), *args)
        return ResidualFront.of(x, y, post.weight, m, None if following is None else following.weight, scale, eps) or join(x, y, post, m, following, scale)

    state = x, h
    for i, layer in enumerate(layers):
        last, m = i + 1 == len(layers), layer.branch_scale
        following = (final_norm, final_scale) if last else (layers[i + 1].pre_mixer_norm,)
        behind_mixer = following if layer.mlp is None else (layer.pre_mlp_norm,)
        if ahead:
            state = single(layer.mixer, (cache, cache_position), state, layer.post_mixer_norm, m, *behind_mixer)
            if layer.mlp is not None:
                state = single(layer.mlp, (), state, layer.post_mlp_norm, m, *following)
            continue
        x, h = sublayer(layer.mixer, (h, cache, cache_position), x, layer.post_mixer_norm, m, *behind_mixer)
        if layer.mlp is not None:
            x, h = sublayer(layer.mlp, (h,), x, layer.post_mlp_norm, m, *following)
        h = h.reshape(shape)
        if collect is not None:
            collect.append(x.clone())
    return (state.joined() if isinstance(state, ResidualFront) else state)[1].reshape(shape) if ahead else h
