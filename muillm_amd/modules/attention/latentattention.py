"""MuiLatentAttention: attention whose keys and values are linear maps of one cached latent row per token
plus a rotated key part shared by all heads, with queries through a latent of their own and a sliding
window. Kernels: csrc/latent_attention.hip, csrc/latent_step.hip.

A layer may read another layer's cached rows (kv_source) instead of keeping its own: it then has no key /
value down projection, only its own up projections, queries and window."""
from dataclasses import dataclass
from typing import Optional

import torch
import torch.nn as nn

from ... import _lib, hybrid_ops, muillm_ext
from ...engineconfig import MuiEngineConfig
from ..kvcache.hybridcache import MuiHybridCache, MuiLatentState
from ..linear import MuiLinear, _MuiLinear
from ..module import MuiModule, heard
from ..multilinear import MuiMultiLinear


@dataclass
class MuiLatentAttentionConfig:
    heads: int
    dim: int        # unrotated query / key dimensions per head
    rot_dim: int    # rotated ones
    vdim: int
    q_rank: int
    kv_rank: int
    scale: float
    rot_base: float
    window: int = 0            # keys a query sees, itself included (0: all)
    kv_source: Optional[int] = None  # layer whose latent rows this one reads

    def __post_init__(self):
        if self.rot_dim % 2:
            raise ValueError("rot_dim must be even")


class MuiLatentAttention(MuiModule):
    takes_real_rows = True

    def takes_behind(self) -> bool:
        return type(self.out_proj) is MuiLinear and not heard(self, self.out_proj)

    def __init__(self, engine_config: MuiEngineConfig, hidden: int, config: MuiLatentAttentionConfig, layer_idx: int,
                 eps: float, device=None, dtype=None):
        super().__init__(engine_config=engine_config)
        c = self.config = config
        self.layer_idx, self.eps = layer_idx, eps
        self.own_rows = c.kv_source is None
        kw = dict(device=device, dtype=dtype)
        outs = [c.q_rank] + ([c.kv_rank, c.rot_dim] if self.own_rows else [])
        self.down = MuiMultiLinear(engine_config, hidden, outs, bias=False, **kw)
        self.q_norm = nn.Parameter(torch.ones(c.q_rank, **kw), requires_grad=False)
        self.kv_norm = nn.Parameter(torch.ones(c.kv_rank, **kw), requires_grad=False) if self.own_rows else None
        self.up_q = MuiLinear(engine_config, c.q_rank, c.heads * (c.dim + c.rot_dim), bias=False, **kw)
        # rows of the key map, then rows of the value map
        self.up_kv = MuiLinear(engine_config, c.kv_rank, c.heads * (c.dim + c.vdim), bias=False, **kw)
        self.out_proj = MuiLinear(engine_config, c.heads * c.vdim, hidden, bias=False, **kw)
        half = torch.arange(c.rot_dim // 2, dtype=torch.float64)
        self.register_buffer("inv_freq", (float(c.rot_base) ** (-2.0 * half / c.rot_dim)).to(device), persistent=False)

    def new_state(self, batch: int, capacity: int, device, dtype) -> Optional[MuiLatentState]:
        if not self.own_rows:
            return None
        return MuiLatentState(batch, capacity, self.config.kv_rank, self.config.rot_dim, device, dtype)

    def forward(self, h: torch.Tensor, cache: MuiHybridCache, cache_position: torch.Tensor, behind=None) -> torch.Tensor:
        """h [B, T, hidden] (normed) -> [B, T, hidden]; the tokens' rows go to slots cache_position."""
        c = self.config
        down = cache.spread(self.down.linear(h))
        b, t = down.shape[0], down.shape[1]
        state: MuiLatentState = cache.layers[self.layer_idx if self.own_rows else c.kv_source]
        w = self.up_kv.weight
        w_uk, w_uv = w[:c.heads * c.dim], w[c.heads * c.dim:]
        step = t == 1 and self._one_launch_is_faster(b, state.c.shape[1], down.dtype) and hybrid_ops.latent_step_serves(down, b, c.heads, c.dim, c.rot_dim, c.vdim, w_uk, w_uv, state.c, state.r, c.window)
        if step and b == 1 and self._norm_goes_with_query(down):
            # the query's norm goes with its projection, the token's rows with the attention
            up = self.up_q.cpp_module
            normed = muillm_ext.MuiLinearModuleHandle(up.engine, up.weights, self.q_norm, self.eps, up.mul_bias, up.add_bias)
            q = _MuiLinear.apply(normed, down[..., :c.q_rank], None)
            kv = down[..., c.q_rank:] if self.own_rows else None
            o = hybrid_ops.latent_step(q, kv, self.kv_norm, self.eps, self.inv_freq, w_uk, w_uv, state.c, state.r, cache_position, cache.row_start, c.heads, c.dim, c.vdim,
                                       c.scale, c.window)
            return self._project(cache.take(o), behind)
        q_latent, cos_sin = hybrid_ops.latent_prepare(down, self.q_norm, self.kv_norm, self.eps, self.inv_freq,
                                                      cache_position, cache.row_start, state.c, state.r)
        q = self.up_q(q_latent)
        route = hybrid_ops.latent_route(h.dtype, t, c.heads, c.dim, c.rot_dim, c.vdim, c.kv_rank)
        if step:
            o = hybrid_ops.latent_step(q, None, None, self.eps, self.inv_freq, w_uk, w_uv, state.c, state.r, cache_position, cache.row_start, c.heads, c.dim, c.vdim, c.scale, c.window)
        elif route == _lib.MUI_LATENT_PREFILL:
            # keys and values of everything the tokens can see, once per call
            q_first = cache.get_seq_length()
            kv_first = max(0, q_first - c.window + 1) if c.window else 0
            kv = self.up_kv(state.c[:b, kv_first:q_first + t].contiguous())
            o = hybrid_ops.latent_prefill_attention(q, cos_sin, kv, kv_first, state.r, cache.row_start, q_first, c.heads, c.dim,
                                                    c.vdim, c.scale, c.window)
        else:
            o = hybrid_ops.latent_attention(q, cos_sin, w_uk, w_uv, state.c, state.r,
                                            cache_position, cache.row_start, c.heads, c.dim, c.vdim, c.scale, c.window, route)
        return self._project(cache.take(o), behind)

    def _one_launch_is_faster(self, batch: int, capacity: int, dtype: torch.dtype) -> bool:
        """Whether single tokens over caches of so many visible rows take latent_step, whose workgroups have all keys of a head one after the other (28 ns each); the launches apart take as
        long for few as for many, and longer where the matrices are (rank). A single fp16 row gains least: in bf16 its preparation goes along, several take longer apart. us from the down
        projection's output to the attention's, apart / one launch, caches full, 1 row of 16 heads of 128 in bf16: rank 64, 128 / 192 / 256 keys 15.7 / 14.8, 15.6 / 16.3, 16.1 / 18.5; 256,
        192 / 256 keys 17.1 / 16.6, 17.1 / 18.7; 512, 256 keys 19.7 / 20.0; in fp16 rank 64, 64 / 128 / 192 keys 15.9 / 13.9, 16.5 / 16.2, 16.5 / 17.7; 512, 192 / 256 keys 20.4 / 19.4,
        20.4 / 21.0; 16 rows of 4 heads without the projection: rank 128, 128 / 256 keys 15.6 / 14.0, 15.6 / 17.2; 512, 256 keys 18.9 / 17.3."""
        c = self.config
        span = min(c.window, capacity) if c.window > 0 else capacity
        return span <= (168 if batch > 1 or dtype == torch.bfloat16 else 104) + 3 * c.kv_rank // 16

    def _norm_goes_with_query(self, down: torch.Tensor) -> bool:
        """Whether the projection's own norm stands in for latent_prepare's. In fp16 it does not: it multiplies latent and gain in 16 bits in front of the scale, where a product beyond
        65504 or below 6e-5 does not fit, and latent_prepare does so in 32 bits behind it. Nor are gains and rows taken that cannot be read 16 bytes at a time."""
        return (down.dtype == torch.bfloat16 and self.config.q_rank % 8 == 0 and type(self.up_q) is MuiLinear and self.up_q.takes_front()
                and all(x is None or x.data_ptr() % 16 == 0 for x in (down, self.q_norm, self.kv_norm)))

    def _project(self, o: torch.Tensor, behind) -> torch.Tensor:
        return self.out_proj(o) if behind is None else self.out_proj(o, behind=behind)
