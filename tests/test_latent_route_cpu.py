"""Routes of latent attention by the widths that its kernels hold (no GPU needed)."""
import pytest

import torch

from muillm_amd import _lib
from muillm_amd.engineconfig import MuiEngineConfig
from muillm_amd.modules.attention.latentattention import MuiLatentAttention, MuiLatentAttentionConfig


@pytest.mark.parametrize("kv_rank,rot,route", [(512, 64, _lib.MUI_LATENT_DECODE), (512, 8, _lib.MUI_LATENT_DECODE), (504, 72, _lib.MUI_LATENT_DECODE),
                                               (520, 8, _lib.MUI_LATENT_PLAIN), (568, 8, _lib.MUI_LATENT_PLAIN), (576, 0, _lib.MUI_LATENT_PLAIN),
                                               (512, 72, _lib.MUI_LATENT_PLAIN)])
def test_decode_route(kv_rank, rot, route):
    """The decode kernel keeps up to 512 latent columns of an output."""
    lib = _lib.load()
    for dtype in (_lib.MUI_DTYPE_F16, _lib.MUI_DTYPE_BF16):
        assert lib.mui_latent_attention_route(dtype, 1, 16, 128, rot, 128, kv_rank) == route
        assert lib.mui_latent_attention_route(dtype, 17, 16, 128, rot, 128, kv_rank) == _lib.MUI_LATENT_PREFILL


@pytest.mark.parametrize("dtype,batch,rank,keys,apart,one", [
    (torch.bfloat16, 1, 64, 128, 15.7, 14.8), (torch.bfloat16, 1, 64, 256, 16.1, 18.5), (torch.bfloat16, 1, 256, 192, 17.1, 16.6), (torch.bfloat16, 1, 256, 256, 17.1, 18.7),
    (torch.bfloat16, 1, 512, 256, 22.0, 20.8), (torch.float16, 1, 64, 64, 15.9, 13.9), (torch.float16, 1, 64, 192, 16.5, 17.7), (torch.float16, 1, 512, 192, 20.4, 19.4),
    (torch.float16, 1, 512, 256, 20.4, 21.0), (torch.float16, 16, 128, 128, 15.6, 14.0), (torch.float16, 16, 128, 256, 15.6, 17.2), (torch.bfloat16, 8, 512, 256, 24.1, 20.1)])
@pytest.mark.parametrize("window", [False, True])
def test_one_launch_for_single_tokens_where_it_is_faster(dtype, batch, rank, keys, apart, one, window):
    """Caches that hold so many keys, or layers that see no more, as measured both ways."""
    c = MuiLatentAttentionConfig(heads=1, dim=16, rot_dim=16, vdim=16, q_rank=16, kv_rank=rank, scale=0.25, rot_base=1e4, window=keys if window else 0)
    layer = MuiLatentAttention(MuiEngineConfig(), 16, c, 0, 1e-5)
    assert layer._one_launch_is_faster(batch, 4096 if window else keys, dtype) == (one < apart)
