"""Routes of latent attention by the widths that its kernels hold (no GPU needed)."""
import pytest

from muillm_amd import _lib


@pytest.mark.parametrize("kv_rank,rot,route", [(512, 64, _lib.MUI_LATENT_DECODE), (512, 8, _lib.MUI_LATENT_DECODE), (504, 72, _lib.MUI_LATENT_DECODE),
                                               (520, 8, _lib.MUI_LATENT_PLAIN), (568, 8, _lib.MUI_LATENT_PLAIN), (576, 0, _lib.MUI_LATENT_PLAIN),
                                               (512, 72, _lib.MUI_LATENT_PLAIN)])
def test_decode_route(kv_rank, rot, route):
    """The decode kernel keeps up to 512 latent columns of an output."""
    lib = _lib.load()
    for dtype in (_lib.MUI_DTYPE_F16, _lib.MUI_DTYPE_BF16):
        assert lib.mui_latent_attention_route(dtype, 1, 16, 128, rot, 128, kv_rank) == route
        assert lib.mui_latent_attention_route(dtype, 17, 16, 128, rot, 128, kv_rank) == _lib.MUI_LATENT_PREFILL
