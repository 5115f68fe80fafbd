"""The choice of pairs per tile of the experts' products (no GPU needed)."""
import pytest

from muillm_amd import _lib


@pytest.mark.parametrize("tokens,top,experts,width,ff,want", [
    (400, 2, 8, 1024, 512, 128), (480, 2, 8, 4096, 1792, 128), (440, 4, 16, 2048, 768, 128), (500, 8, 32, 1024, 512, 128),  # few tiles: the chip stays idle
    (440, 4, 16, 4096, 1792, 256), (440, 8, 32, 2048, 768, 256), (800, 8, 64, 4096, 1792, 256), (1100, 6, 64, 2048, 1408, 256),
    (700, 8, 64, 4096, 1792, 128), (700, 2, 8, 1024, 512, 256), (10, 8, 64, 4096, 1792, 16)])
def test_tile_pairs(tokens, top, experts, width, ff, want):
    assert _lib.load().mui_moe_tile_pairs(_lib.MUI_DTYPE_BF16, tokens, top, experts, width, ff) == want
