"""The choice of pairs per tile of the experts' products (no GPU needed)."""
import pytest

from muillm_amd import _lib


@pytest.mark.parametrize("tokens,top,experts,width,ff,want", [
    (400, 2, 8, 1024, 512, 128), (480, 2, 8, 4096, 1792, 128), (500, 8, 32, 1024, 512, 128),  # few tiles of gate and up: the chip stays idle
    (480, 4, 16, 1024, 2048, 128), (516, 4, 16, 1024, 2048, 256),  # few tiles of down, up to 128 pairs
    (428, 2, 8, 4096, 4096, 128), (432, 2, 8, 4096, 4096, 256), (430, 8, 32, 1024, 1024, 128), (432, 8, 32, 1024, 1024, 256),  # half as many as CUs
    (440, 4, 16, 4096, 1792, 256), (760, 8, 64, 4096, 1792, 128), (770, 8, 64, 4096, 1792, 256),  # the mean foretells an expert's pairs the better
    (1100, 6, 64, 2048, 1408, 128), (1120, 6, 64, 2048, 1408, 256), (410, 8, 32, 2048, 1024, 128), (420, 8, 32, 2048, 1024, 256),  # the more there are
    (714, 4, 24, 2048, 1408, 128), (720, 4, 24, 2048, 1408, 256),
    (700, 2, 8, 1024, 512, 256), (10, 8, 64, 4096, 1792, 16)])
def test_tile_pairs(tokens, top, experts, width, ff, want):
    assert _lib.load().mui_moe_tile_pairs(_lib.MUI_DTYPE_BF16, tokens, top, experts, width, ff) == want
