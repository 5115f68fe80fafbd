"""Where linears of more than 128 tokens share K between workgroups: products that were measured both ways (256 CUs)."""
import pytest

from muillm_amd import _lib
from tests.prompt_util import prompt_shares


@pytest.mark.parametrize("weights,n,k,tokens,whole,shared", [
    ("bf16", 4096, 14336, 200, 61, 49), ("fp16", 4096, 14336, 333, 93, 62), ("bf16", 4096, 14336, 768, 127, 88), ("bf16", 4096, 14336, 1280, 173, 128),
    ("bf16", 2048, 8192, 768, 56, 40), ("bf16", 6144, 4096, 333, 42, 38), ("bf16", 6144, 4096, 2048, 84, 116),
    ("bf16", 4096, 4096, 2048, 63, 75), ("bf16", 2048, 2048, 1280, 25, 27), ("bf16", 4096, 14336, 4096, 348, 400)])
def test_k_is_shared_where_it_is_faster(weights, n, k, tokens, whole, shared):
    assert (prompt_shares(weights, n, k, tokens)[1] > 1) == (shared < whole)


@pytest.mark.parametrize("weights,n,k,tokens,whole,shared", [
    ("bf16", 2112, 4096, 217, 23.3, 24.3), ("bf16", 2112, 4096, 241, 23.4, 25.0), ("bf16", 1024, 4096, 539, 24.1, 24.6), ("bf16", 4096, 4096, 129, 24.6, 25.7),
    ("int8", 2048, 3072, 322, 24.1, 26.2), ("int8_group", 1024, 4096, 344, 23.2, 24.9), ("int8", 1024, 4096, 160, 21.0, 18.5)])
def test_shares_of_eight_k_steps_and_fewer(weights, n, k, tokens, whole, shared):
    assert (prompt_shares(weights, n, k, tokens)[1] > 1) == (shared < whole)


def test_never():
    for weights, n, k, tokens in [("bf16", 4096, 14336, 128), ("bf16", 4098, 14336, 333), ("bf16", 4096, 14336 + 8, 333), ("bf16", 4096, 640, 333), ("bf16", 1 << 20, 14336, 333)]:
        assert prompt_shares(weights, n, k, tokens)[1] == 1


def test_groups_that_do_not_divide_k():
    """The last group's part would have no (scale, smallest value) pair."""
    assert prompt_shares("int8_group", 2048, 8320, 333, shift=7)[1] > 1  # 65 groups
    assert prompt_shares("int8_group", 2048, 8320, 333, shift=8)[1] == 1  # 32 and a half
    for shift in (-1, 31):
        with pytest.raises(_lib.MuiLibraryError):
            prompt_shares("int8_group", 2048, 8320, 333, shift=shift)
