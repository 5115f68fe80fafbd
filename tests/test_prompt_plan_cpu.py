"""Where the last few tokens of a prompt are a launch of their own: products that were measured both ways and differ by 5 % or more (256 CUs)."""
import pytest

from tests.prompt_util import prompt_plan

# us in one launch / two
TWO = [("bf16", "gateup", 14336, 4096, 520, 165, 146), ("bf16", "gateup", 14336, 2880, 520, 120, 110), ("bf16", "gateup", 14336, 4160, 1032, 271, 237),
       ("fp16", "gateup", 8192, 8192, 2176, 533, 461), ("int8", "gateup", 14336, 4096, 520, 180, 130), ("int8", "gateup", 14336, 2880, 1032, 213, 187),
       ("int8_group", "gateup", 8192, 5120, 1124, 233, 199), ("bf16", "linear", 4096, 14400, 4104, 449, 361), ("bf16", "linear", 4096, 4096, 4104, 153, 121),
       ("int8", "linear", 4096, 4160, 4104, 160, 124), ("fp16", "linear", 5120, 14336, 3089, 451, 357), ("bf16", "linear", 8192, 4096, 2120, 140, 123), ("bf16", "linear", 4096, 14336, 2056, 237, 219)]
ONE = [("int8", "gateup", 2048, 8256, 529, 69, 123), ("int8", "gateup", 2560, 11008, 2305, 238, 452), ("int8", "gateup", 1024, 11008, 1089, 88, 160),
       ("int8", "gateup", 4096, 8256, 562, 107, 140), ("int8_group", "gateup", 2560, 14336, 868, 198, 254), ("int8_group", "gateup", 8192, 5120, 640, 125, 141),
       ("bf16", "gateup", 8192, 8256, 552, 169, 178), ("bf16", "gateup", 8192, 11008, 1664, 460, 494), ("bf16", "gateup", 4096, 1408, 1088, 35, 40),
       ("fp16", "linear", 2048, 5120, 5889, 108, 182), ("bf16", "linear", 4096, 14400, 2088, 223, 247), ("int8", "linear", 1536, 8256, 5160, 132, 154)]


@pytest.mark.parametrize("weights,form,n,k,tokens,one,two", TWO + ONE)
def test_last_tokens_are_a_launch_of_their_own_where_it_is_faster(weights, form, n, k, tokens, one, two):
    rest = prompt_plan(weights, form, n, k, tokens)[0]
    assert rest == (tokens % 256 if two < one else 0)


def test_never():
    for weights, form, n, k, tokens in [("bf16", "gateup", 14336, 4096, 512), ("bf16", "gateup", 14336, 4096, 512 + 129), ("bf16", "gateup", 14336, 4096, 511),
                                        ("bf16", "linear", 4096, 4096, 2047), ("bf16", "gateup", 14336, 4096 + 8, 520), ("int8", "gateup", 14336, 4096 + 16, 520)]:
        assert prompt_plan(weights, form, n, k, tokens)[0] == 0


@pytest.mark.parametrize("weights,form,n,k,tokens,tile", [
    ("bf16", "gateup", 1024, 1024, 5392, 4), ("bf16", "gateup", 2304, 11008, 388, 9), ("int8_group", "linear", 2304, 14336, 772, 9), ("int8", "linear", 4104, 14336, 2700, 4),
    ("fp16", "linear", 3584, 14336, 1032, 7), ("fp16", "linear", 5120, 14336, 2198, 4), ("int8", "linear", 5120, 1024, 3199, 8)])
def test_rounds_are_counted_by_the_fullest_xcd(weights, form, n, k, tokens, tile):
    """Row tiles that do not come out even over the eight XCDs: products that took 1.4 to 1.6 times as long on another tile."""
    assert prompt_plan(weights, form, n, k, tokens)[1] == tile
