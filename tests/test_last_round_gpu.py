"""Products whose 256 x 256 tiles leave a last round of workgroups at most half full, which is a launch of its own of halves (1) or quarters (2) of the tiles: with outputs
and tokens that do not come out even, with bias and residual, and where the XCDs divide rows and tokens (4096 x 5120), against products in 32 bits, and the same in one launch."""
import pytest
import torch

from muillm_amd import _lib

from tests.prompt_util import prompt_plan, prompt_product

pytestmark = pytest.mark.gpu
REL = {"bf16": 2 ** -7, "fp16": 2 ** -10, "int8": 2 ** -10, "int8_group": 2 ** -10}  # as a share of the largest output: four times one rounding to 16 bits
CASES = [(w, "gateup", *s) for w in ("bf16", "fp16", "int8") for s in
         [(8192, 1024, 2500, 1), (14336, 1024, 3500, 2), (12290, 1024, 2500, 2), (4100, 512, 6144, 1), (14300, 512, 2500, 1)]] + \
        [("int8_group", "gateup", *s) for s in [(12290, 2048, 1281, 1), (8192, 1024, 1281, 1), (11008, 1024, 700, 2)]] + \
        [(w, "linear", *s) for w in ("bf16", "fp16", "int8") for s in
         [(14330, 2048, 3500, 2), (14336, 2048, 3585, 1), (4096, 5120, 4352, 2), (4100, 8192, 4352, 1)]] + \
        [("int8_group", "linear", *s) for s in [(12288, 4096, 1281, 2), (12290, 8192, 1281, 1)]]


@pytest.mark.parametrize("weights,form,n,k,tokens,last", CASES)
def test_last_round(weights, form, n, k, tokens, last):
    assert prompt_plan(weights, form, n, k, tokens) == (0, 4, last)
    call, ref = prompt_product(weights, form, n, k, tokens)
    lib, most = _lib.load(), float(ref.abs().max())
    y = call()
    assert lib.mui_tune_prefill(3200, 0) == 0
    try:
        one = call()
    finally:
        lib.mui_tune_prefill(0, 0)
    for out in (y, one):
        assert float((out.float() - ref).abs().max()) <= REL[weights] * most
