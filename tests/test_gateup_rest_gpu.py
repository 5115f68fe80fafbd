"""Prompts that end a little beyond whole 256-token tiles, whose last tokens are a launch of their own: one of them and as many as there can be, taken by the kernel that streams
the weights and by tiles, with outputs that come out even and not, against products in 32 bits, and the same in one launch."""
import pytest
import torch

from muillm_amd import _lib

from tests.prompt_util import prompt_plan, prompt_product

pytestmark = pytest.mark.gpu
REL = {"bf16": 2 ** -7, "fp16": 2 ** -10, "int8": 2 ** -10, "int8_group": 2 ** -10}  # as a share of the largest output: four times one rounding to 16 bits
GATEUP = [(14340, 2048, 513), (8192, 1024, 1025), (8192, 1024, 1088), (14340, 1024, 577), (14340, 1024, 640), (12288, 1024, 1313)]
LINEAR = [(8192, 2048, 2056), (8190, 4096, 2056), (8192, 4096, 2057)]


@pytest.mark.parametrize("weights,form,n,k,tokens", [(w, "gateup", *s) for w in REL for s in GATEUP] +
                         [(w, "linear", *s) for w in REL for s in LINEAR if w != "int8_group"])  # (groups of that many tokens are dequantised)
def test_two_launches(weights, form, n, k, tokens):
    assert prompt_plan(weights, form, n, k, tokens)[0] == tokens % 256
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
