"""What the built-in rules do with a prompt product, for tests that are about one route and have to take it."""
import ctypes

from muillm_amd import _lib

WEIGHTS = {"fp16": (0, 0), "bf16": (1, 0), "int8": (0, 1), "int8_group": (0, 2), "int8_bf16": (1, 1)}  # dtype code, weight format


def prompt_plan(weights: str, form: str, n: int, k: int, tokens: int, shift: int = 7, scratch: bool = True):
    """(tokens in a launch of their own, tile of the others, what becomes of its last round: 0 as it is, 1 halves, 2 quarters); form "gateup" or "linear"."""
    (dtype, fmt), out = WEIGHTS[weights], [ctypes.c_int() for _ in range(3)]
    _lib.check(_lib.load().mui_probe_prefill_plan(dtype, fmt, int(form == "gateup"), n, k, tokens, shift if fmt == 2 else 0, int(scratch),
                                                  *[ctypes.byref(x) for x in out]), "mui_probe_prefill_plan")
    return tuple(x.value for x in out)
