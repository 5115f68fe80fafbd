"""The tokens of a left-padded batch of prompts that are no padding. What works on one token at a time -- linears, norms, experts -- need not
see the others: their rows are laid out one after the other, and only what looks at a token's neighbours (attention, recurrences) gets [batch, tokens] with zeros for the padding."""
from typing import NamedTuple, Optional

import torch

from .. import muillm_ext
from .module import heard


# Leaving padding out costs a layer two launches and two passes over its projections (6 to 10 us), and where the modules are called one by one 33 us of host time. Linears of up to
# 128 tokens are bound by their weights and beyond work on tiles of 256, so they take as long for fewer tokens unless tiles fall away; experts deal their tokens out and take less for
# every one that is missing. In operations per layer (24 hidden^2 for a token; 0.9e9 a us): the padding's, those of the tiles that fall away, and, per token and value of its width, what the
# passes cost where no tile pays for them. us, with it / without, prompts alone on eight layers (tokens -> real ones):
#   Llama, one call: 2048 wide 319 -> 200 1656 / 1546, 640 -> 463 2014 / 1806, 900 -> 657 2193 / 2136, 928 -> 668 2089 / 2046, 4096 wide 192 -> 118 2379 / 1879, 320 -> 214 2979 / 2541;
#     2050 -> 2020 7763 / 7316, 4100 -> 4066 13170 / 12880; no tile less: 2048 wide 256 -> 176 1473 / 1498, 450 -> 310 1653 / 1677, 4096 wide 256 -> 176 2461 / 2442, int8 2523 / 2582, 480 -> 342 3214 / 3174
#   Zufadra: two tiles less 2048 wide 1200 -> 763 2938 / 2588, one 4096 wide 192 -> 118 2572 / 2206, 319 -> 200 3277 / 2913, 260 -> 173 3059 / 2658, 2048 wide 319 -> 200 1911 / 2039,
#     900 -> 581 2336 / 2414, 1000 -> 570 2452 / 2466; none 4096 wide 256 -> 176 2668 / 2727, 400 -> 307 3211 / 3262
#   Salepel: 2048 wide 256 -> 176 3335 / 3319, 319 -> 200 3636 / 3433, 450 -> 310 3685 / 3514, 1200 -> 763 4536 / 4132, 4096 wide 192 -> 118 6223 / 5994, 400 -> 307 7095 / 6614; few
#     of many: 2048 wide 2056 -> 1926 5399 / 5766, 4096 wide 1026 -> 996 8524 / 8654, 4100 -> 4066 19464 / 20024
class Worth(NamedTuple):
    padding: float
    tiles: float = 0.0
    passes: float = 0.0


MOST_WEIGHT_BOUND, TOKEN_TILE = 128, 256


def _tiles(tokens: int) -> float:
    return 0.5 if tokens <= MOST_WEIGHT_BOUND else -(-tokens // TOKEN_TILE)


def worth_it(worth: Worth, hidden: int, tokens: int, padding: int) -> bool:
    per_token = 24.0 * hidden ** 2
    return (tokens > MOST_WEIGHT_BOUND and padding * per_token >= worth.padding + worth.passes * tokens * hidden
            and (_tiles(tokens) - _tiles(tokens - padding)) * TOKEN_TILE * per_token >= worth.tiles)


def on_device(x: torch.Tensor, device) -> torch.Tensor:
    """A small host tensor on its way to the device: nobody waits for it."""
    return x.pin_memory().to(device, non_blocking=True) if torch.device(device).type == "cuda" else x.to(device)


class RealRows:
    def __init__(self, mask: torch.Tensor, device):
        """mask: bool [B, T] in host memory, true for real tokens; every row ends with one."""
        self.mask, self.device = mask, device
        self.batch, self.tokens = mask.shape
        self.n = int(mask.sum())

    def __getattr__(self, name: str) -> torch.Tensor:
        """rows, slots, last: places in [B * T] of the real rows; every token's place among those, or -1; the same of every last token. Laid out when first asked for:
        a model that takes the whole prompt after all need not wait."""
        if name not in ("rows", "slots", "last"):
            raise AttributeError(name)
        flat = self.mask.reshape(-1)
        rows = flat.nonzero().reshape(-1)
        slots = (flat.cumsum(0) - 1).masked_fill_(~flat, -1)
        both = on_device(torch.cat([rows, slots, slots.view(self.mask.shape)[:, -1]]), self.device)
        self.rows, self.slots, self.last = both.split([self.n, flat.numel(), self.batch])
        return self.__dict__[name]

    @staticmethod
    def of(lm, mask: torch.Tensor, device) -> Optional["RealRows"]:
        """For a padded prompt of a causal LM whose forward takes `real`; None for any other, where it is not worth it (`padding_worth` of the model's class) and where
        somebody listens to what it is given."""
        model = getattr(lm, "model", None)
        if torch.device(device).type != "cuda" or mask.dim() != 2 or not all("takes_real_rows" in type(m).__dict__ for m in (lm, model)) or heard(lm, model):
            return None
        padding = mask.numel() - int(mask.sum())
        if not padding or not worth_it(lm.padding_worth, lm.config.hidden_size, mask.numel(), padding) or not bool(mask[:, -1].all()):
            return None
        return RealRows(mask, device)

    def take(self, x: torch.Tensor) -> torch.Tensor:
        """[B, T, w] -> [1, real rows, w]"""
        return muillm_ext.take_rows(x.reshape(-1, x.shape[-1]), self.rows)[None]

    def spread(self, x: torch.Tensor) -> torch.Tensor:
        """[1, real rows, w] -> [B, T, w], zeros where the padding is"""
        return muillm_ext.take_rows(x.reshape(-1, x.shape[-1]), self.slots).view(self.batch, self.tokens, -1)

    def last_of(self, x: torch.Tensor) -> torch.Tensor:
        """[1, real rows, w] -> [B, 1, w]: every batch row's last token"""
        return muillm_ext.take_rows(x.reshape(-1, x.shape[-1]), self.last)[:, None]
