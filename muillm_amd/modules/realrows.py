"""The tokens of a left-padded batch of prompts that are no padding. What works on one token at a time -- linears, norms, experts -- need not
see the others: their rows are laid out one after the other, and only what looks at a token's neighbours (attention, recurrences) gets [batch, tokens] with zeros for the padding."""
from typing import Optional

import torch

from .. import muillm_ext
from .module import heard


# Leaving padding out costs a layer two launches and two passes over its projections (6 to 10 us), and up to a few hundred tokens linears take as long for fewer:
# what is left out has to be beyond the 128 tokens whose linears are bound by their weights, and this many operations per layer (a layer has about 12 hidden^2
# weights that a token meets; 30 us at 0.9 PFLOP/s). Eight layers of width 2048, 319 tokens of which 213 are real: 3743 us with the padding, 3777 without; 2048 wide,
# eight prompts of up to 150 tokens (mLSTM, latent attention, experts) 12752 / 12309; 4096 wide (int8), 14 of up to 557 35357 / 29521.
MOST_WEIGHT_BOUND = 128
LEAST_OPERATIONS = 2.7e10


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
        """For a padded prompt of a causal LM whose forward takes `real`; None for any other, and where somebody listens to what it is given."""
        model = getattr(lm, "model", None)
        if torch.device(device).type != "cuda" or mask.dim() != 2 or not all("takes_real_rows" in type(m).__dict__ for m in (lm, model)) or heard(lm, model):
            return None
        padding = mask.numel() - int(mask.sum())
        if not padding or mask.numel() <= MOST_WEIGHT_BOUND or padding * 24.0 * lm.config.hidden_size ** 2 < LEAST_OPERATIONS or not bool(mask[:, -1].all()):
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
