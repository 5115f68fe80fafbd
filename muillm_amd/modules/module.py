"""MuiModule -- muillm/modules/module.py:6-32: base class of every replacement layer with
the finalize_init()/finalize_deinit() protocol run by init_engine."""
import torch.nn as nn

from ..engineconfig import MuiEngineConfig


def heard(*modules: nn.Module) -> bool:
    """Whether a hook listens to calls of one of them, or a forward of its own stands in for its class's: a hook may change what comes out in ways that cannot be seen from
    outside (through .data, or by a kernel of its own), and another forward knows the documented arguments only."""
    every = nn.modules.module
    if every._global_forward_hooks or every._global_forward_pre_hooks:
        return True
    return any(m.__dict__["_forward_hooks"] or m.__dict__["_forward_pre_hooks"] or "forward" in m.__dict__ for m in modules)


class MuiModule(nn.Module):
    def __init__(self, engine_config: MuiEngineConfig = None, **kargs) -> None:
        if engine_config is None:
            # a cooperative super().__init__() from a class with several bases: the real
            # initialisation call with an engine config follows
            return None
        nn.Module.__init__(self, **kargs)
        self.engine_config = engine_config

    def __del__(self):
        try:
            self.finalize_deinit()
        except Exception:
            pass

    def finalize_init(self) -> None:
        """Called post-order once all layers are replaced and on their device."""

    def finalize_deinit(self) -> None:
        """Called on destruction."""
