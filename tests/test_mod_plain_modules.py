"""When a MoD wrapper's inner modules may be run without calling them: only if
nothing hooks into the call."""
from __future__ import annotations

import pytest
import torch.nn as nn
from torch.nn.modules import module as nn_module


@pytest.mark.parametrize("kind", ["own", "pre", "backward", "global", "global_pre", "instance"])
def test_hooked_modules_are_called(kind):
    from hydra_amd.routing.mixture_of_depths import _plain

    a, b = nn.Linear(4, 1), nn.Linear(4, 1)
    assert _plain(a, b)
    register = {"own": b.register_forward_hook, "pre": b.register_forward_pre_hook,
                "backward": b.register_full_backward_hook, "global": nn_module.register_module_forward_hook,
                "global_pre": nn_module.register_module_forward_pre_hook}.get(kind)
    if register is None:
        b.forward = lambda x: x
        assert not _plain(a, b)
        return
    handle = register(lambda *args: None)
    try:
        assert not _plain(a, b)
    finally:
        handle.remove()
    assert _plain(a, b)
