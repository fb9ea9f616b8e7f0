"""When a MoD wrapper's inner modules may be run without calling them: only if
nothing hooks into the call."""
from __future__ import annotations

import pytest
import torch
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


def test_an_overridden_mlp_forward_is_called():
    """A wrapped SwiGLU MLP whose forward is another (by its class or on the
    instance) runs that forward, not the parts of the parent's."""
    from hydra_amd.layers import SwiGLUMLPFused
    from hydra_amd.model.framework.blocks import _mlp_residual
    from hydra_amd.routing.mixture_of_depths import MoDMLPWrapper

    class Doubling(SwiGLUMLPFused):
        def forward(self, x):
            return 2 * x

    on_instance = SwiGLUMLPFused(8, 16)
    on_instance.forward = lambda x: 2 * x
    h, y = torch.randn(2, 3, 8), torch.randn(2, 3, 8)
    for mlp in (Doubling(8, 16), on_instance):
        with torch.no_grad():
            assert torch.equal(_mlp_residual(MoDMLPWrapper(mlp, 8).eval(), h, y), h + 2 * y)


@pytest.mark.parametrize("wrapped", [False, True])
@pytest.mark.parametrize("how", ["class", "instance", "hook", "residual"])
def test_a_changed_mlp_is_used_as_it_is(how, wrapped):
    """Alone as under a wrapper, an MLP with another forward (by its class or
    on the instance) or with hooks is called; one whose class has its own
    forward_residual(h, x) gets the two arguments that it takes."""
    from hydra_amd.layers import SwiGLUMLPFused
    from hydra_amd.model.framework.blocks import _mlp_residual
    from hydra_amd.routing.mixture_of_depths import MoDMLPWrapper

    class Doubling(SwiGLUMLPFused):
        def forward(self, x):
            return 2 * x

    class Residual(Doubling):
        def forward_residual(self, h, x):
            return h + 2 * x

    mlp = {"class": Doubling, "residual": Residual}.get(how, SwiGLUMLPFused)(8, 16)
    if how == "instance":
        mlp.forward = lambda x: 2 * x
    elif how == "hook":  # the parent's forward needs a GPU: the hook must come before it
        def hook(module, args):
            raise KeyError("called")
        mlp.register_forward_pre_hook(hook)
    h, y = torch.randn(2, 3, 8), torch.randn(2, 3, 8)
    block = MoDMLPWrapper(mlp, 8).eval() if wrapped else mlp
    with torch.no_grad():
        if how == "hook":
            with pytest.raises(KeyError, match="called"):
                _mlp_residual(block, h, y)
        else:
            assert torch.equal(_mlp_residual(block, h, y), h + 2 * y)


def test_methods_of_their_own():
    from hydra_amd.routing.base import BaseRouter
    from hydra_amd.routing.mixture_of_depths import MoDRouter, _own

    class Noisy(MoDRouter):
        def _apply_jitter(self, logits):
            return logits + 1

    names = ("forward_logits", "_apply_jitter")
    router = MoDRouter(8)
    assert _own(router, BaseRouter, *names) and not _own(Noisy(8), BaseRouter, *names)
    router.forward_logits = lambda x: x[..., 0]
    assert not _own(router, BaseRouter, *names)


def test_tensors_under_a_transform_are_not_read_in_place():
    from hydra_amd.routing.mixture_of_depths import _plain_tensor

    seen = []
    look = lambda x: (seen.append(_plain_tensor(x)), x * 1)[1]
    x = torch.randn(3, 4)
    look(x)
    torch.func.vmap(look)(x)
    torch.func.jvp(look, (x,), (x,))
    with torch.autograd.forward_ad.dual_level():
        look(torch.autograd.forward_ad.make_dual(x, x))
    torch.jit.trace(look, (x,), check_trace=False)
    look(x)
    assert seen == [True, False, False, False, False, True]
