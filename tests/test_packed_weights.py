"""When packed weights are packed again, and what a copy of their module holds
(the values are compared, on any device; streams and graphs in
test_gpu_graph.py)."""
from __future__ import annotations

import copy
import pickle

import numpy as np
import pytest
import torch
import torch.nn as nn


def _asked(packs, *ws):
    """The packed values of ws (here: their negatives), and whether they were
    packed anew."""
    out = packs.get(ws, "order")
    anew = out is None
    if anew:
        out = packs.put(ws, "order", tuple(-w.detach() for w in ws))
    assert all(torch.equal(o, -w) for o, w in zip(out, ws))
    return anew


def test_packed_once_and_again_after_a_change():
    from hydra_amd.attention.backends.ccgqa.ops import PackedWeights

    packs = PackedWeights()
    a, b = nn.Parameter(torch.randn(4, 4)), nn.Parameter(torch.randn(4))
    assert _asked(packs, a, b) and not _asked(packs, a, b)
    with torch.no_grad():
        b.mul_(2)
    assert _asked(packs, a, b) and not _asked(packs, a, b)
    a.data = torch.randn(4, 4)
    assert _asked(packs, a, b) and not _asked(packs, a, b)


def test_another_tensor_at_the_same_address():
    """A replaced parameter may lie where an earlier one did, with the same
    version counter."""
    from hydra_amd.attention.backends.ccgqa.ops import PackedWeights

    packs = PackedWeights()
    memory, states = np.zeros(8, np.float32), set()
    for value in (1.0, 2.0):
        memory[:] = value
        w = nn.Parameter(torch.from_numpy(memory))
        states.add((w._version, w.data_ptr()))
        assert _asked(packs, w)
        del w
    assert len(states) == 1


def test_a_layout_that_is_the_weights_own_is_copied():
    from hydra_amd.attention.backends.ccgqa.ops import PackedWeights

    w = nn.Parameter(torch.randn(4))
    (t,) = PackedWeights().put((w,), None, (w.detach(),))
    assert t.data_ptr() != w.data_ptr() and torch.equal(t, w)


@pytest.mark.parametrize("how", [copy.deepcopy, lambda m: pickle.loads(pickle.dumps(m))])
def test_a_copied_module_packs_its_own(how):
    from hydra_amd.attention import CCGQAAttention

    m = CCGQAAttention(dim=512, n_heads=8, n_kv_heads=2, max_seq_len=16)
    convs = lambda n: (n.q_conv.conv1.weight, n.q_conv.conv2.weight, n.k_conv.conv1.weight, n.k_conv.conv2.weight)
    m._packed_conv_weights(convs(m), torch.float32)
    n = how(m)
    with torch.no_grad():
        n.q_conv.conv1.weight.fill_(3)
    assert (n._packed_conv_weights(convs(n), torch.float32)[0] == 3).all()
    assert not (m._packed_conv_weights(convs(m), torch.float32)[0] == 3).any()


def test_packing_in_one_launch_refuses_host_memory(monkeypatch):
    """The one-launch packing hands addresses to a kernel: weights that are not
    all on one GPU take the torch operations, after which the caller's own
    device check speaks."""
    from hydra_amd import _lib
    from hydra_amd.attention.backends.ccgqa.ops import ccgqa_prep, pack_conv_weight, pack_conv_weights_tiled

    monkeypatch.setattr(_lib, "call", lambda *a: pytest.fail("a launch on host memory"))
    ws = [torch.randn(*s, 3).to(torch.bfloat16) for s in ((128, 64), (128, 128), (64, 64), (64, 64))]
    for got, w in zip(pack_conv_weights_tiled(ws, torch.bfloat16, 2, 1, 64), ws):
        assert torch.equal(got, pack_conv_weight(w, torch.bfloat16, True))
    with pytest.raises(RuntimeError, match="GPU tensors only"):
        ccgqa_prep(torch.zeros(1, 8, 256, dtype=torch.bfloat16), 2, 1, 64, 1 | 64, *ws)


def test_a_captured_pack_of_another_form_is_left_alone():
    """Weights that moved, or are packed to another shape or type since a
    capture read them, get tensors of their own."""
    from hydra_amd.attention.backends.ccgqa.ops import PackedWeights

    packs = PackedWeights()
    w = nn.Parameter(torch.randn(4))
    (old,) = packs.put((w,), None, (-w.detach(),))
    p = packs._last[None]
    p.captured = True
    packs._captured.append((None, p))
    before = old.clone()
    for data in (torch.randn(6), torch.randn(4, dtype=torch.float64)):
        w.data = data
        assert packs.get((w,), None) is None
        (new,) = packs.put((w,), None, (-w.detach(),))
        assert torch.equal(new, -w) and new.dtype == w.dtype
        assert packs.get((w,), None)[0] is new
        assert torch.equal(old, before)
