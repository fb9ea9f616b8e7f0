"""GPU parity of the attention backward over the forms its kernels divide
between: head dims at and off the tile sizes, sequence lengths around the
32- and 64-row tiles, one key/value head or several, the two key masks.

Reference: fp64 autograd through the oracle's masked softmax on the same
rounded inputs.  Error measure: 2-norm of the difference over 2-norm of the
gradient.  What a correct kernel shows: half an ulp per output (u / 2 each,
u = 2^-8 for bf16, 2^-11 for fp16), the same again through D = rowsum(dO * O)
from the rounded O and through the forward's rounded output; four half ulps,
2 u, bound their sum.  For fp32 the sums' own rounding counts: products over
S keys or queries with unit roundoff 2^-24, at most sqrt(S) x a few of it at
the tested S <= 333, 2^-17 with room."""
from __future__ import annotations

import pytest
import torch

from oracle import ccgqa as occ

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10, torch.float32: 2.0 ** -17}


def _masks(B, S, form):
    """[B, S] 0/1 key masks: right-padded lengths, left-padded (rows without
    a visible key under causality), scattered, or nothing masked."""
    at = torch.arange(S)
    cut = torch.tensor([[max(1, S - 1 - 45 * b)] for b in range(B)])
    if form == "right":
        return (at < cut).long()
    if form == "left":
        return (at >= S - cut).long()
    if form == "holes":
        return ((at + torch.arange(B)[:, None]) % 3 != 0).long()
    return torch.ones(B, S, dtype=torch.long)


def _reference(q, k, v, go, causal, mask, mode):
    q, k, v = (t.double().requires_grad_() for t in (q, k, v))
    if mode == "reference":  # query s sees key t > s, or a padded key; a row with neither gives 0
        B, H, S, hd = q.shape
        g = H // k.shape[1]
        vis = torch.ones(S, S, dtype=torch.bool).triu(1) | (mask == 0).view(B, 1, 1, S)
        sc = (q @ k.repeat_interleave(g, 1).transpose(-1, -2)) * hd ** -0.5
        p = torch.softmax(sc.masked_fill(~vis, -1e30), -1) * vis
        out = p @ v.repeat_interleave(g, 1)
    else:
        out = occ.attention_key_padding(q, k, v, causal=causal, mask=mask)
    out.backward(go.double())
    return q.grad, k.grad, v.grad


def _case(cuda, B, Hq, Hkv, S, hd, dtype, causal, form, mode):
    from hydra_amd.attention.backends.ccgqa.ops import (MASK_KEY_PADDING, MASK_NONE, MASK_REFERENCE_SDPA,
                                                        attention_backward, attention_forward)

    g = torch.Generator().manual_seed(S * 131 + hd)
    q, go = (torch.randn(B, Hq, S, hd, generator=g).to(dtype) for _ in range(2))
    k, v = (torch.randn(B, Hkv, S, hd, generator=g).to(dtype) for _ in range(2))
    mask = None if form is None else _masks(B, S, form)
    mm = {None: MASK_NONE, "key_padding": MASK_KEY_PADDING, "reference": MASK_REFERENCE_SDPA}[mode]
    qd, kd, vd, god = (t.to(cuda) for t in (q, k, v, go))
    md = None if mask is None else mask.to(cuda)
    out, lse = attention_forward(qd, kd, vd, causal=causal, key_mask=md, mask_mode=mm, want_lse=True)
    got = attention_backward(qd, kd, vd, out, lse, god, causal=causal, key_mask=md, mask_mode=mm)
    for name, a, r in zip(("dq", "dk", "dv"), got, _reference(q, k, v, go, causal, mask, mode)):
        a = a.double().cpu()
        assert torch.isfinite(a).all(), name
        err = float((a - r).norm() / r.norm())
        assert err < TOL[dtype], f"{name}: {err:.3g}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("shape", [(2, 4, 2, 2, 16), (1, 3, 1, 31, 16), (2, 7, 1, 65, 16), (1, 4, 4, 129, 16),
                                   (1, 2, 1, 333, 16), (1, 2, 1, 64, 32), (1, 6, 2, 97, 64), (1, 2, 1, 161, 128),
                                   (2, 2, 2, 40, 24), (1, 2, 1, 33, 80)])
def test_backward_forms(cuda, shape, causal, dtype):
    _case(cuda, *shape, dtype, causal, None, None)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("mode,causal", [("key_padding", True), ("key_padding", False), ("reference", True)])
@pytest.mark.parametrize("form", ["right", "left", "holes", "none"])
@pytest.mark.parametrize("shape", [(3, 4, 1, 200, 64), (2, 2, 2, 65, 16), (2, 3, 1, 129, 32), (2, 2, 1, 97, 128)])
def test_backward_key_mask_forms(cuda, shape, form, mode, causal, dtype):
    if mode == "key_padding" and form == "left" and not causal:
        form = "right"  # without causality every row sees the same keys
    _case(cuda, *shape, dtype, causal, form, mode)
