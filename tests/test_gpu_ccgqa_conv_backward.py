"""GPU parity of the bf16 prep backward in one call (hydra_ccgqa_prep_bwd_conv)
at the edges of its tiles: token counts around the 128-token conv tiles and
64-token weight-gradient steps, channel counts off and on the 64-channel
blocks, groups narrower than, as wide as and wider than a block, one and
several heads, and head_dim 24, which stays on the composed path.

Reference: fp64 autograd through the oracle's prep on the same bf16 inputs.
Error: 2-norm of the difference over 2-norm of the gradient.  A gradient passes
at most four bf16 roundings (y1, the pre-norm value, dy2, dy1) of 2^-8 each
before its own: 2^-6 bounds them with the output's."""
from __future__ import annotations

import pytest
import torch

from oracle import ccgqa as occ

pytestmark = pytest.mark.gpu

NAMES = ("q_conv.conv1.weight", "q_conv.conv2.weight", "k_conv.conv1.weight", "k_conv.conv2.weight")


def _grads(cuda, B, S, Hq, Hkv, hd, features):
    from hydra_amd.attention.backends.ccgqa.autograd import ccgqa_prep_train
    from hydra_amd.attention.backends.ccgqa.ops import prep_flags

    use_mean, use_shift, use_norm, use_rope = features
    cfg = occ.CCGQAConfig(dim=4 * Hq * hd, n_heads=Hq, n_kv_heads=Hkv, compression_factor=4, max_seq_len=512,
                          use_qk_mean=use_mean, use_value_shift=use_shift, use_qk_norm=use_norm, use_rope=use_rope)
    g = torch.Generator().manual_seed(S * 7 + hd + Hq)
    L, K = Hq * hd, Hkv * hd
    params = {k: v.to(torch.bfloat16) for k, v in occ.init_params(cfg, g, std=0.1, temperature=1.7).items()}
    rand = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)  # noqa: E731
    qkv, gq, gk, gv = rand(B, S, L + 2 * K), rand(B, Hq, S, hd), rand(B, Hkv, S, hd), rand(B, Hkv, S, hd)
    cos, sin = occ.fused_ops.rope_cache(hd, S)
    p64 = {k: v.double().requires_grad_() for k, v in params.items()}
    x64 = qkv.double().requires_grad_()
    q, k, v = occ.prep(p64, x64, cfg, cos.double(), sin.double())
    wrt = [x64] + [p64[n] for n in NAMES] + ([p64["key_temperature"]] if use_norm else [])
    ref = torch.autograd.grad((q * gq.double()).sum() + (k * gk.double()).sum() + (v * gv.double()).sum(), wrt)

    dp = {k: v.to(cuda).requires_grad_() for k, v in params.items()}
    xd = qkv.to(cuda).requires_grad_()
    flags = prep_flags(True, use_mean, use_shift, use_norm, use_rope)
    outs = ccgqa_prep_train(xd, Hq, Hkv, hd, flags, *(dp[n] for n in NAMES),
                            temperature=dp["key_temperature"] if use_norm else None,
                            cos=cos.to(cuda) if use_rope else None, sin=sin.to(cuda) if use_rope else None)
    wrt = [xd] + [dp[n] for n in NAMES] + ([dp["key_temperature"]] if use_norm else [])
    # the temperature's gradient is the sum of <dk, k> / temperature over tokens and heads
    terms = ((k * gk.double()).sum(-1) / p64["key_temperature"]).detach() if use_norm else None
    return torch.autograd.grad(outs, wrt, [t.to(cuda) for t in (gq, gk, gv)]), ref, terms


def _check(got, ref, terms):
    for i, (a, r) in enumerate(zip(got, ref)):
        a = a.double().cpu()
        assert a.shape == r.shape and torch.isfinite(a).all(), i
        if r.numel() > 1:
            err = float((a - r).norm() / r.norm())
            assert err < 2.0 ** -6, f"output {i}: {err:.3g}"
        else:
            # One value, a sum of signed terms.  The roundings above reach each
            # term apart, at 2^-8 of its size where they fall, so their sum
            # grows as the terms' 2-norm; the result's own is 2^-9 of it.  One
            # token's terms left out are 1 / sqrt(tokens) of that norm: 0.05 at
            # the most tokens tested, against 2^-6 = 0.016.
            err, size = float((a - r).abs()), float(terms.norm())
            assert err < 2.0 ** -6 * size + 2.0 ** -9 * float(r.abs()), f"temperature: {err / size:.3g}"


@pytest.mark.parametrize("heads", [(2, 2, 8), (4, 2, 16), (28, 4, 16), (3, 3, 32), (6, 2, 32), (8, 2, 64), (2, 1, 128),
                                   (4, 2, 128), (2, 1, 24)])
@pytest.mark.parametrize("B,S", [(1, 1), (2, 2), (1, 64), (1, 127), (3, 129), (2, 200)])
def test_conv_backward_shapes(cuda, heads, B, S):
    _check(*_grads(cuda, B, S, *heads, (True, True, True, True)))


@pytest.mark.parametrize("features", [(False, False, False, False), (True, False, False, True),
                                      (False, True, True, False)])
def test_conv_backward_features(cuda, features):
    _check(*_grads(cuda, 2, 70, 4, 2, 32, features))


@pytest.mark.parametrize("hd,S", [(16, 70), (64, 33), (128, 129)])
def test_bf16_rope_tables(cuda, hd, S):
    """bf16 RoPE tables (a module cast to bf16) are widened inside the kernels:
    the same bits as tables converted to fp32 before the call, forward and
    backward, also from a longer [1, 1, Smax, hd/2] cache."""
    from hydra_amd.attention.backends.ccgqa.autograd import ccgqa_prep_train
    from hydra_amd.attention.backends.ccgqa.ops import prep_flags

    Hq, Hkv = 4, 2
    g = torch.Generator().manual_seed(hd + S)
    L, K = Hq * hd, Hkv * hd
    rand = lambda *s: (torch.randn(*s, generator=g) * 0.3).to(torch.bfloat16).to(cuda)  # noqa: E731
    ws = [rand(L, hd, 3), rand(L, L, 3), rand(K, hd, 3), rand(K, K, 3)]
    qkv, temp = rand(2, S, L + 2 * K), torch.ones(1, dtype=torch.bfloat16, device=cuda)
    gos = [rand(2, h, S, hd) for h in (Hq, Hkv, Hkv)]
    cos, sin = (t.to(torch.bfloat16).to(cuda) for t in occ.fused_ops.rope_cache(hd, 200))
    flags = prep_flags(True, True, True, True, True)
    res = []
    for c, s in ((cos, sin), (cos.float(), sin.float())):
        leaves = [t.clone().requires_grad_() for t in (qkv, *ws, temp)]
        outs = ccgqa_prep_train(leaves[0], Hq, Hkv, hd, flags, *leaves[1:5], temperature=leaves[5], cos=c, sin=s)
        res.append([*outs, *torch.autograd.grad(outs, leaves, gos)])
    for a, b in zip(*res):
        assert torch.equal(a, b)
