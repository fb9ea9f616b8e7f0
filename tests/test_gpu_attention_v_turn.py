"""GPU parity of the attention forward on row-major V around the rule that
transposes V first (more than one 64-key tile, few items) and at the padded
last chunk of V^T rows (S off a multiple of 8), over head dims, masks and
strided views.  bf16 against the oracle in fp64: two roundings of P and of the
output (2^-9 relative on average each) -- 2-norm below 2^-7."""
from __future__ import annotations

import pytest
import torch

from oracle import ccgqa as occ

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd", [16, 32, 64, 128])
@pytest.mark.parametrize("S", [63, 64, 65, 71, 72, 127, 200, 333])
@pytest.mark.parametrize("causal,masked", [(True, False), (False, False), (True, True)])
def test_row_major_v(cuda, S, hd, causal, masked):
    from hydra_amd.attention.backends.ccgqa.ops import MASK_KEY_PADDING, MASK_NONE, attention_forward

    B, Hq, Hkv = 2, 4, 2
    g = torch.Generator().manual_seed(S + hd)
    q = torch.randn(B, Hq, S, hd, generator=g).to(torch.bfloat16)
    k = torch.randn(B, Hkv, S, hd, generator=g).to(torch.bfloat16)
    wide = torch.randn(B, S, Hkv, hd + 8, generator=g).to(torch.bfloat16)  # v: a view with padded rows
    v = wide[..., :hd].transpose(1, 2)
    mask = None
    if masked:
        mask = torch.ones(B, S, dtype=torch.long)
        mask[1, S // 2:] = 0
    kw = dict(key_mask=mask.to(cuda), mask_mode=MASK_KEY_PADDING) if masked else dict(mask_mode=MASK_NONE)
    vd = wide.to(cuda)[..., :hd].transpose(1, 2)
    out, lse = attention_forward(q.to(cuda), k.to(cuda), vd, causal=causal, want_lse=True, **kw)
    ref = occ.attention_key_padding(q, k, v, causal=causal, mask=mask)
    got = out.double().cpu()
    assert torch.isfinite(got).all() and torch.isfinite(lse).all()
    assert float((got - ref).norm() / ref.norm()) < 2.0 ** -7
