"""A key mask reaches the attention kernels as bytes: a bool mask's own, any
other type compared with zero.  Every form of one mask gives the same bits,
forward and backward, and the token-row output layout gives those of the
head-major one."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

FORMS = {"long": lambda m: m.long(), "float": lambda m: m.float() * 0.25, "bool": lambda m: m,
         "strided": lambda m: torch.stack((m, ~m), -1)[..., 0], "transposed": lambda m: m.t().contiguous().t(),
         "expanded": lambda m: m}


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("token_rows", [False, True])
def test_mask_forms(cuda, form, token_rows):
    from hydra_amd.attention.backends.ccgqa.kernels.fused_attention import MaskedAttentionFunction
    from hydra_amd.attention.backends.ccgqa.ops import MASK_KEY_PADDING

    g = torch.Generator().manual_seed(4)
    B, Hq, Hkv, S, hd = 3, 4, 2, 77, 64
    q, k, v = (torch.randn(B, h, S, hd, generator=g).to(cuda, torch.bfloat16) for h in (Hq, Hkv, Hkv))
    go = torch.randn(B, Hq, S, hd, generator=g).to(cuda, torch.bfloat16)
    if form == "expanded":
        mask = (torch.rand(1, S, generator=g) < 0.7).to(cuda).expand(B, S)
    else:
        mask = (torch.rand(B, S, generator=g) < 0.7).to(cuda)

    def run(m, *extra):
        ts = [t.clone().requires_grad_() for t in (q, k, v)]
        out = MaskedAttentionFunction.apply(*ts, m, MASK_KEY_PADDING, True, *extra)
        return [out.detach(), *torch.autograd.grad(out, ts, go)]

    want = run(mask.to(torch.int32).contiguous())
    got = run(FORMS[form](mask), token_rows)
    if token_rows:
        assert got[0].transpose(1, 2).is_contiguous()
    assert all(torch.equal(a, b) for a, b in zip(got, want))
