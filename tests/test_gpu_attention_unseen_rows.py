"""What a query does not see stays out of it, whatever it holds: a key or value
row full of infinities and NaNs changes nothing for queries that do not see it
(masked, or later than they are), a query row nothing for keys that it does not
see.  In a product over a whole tile the unseen rows meet weights of 0, and
0 * inf is NaN, so the kernels skip them by rule and not by weight.

Forms: every attention backward but that of unmasked bf16 at head dims 32, 64
and 128, and the forward of the same element types and head dims (bf16 forwards
at 16, 32, 64 and 128 excepted).  Compared with the clean run by 2-norm: two
results of the same kernel family, each within u of the exact one (u = 2^-8
bf16, 2^-11 fp16: half an ulp, and the same through D and the forward's
rounding; fp32: sums of at most 200 terms, 2^-17)."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10, torch.float32: 2.0 ** -16}
BAD = torch.tensor([float("inf"), float("nan"), -float("inf"), 1.0])
S = 150


def _poison(t, row):
    t = t.clone()
    t[:, :, row] = BAD.repeat(t.shape[-1] // 4 + 1)[:t.shape[-1]].to(t)
    return t


def _sees(mode, causal, mask):
    """[B, S, S]: query s sees key t."""
    s, t = torch.arange(S)[:, None], torch.arange(S)[None]
    keep = mask.bool()[:, None]
    if mode == 2:
        return (t > s) | ~keep
    seen = (t <= s) if causal else torch.ones(S, S, dtype=torch.bool)
    return seen & (keep if mode == 1 else torch.ones_like(keep))


def _case(cuda, dtype, hd, mode):
    g = torch.Generator().manual_seed(hd)
    B, Hq, Hkv = 2, 4, 2
    q, go = (torch.randn(B, Hq, S, hd, generator=g).to(cuda, dtype) for _ in range(2))
    k, v = (torch.randn(B, Hkv, S, hd, generator=g).to(cuda, dtype) for _ in range(2))
    mask = torch.arange(S)[None] % 5 != torch.tensor([[1], [3]])
    mask[1, 100:] = False
    kw = {"causal": True, "mask_mode": mode, "key_mask": mask.to(cuda) if mode else None}
    return q, k, v, go, mask, kw


def _same(name, got, want, rows, dtype):
    """rows [B, S]: the rows that must not differ."""
    rows = rows[:, None].expand(got.shape[:3])
    got, want = got.double().cpu()[rows], want.double().cpu()[rows]
    assert rows.any() and torch.isfinite(got).all(), name
    assert float((got - want).norm()) <= TOL[dtype] * float(want.norm()), name


FORMS = [(torch.bfloat16, 16, 0), (torch.bfloat16, 80, 0), (torch.float16, 64, 0), (torch.float16, 16, 0),
         (torch.float16, 40, 0), (torch.float32, 64, 0), (torch.float32, 128, 0), (torch.float32, 24, 0)]
FORMS += [(dt, hd, mode) for mode in (1, 2) for dt, hd in
          [(torch.bfloat16, 16), (torch.bfloat16, 32), (torch.bfloat16, 64), (torch.bfloat16, 128), (torch.bfloat16, 80),
           (torch.float16, 64), (torch.float16, 128), (torch.float32, 32), (torch.float32, 80)]]


@pytest.mark.parametrize("dtype,hd,mode", FORMS)
@pytest.mark.parametrize("row", [0, 70, 131, S - 1])
def test_backward(cuda, dtype, hd, mode, row):
    from hydra_amd.attention.backends.ccgqa.ops import attention_backward, attention_forward

    q, k, v, go, mask, kw = _case(cuda, dtype, hd, mode)
    out, lse = attention_forward(q, k, v, want_lse=True, **kw)
    clean = attention_backward(q, k, v, out, lse, go, **kw)
    sees = _sees(mode, True, mask).expand(2, S, S)
    others = (torch.arange(S) != row).expand(2, S)
    # a bad key and value row: dq of the queries that do not see it, dk and dv
    # of the other keys
    got = attention_backward(q, _poison(k, row), _poison(v, row), out, lse, go, **kw)
    if (~sees[:, :, row]).any():
        _same("dq, bad key", got[0], clean[0], ~sees[:, :, row], dtype)
    _same("dk, bad key", got[1], clean[1], others, dtype)
    _same("dv, bad key", got[2], clean[2], others, dtype)
    # a bad query row: dk and dv of the keys that it does not see, dq of the
    # other queries
    got = attention_backward(_poison(q, row), k, v, out, lse, _poison(go, row), **kw)
    _same("dq, bad query", got[0], clean[0], others, dtype)
    if (~sees[:, row]).any():
        _same("dk, bad query", got[1], clean[1], ~sees[:, row], dtype)
        _same("dv, bad query", got[2], clean[2], ~sees[:, row], dtype)


@pytest.mark.parametrize("dtype,hd,mode", [f for f in FORMS if f[0] != torch.bfloat16 or f[1] == 80])
@pytest.mark.parametrize("row", [0, 70, 131, S - 1])
@pytest.mark.parametrize("heads", [1, 64])
def test_forward(cuda, dtype, hd, mode, row, heads):
    """heads: few workgroups (key groups share a walk) and many."""
    from hydra_amd.attention.backends.ccgqa.ops import attention_forward

    q, k, v, _, mask, kw = _case(cuda, dtype, hd, mode)
    q, k, v = (t.repeat(1, heads, 1, 1) for t in (q, k, v))
    out, lse = attention_forward(q, k, v, want_lse=True, **kw)
    unseen = ~_sees(mode, True, mask).expand(2, S, S)[:, :, row]
    if not unseen.any():
        pytest.skip("every query sees the row")
    got, glse = attention_forward(q, _poison(k, row), _poison(v, row), want_lse=True, **kw)
    _same("out", got, out, unseen, dtype)
    seen = unseen[:, None].expand(glse.shape).to(cuda) & torch.isfinite(lse)
    assert torch.allclose(glse[seen], lse[seen], rtol=1e-5, atol=1e-5)
