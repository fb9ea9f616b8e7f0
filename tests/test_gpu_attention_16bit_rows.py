"""Attention of 16-bit rows outside the bf16 tile kernels (fp16, odd head
dims): rows multiply on the 16-bit matrix instructions, probabilities and
score gradients as planes of 16-bit values.  What can go wrong there: tile
edges, subnormal fp16 elements, score gradients past fp16's range, and
infinities, which a plane's zero or negative remainder would turn into NaN.

Reference: fp64 softmax of the same rounded inputs.  2-norm errors: a
rounding of the output is u / 2 at most (u = 2^-11 fp16, 2^-8 bf16), u bounds
it with the sums' own; gradients add D = rowsum(dO * O) from the rounded O and
the forward's own rounding, 2 u."""
from __future__ import annotations

import pytest
import torch

from oracle import ccgqa as occ

pytestmark = pytest.mark.gpu

U = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _inputs(B, Hq, Hkv, S, hd, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    mk = lambda h: torch.randn(B, h, S, hd, generator=g)
    return [t.to(dtype) for t in (mk(Hq), mk(Hkv), mk(Hkv), mk(Hq))]


def _run(cuda, q, k, v, go, causal, scale=None):
    from hydra_amd.attention.backends.ccgqa.ops import attention_backward, attention_forward

    qd, kd, vd, god = (t.to(cuda) for t in (q, k, v, go))
    kw = {} if scale is None else {"scale": scale}
    out, lse = attention_forward(qd, kd, vd, causal=causal, want_lse=True, **kw)
    return [t.double().cpu() for t in (out, *attention_backward(qd, kd, vd, out, lse, god, causal=causal, **kw), lse)]


def _reference(q, k, v, go, causal):
    q, k, v = (t.double().requires_grad_() for t in (q, k, v))
    out = occ.attention_key_padding(q, k, v, causal=causal, mask=None)
    out.backward(go.double())
    return [out.detach(), q.grad, k.grad, v.grad]


def _check(got, want, dtype):
    for name, a, r, tol in zip(("out", "dq", "dk", "dv"), got, want, (U[dtype], *[2 * U[dtype]] * 3)):
        err = float((a - r).norm() / r.norm())
        assert err < tol, f"{name}: {err:.3g}"


@pytest.mark.parametrize("dtype,hd", [(torch.float16, 16), (torch.float16, 32), (torch.float16, 64),
                                      (torch.float16, 128), (torch.float16, 40), (torch.bfloat16, 80)])
@pytest.mark.parametrize("S,causal", [(1, True), (31, False), (33, True), (64, False), (127, True), (1030, True)])
def test_tile_edges(cuda, dtype, hd, S, causal):
    ins = _inputs(2, 4, 2, S, hd, dtype, S + hd)
    got, want = _run(cuda, *ins, causal), _reference(*ins, causal)
    if S == 1:  # dS is 0 up to the rounding of O inside D
        got, want = [got[0], got[3]], [want[0], want[3]]
    _check(got, want, dtype)


@pytest.mark.parametrize("hd", [16, 64])
def test_subnormal_rows(cuda, hd):
    """Subnormal q (2^-15 and below, lost entirely if flushed) against keys of
    2^13: scores of order 1.  Subnormal v: the output to fp16's smallest step."""
    q, k, v, go = _inputs(1, 4, 1, 200, hd, torch.float16, hd)
    q, k = (q.float() * 2.0 ** -15).half(), (k.float() * 2.0 ** 13).half()
    got, want = _run(cuda, q, k, v, go, True), _reference(q, k, v, go, True)
    assert float((got[0] - want[0]).norm() / want[0].norm()) < U[torch.float16]
    assert float((got[3] - want[3]).norm() / want[3].norm()) < 2 * U[torch.float16]
    v = (v.float() * 2.0 ** -18).half()
    got, want = _run(cuda, q, k, v, go, True), _reference(q, k, v, go, True)
    assert float((got[0] - want[0]).abs().max()) <= 2.0 ** -24


def test_score_gradients_past_fp16(cuda):
    """|dS| up to 1e6: past fp16's largest value, and results inside it."""
    q, k, v, go = _inputs(1, 2, 1, 97, 64, torch.float16, 5)
    q, k, v, go = (q.float() * 0.004).half(), (k.float() * 0.004).half(), (v * 100), (go * 300)
    got, want = _run(cuda, q, k, v, go, True), _reference(q, k, v, go, True)
    assert max(float(w.abs().max()) for w in want) < 65504
    # D is a sum of 64 products of the rounded O; its error enters dS beside a
    # dP of the same size, so the four half ulps of the bound stand
    _check(got, want, torch.float16)


@pytest.mark.parametrize("dtype,hd", [(torch.float16, 64), (torch.float16, 16), (torch.bfloat16, 80)])
def test_infinities(cuda, dtype, hd):
    """An infinite v element: an infinite output element for every query that
    sees the key, the others as without it.  An infinite dO element: the same
    for dv of every key that its query sees."""
    q, k, v, go = _inputs(1, 2, 1, 150, hd, dtype, 3)
    base = _run(cuda, q, k, v, go, True)
    v2 = v.clone()
    v2[0, 0, 70, 5] = float("inf")
    out = _run(cuda, q, k, v2, go, True)[0]
    assert (out[0, :, 70:, 5] == float("inf")).all()
    before = (out[0, :, :70] - base[0][0, :, :70]).norm() / base[0][0, :, :70].norm()
    assert float(before) < U[dtype]  # NaN fails
    keep = [d for d in range(hd) if d != 5]
    assert float((out[..., keep] - base[0][..., keep]).norm() / base[0].norm()) < U[dtype]
    go2 = go.clone()
    go2[0, 1, 70, 5] = float("-inf")
    dv = _run(cuda, q, k, v, go2, True)[3]
    assert (dv[0, 0, :71, 5] == float("-inf")).all()
    after = (dv[0, 0, 71:] - base[3][0, 0, 71:]).norm() / base[3][0, 0, 71:].norm()
    assert float(after) < 2 * U[dtype]
    assert float((dv[..., keep] - base[3][..., keep]).norm() / base[3].norm()) < 2 * U[dtype]
