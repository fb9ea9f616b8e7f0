"""Backward passes asked to record themselves (create_graph): the gradients are
those of a plain backward, and what torch can record of them is recorded."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_cross_entropy(cuda, dtype):
    from hydra_amd.kernels.fused_ops import chunked_cross_entropy

    g = torch.Generator().manual_seed(5)
    h = torch.randn(2, 9, 16, generator=g).to(dtype).to(cuda).requires_grad_()
    w = (torch.randn(41, 16, generator=g) / 4).to(dtype).to(cuda).requires_grad_()
    t = torch.randint(0, 41, (2, 9), generator=g).to(cuda)
    want = torch.autograd.grad(chunked_cross_entropy(h, w, t, chunk_size=7), (h, w))
    got = torch.autograd.grad(chunked_cross_entropy(h, w, t, chunk_size=7), (h, w), create_graph=True)
    for a, b in zip(got, want):  # two orders of the same sums, rounded once each to dtype
        tol = 2.0 ** -8 if dtype == torch.bfloat16 else 1e-6
        assert float((a - b).detach().double().norm()) <= tol * float(b.double().norm())


def test_weighted_scatter(cuda):
    """grad_w = <g[idx], values>: its derivative by values is the selected
    rows of g."""
    from hydra_amd.routing.ops import weighted_residual_scatter

    g = torch.Generator().manual_seed(6)
    x = torch.randn(2, 12, 8, generator=g).to(cuda)
    vals = torch.randn(2, 5, 8, generator=g).to(cuda).requires_grad_()
    w = torch.rand(2, 5, generator=g).to(cuda).requires_grad_()
    idx = torch.stack([torch.randperm(12, generator=g)[:5].sort().values for _ in range(2)]).to(cuda)
    go = torch.randn(2, 12, 8, generator=g).to(cuda)
    want = torch.autograd.grad(weighted_residual_scatter(x.clone(), vals, idx, w), (vals, w), go)
    got = torch.autograd.grad(weighted_residual_scatter(x.clone(), vals, idx, w), (vals, w), go, create_graph=True)
    torch.testing.assert_close(got[0].detach(), want[0], rtol=1e-6, atol=0)
    torch.testing.assert_close(got[1].detach(), want[1], rtol=1e-5, atol=1e-5)  # sums of 8 terms of ~1
    (second,) = torch.autograd.grad(got[1].sum(), vals)
    assert torch.equal(second, go.gather(1, idx[..., None].expand(2, 5, 8)))
