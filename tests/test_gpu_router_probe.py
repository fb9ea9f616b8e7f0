"""The MoD wrapper's dense path without gradients: router scores and their
probabilities' mean and deviation from hydra_router_probe, the block's residual
add inside the down projection.

Bounds: scores are one rounding of an fp32 sum of D products (u per element,
u = 2^-8 bf16, 2^-11 fp16; fp32: D roundings of 2^-24 of the absolute
products, D = 1800 at most, over its square root in the mean: 2^-18 with room).
Mean and deviation are computed from the device's own scores: one rounding of
p (u / 2), of the result (u / 2): u."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

U = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -18}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,dim", [(2, 8), (3, 33), (255, 64), (4097, 1792), (5, 4100), (9000, 72)])
@pytest.mark.parametrize("view", [False, True])
def test_router_probe(cuda, rows, dim, dtype, view):
    from hydra_amd.routing.ops import router_probe

    g = torch.Generator().manual_seed(rows + dim)
    x = torch.randn(rows, dim + 3 if view else dim, generator=g).to(dtype).to(cuda)[:, :dim]
    w = (torch.randn(1, dim, generator=g) / dim ** 0.5 * 2).to(dtype).to(cuda)
    b = torch.randn(1, generator=g).to(dtype).to(cuda)
    scores, stats = router_probe(x, w, b)
    want = x.double() @ w.double().t()[:, 0] + b.double()
    size = x.double().abs() @ w.double().abs().t()[:, 0] + b.double().abs()
    tol = U[dtype] * (size if dtype == torch.float32 else want.abs() + 2.0 ** -12 * size)
    assert ((scores.double() - want).abs() <= tol).all()
    p = torch.sigmoid(scores.double().clamp(-10, 10))
    for got, ref in ((stats[0], p.mean()), (stats[1], p.std())):
        assert abs(float(got) - float(ref)) <= U[dtype] * max(float(ref), float(p.mean()))


def test_router_probe_edges(cuda):
    from hydra_amd.routing.ops import router_probe

    x = torch.ones(1, 16, device=cuda)
    w, b = torch.full((1, 16), 100.0, device=cuda), torch.zeros(1, device=cuda)
    scores, stats = router_probe(x, w, b)  # one row: no deviation; scores past the clamp
    assert float(scores[0]) == 1600.0 and torch.isnan(stats[1])
    assert abs(float(stats[0]) - float(torch.sigmoid(torch.tensor(10.0)))) < 1e-6
    x = torch.ones(70, 16, device=cuda)
    x[69, 3] = float("nan")
    scores, stats = router_probe(x, w, b)
    assert torch.isnan(scores[69]) and torch.isnan(stats).all() and (scores[:69] == 1600.0).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_block_dense_wrapper(cuda, dtype):
    """The fixed path of a MoR block over a wrapper that does not route yet:
    the same as with the modules called one by one (what a forward hook makes
    it do), statistics included; the input is left alone."""
    from hydra_amd.model.framework.blocks import HydraMoRBlock

    torch.manual_seed(3)
    blk = HydraMoRBlock(256, n_heads=8, n_kv_heads=2, max_seq_len=64, max_recursions=3, adaptive=False,
                        attention_type="ccqa", mod_mlp_capacity=0.5).to(cuda, dtype).eval()
    x = torch.randn(2, 48, 256, device=cuda).to(dtype)
    kept = x.clone()
    wrap = blk.mod_mlp_wrapper
    with torch.no_grad():
        got = blk(x)
        noted = [float(wrap._last_probs_mean_t), float(wrap._last_probs_std_t), wrap.get_routing_stats()["routing_mode"]]
        scores = wrap._last_scores.double()
        again = blk(x)
        calls = []
        hooks = [wrap.register_forward_hook(lambda *a: calls.append("wrapper")),
                 wrap.mod_router.router.register_forward_hook(lambda *a: calls.append("router"))]
        want = blk(x)
        for h in hooks:
            h.remove()
    assert calls == ["router", "wrapper"] * 3
    assert torch.equal(x, kept) and torch.equal(got, again)
    # three recursions, one residual rounding (u / 2) each that the two forms place differently
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -20
    assert float((got - want).double().norm() / want.double().norm()) < 3 * u
    assert float((scores - wrap._last_scores.double()).norm() / scores.norm()) < 4 * u
    assert abs(noted[0] - float(wrap._last_probs_mean_t)) <= 4 * u and noted[2] == "disabled"
    assert abs(noted[1] - float(wrap._last_probs_std_t)) <= 4 * u
