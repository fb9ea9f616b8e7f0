"""The CCGQA forward captured in a HIP graph (torch.cuda.graph) replays to
the eager result: several replays with eager work and synchronisations in
between, each compared bit for bit (the same kernels run on the same
inputs; every kernel on the path is deterministic), then a replay on new
input content against the eager forward of that content.  bench.py times
the config-3 step this way."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def test_ccgqa_forward_graph_replays_match_eager(cuda):
    from hydra_amd.attention import CCGQAAttention

    torch.manual_seed(3)
    m = CCGQAAttention(dim=1024, n_heads=4, n_kv_heads=1, compression_factor=4, max_seq_len=1024)
    with torch.no_grad():
        for p in m.parameters():
            p.copy_(torch.randn(p.shape) * 0.02)
        m.key_temperature.fill_(1.0)
    m = m.to(cuda, torch.bfloat16).eval()
    g = torch.Generator(device=cuda).manual_seed(4)
    x = torch.randn(2, 1024, 1024, device=cuda, generator=g).to(torch.bfloat16)
    with torch.no_grad():
        m(x)
        want = m(x).clone()
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            m(x)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = m(x)
    for r in range(4):
        noise = torch.randn(4096, 4096, device=cuda, generator=g).sum()  # eager work between replays
        torch.cuda.synchronize()
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want), f"replay {r} differs from the eager forward"
        del noise
    x2 = torch.randn(x.shape, device=cuda, generator=g).to(torch.bfloat16)
    with torch.no_grad():
        want2 = m(x2).clone()
    x.copy_(x2)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(y, want2)
    del graph


def test_hydra_model_forward_graph_replays_match_eager(cuda):
    """The config-5 model path (MoR blocks, MoD middle blocks, tied LM head)
    captured in a HIP graph: routing is capacity-based, so every shape is
    fixed and the forward has no host synchronisation.  Replays with eager
    work in between equal the eager logits bit for bit, and a replay on new
    token ids equals the eager forward of those ids.  bench.py times config
    5 this way."""
    from test_gpu_blocks import _model_from_checkpoint

    m, z, meta = _model_from_checkpoint(cuda, torch.bfloat16)
    g = torch.Generator(device=cuda).manual_seed(5)
    ids = torch.from_numpy(z["ids"]).to(cuda)
    with torch.no_grad():
        m(ids)
        want = m(ids).clone()
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            m(ids)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = m(ids)
    for r in range(3):
        noise = torch.randn(4096, 4096, device=cuda, generator=g).sum()
        torch.cuda.synchronize()
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want), f"replay {r} differs from the eager forward"
        del noise
    ids2 = torch.randint(0, meta["vocab_size"], ids.shape, device=cuda, generator=g)
    with torch.no_grad():
        want2 = m(ids2).clone()
    ids.copy_(ids2)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(y, want2)
    del graph


def _layer(cuda, seed=3):
    from hydra_amd.attention import CCGQAAttention

    torch.manual_seed(seed)
    m = CCGQAAttention(dim=1024, n_heads=4, n_kv_heads=1, compression_factor=4, max_seq_len=512)
    with torch.no_grad():
        for p in m.parameters():
            p.copy_(torch.randn(p.shape) * 0.02)
        m.key_temperature.fill_(1.0)
    return m.to(cuda, torch.bfloat16).eval()


def _input(cuda):
    g = torch.Generator(device=cuda).manual_seed(4)
    return torch.randn(2, 512, 1024, device=cuda, generator=g).to(torch.bfloat16)


def _captured(m, x):
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):  # the libraries' own first calls
        _layer(x.device)(x)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = m(x)
    return graph, y


def test_first_call_in_a_capture(cuda):
    """Weights packed inside the capture exist once the graph replays: an
    eager call before that packs its own."""
    x = _input(cuda)
    with torch.no_grad():
        want = _layer(cuda)(x).clone()
        m = _layer(cuda)
        graph, y = _captured(m, x)
        assert torch.equal(m(x), want)
        for _ in range(3):
            y.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, want)
            assert torch.equal(m(x), want)
    del graph


def test_weights_changed_after_a_capture(cuda):
    """Replays read the packed weights that the last eager call left, in the
    memory that the capture saw."""
    x = _input(cuda)
    with torch.no_grad():
        m = _layer(cuda)
        m(x)
        graph, y = _captured(m, x)
        for seed in (5, 6):
            for p, q in zip(m.parameters(), _layer(cuda, seed).parameters()):
                p.copy_(q)
            want = m(x).clone()
            other = torch.full((1 << 24,), 7.0, device=cuda)  # what a freed pack's memory would hold
            for _ in range(3):
                y.zero_()
                graph.replay()
                torch.cuda.synchronize()
                assert torch.equal(y, want)
            del other
        assert torch.equal(want, _layer(cuda, 6)(x))
    del graph


def test_first_call_on_another_stream(cuda):
    """A call on the default stream right after the packing one on a busy
    stream."""
    x = _input(cuda)
    with torch.no_grad():
        want = _layer(cuda)(x).clone()
        a = torch.randn(8192, 8192, device=cuda).to(torch.bfloat16)
        a @ a
        m = _layer(cuda)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(8):
                a @ a
            y = m(x)
        got = m(x)
        torch.cuda.synchronize()
        assert torch.equal(y, want) and torch.equal(got, want)


def _replays_equal(step, leaf, again):
    """Captures step() (outputs: a list of tensors) and compares every output
    of several replays, eager work and synchronizations between them, with the
    eager call; then once more with `again` written into leaf."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = step()
    for new in (None, again):
        if new is not None:
            with torch.no_grad():
                leaf.copy_(new)
        want = [t.clone() for t in step()]
        for r in range(3):
            noise = torch.randn(2048, 2048, device=leaf.device).sum()
            torch.cuda.synchronize()
            for t in outs:
                t.zero_()
            graph.replay()
            torch.cuda.synchronize()
            for i, (a, b) in enumerate(zip(outs, want)):
                assert torch.equal(a, b), f"replay {r}, output {i} of {len(outs)}"
            del noise
    del graph


@pytest.mark.parametrize("padded", [False, True])
def test_layer_training_step(cuda, padded, monkeypatch):
    monkeypatch.setenv("HYDRA_CCGQA_MASK_SEMANTICS", "key_padding")
    m, x = _layer(cuda).train(), _input(cuda).requires_grad_()
    go = torch.randn(x.shape, device=cuda).to(torch.bfloat16)
    mask = torch.arange(512, device=cuda) < torch.tensor([[512], [300]], device=cuda) if padded else None

    def step():
        y = m(x, mask=mask)
        return [y.detach(), *torch.autograd.grad(y, [x, *m.parameters()], go)]

    _replays_equal(step, x, torch.randn_like(x))


@pytest.mark.parametrize("n,V", [(3000, 32000), (3000, 4099), (70000, 512)])
def test_loss_step(cuda, n, V):
    from hydra_amd.kernels import chunked_cross_entropy

    h = torch.randn(n, 256, device=cuda).to(torch.bfloat16).requires_grad_()
    w = (torch.randn(V, 256, device=cuda) * 0.05).to(torch.bfloat16).requires_grad_()
    t = torch.randint(0, V, (n,), device=cuda)
    t[::7] = -100

    def step():
        loss = chunked_cross_entropy(h, w, t, chunk_size=2048)
        return [loss.detach(), *torch.autograd.grad(loss, [h, w])]

    _replays_equal(step, h, torch.randn_like(h))


def test_mod_training_step(cuda):
    from hydra_amd.kernels import fused_rms_norm
    from hydra_amd.routing import gather_by_indices, mod_topk, weighted_residual_scatter

    B, L, D, k = 4, 1024, 512, 768
    scores = torch.randn(B, L, device=cuda)
    x = torch.randn(B, L, D, device=cuda).to(torch.bfloat16).requires_grad_()
    gain = torch.ones(D, device=cuda, dtype=torch.bfloat16).requires_grad_()
    weights = torch.rand(B, k, device=cuda).requires_grad_()
    go = torch.randn(B, L, D, device=cuda).to(torch.bfloat16)

    def step():
        _, idx, _ = mod_topk(scores, k)
        y = fused_rms_norm(gather_by_indices(x, idx, distinct=True), gain)
        out = weighted_residual_scatter(x.clone(), y, idx, weights)
        return [out.detach(), *torch.autograd.grad(out, [x, gain, weights], go)]

    _replays_equal(step, x, torch.randn_like(x))
