"""The bf16 attention backward on both sides of the line past which dQ runs on
the library's side stream (2048 keys; head_dim 128; 6 G products): gradients
against the reference of test_gpu_attention_backward.py with its bounds, the
same bits from two user streams at once, and from replays of a captured graph
with eager calls between them."""
from __future__ import annotations

import pytest
import torch

from test_gpu_attention_backward import TOL, _check, _inputs

pytestmark = pytest.mark.gpu

SHAPES = [(1, 2, 1, 2048, 64), (1, 2, 1, 2049, 64), (1, 2, 1, 2080, 16), (1, 2, 2, 300, 128)]


def _call(q, k, v, go, causal):
    from hydra_amd.attention.backends.ccgqa.ops import attention_backward, attention_forward

    out, lse = attention_forward(q, k, v, causal=causal, want_lse=True)
    return (q, k, v, out, lse, go), attention_backward(q, k, v, out, lse, go, causal=causal)


@pytest.mark.parametrize("shape", SHAPES)
def test_overlap_line(cuda, shape):
    from hydra_amd.attention.backends.ccgqa.ops import attention_backward

    host = _inputs(*shape, torch.bfloat16, seed=5)
    first, want = _call(*(t.to(cuda) for t in host), True)
    _check(want, *host, True, TOL[torch.bfloat16])
    second, want2 = _call(*(t.to(cuda) for t in _inputs(*shape, torch.bfloat16, seed=6)), True)
    torch.cuda.synchronize()
    streams, got = [torch.cuda.Stream(), torch.cuda.Stream()], []
    for st, c in zip(streams, (first, second)):
        with torch.cuda.stream(st):
            got.append(attention_backward(*c, causal=True))
    torch.cuda.synchronize()
    for g, w in zip(got, (want, want2)):
        assert all(torch.equal(a, b) for a, b in zip(g, w))

    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = attention_backward(*first, causal=True)
    for _ in range(3):
        for t in out:
            t.zero_()
        graph.replay()
        eager = attention_backward(*second, causal=True)
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, want))
        assert all(torch.equal(a, b) for a, b in zip(eager, want2))
