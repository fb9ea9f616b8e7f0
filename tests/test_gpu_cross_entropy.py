"""GPU parity of the chunked LM-head cross-entropy (hydra_ce_rows plus the
GEMMs around it) against the oracle's fp64 restatement of
ChunkedCrossEntropyFunction (pinned by autograd of F.cross_entropy in
tests/test_oracle_pins.py): the loss and both gradients.  Tolerance: fp32
1e-5, bf16 2e-2 (max-rel-err; the forward's logits are bf16 GEMM outputs, as
in the reference)."""
from __future__ import annotations

import pytest
import torch

from conftest import max_rel_err
from oracle import fused_ops as ofo

pytestmark = pytest.mark.gpu


def _case(B, S, D, V, dtype, seed, ignore_frac=0.1):
    g = torch.Generator().manual_seed(seed)
    h = torch.randn(B, S, D, generator=g).to(dtype)
    w = (torch.randn(V, D, generator=g) * 0.05).to(dtype)
    t = torch.randint(0, V, (B, S), generator=g)
    t[torch.rand(B, S, generator=g) < ignore_frac] = -100
    return h, w, t


@pytest.mark.parametrize("dtype,shape,chunk", [
    (torch.float32, (2, 300, 64, 1000), 128),    # ragged last chunk
    (torch.float32, (1, 50, 32, 1001), 4096),    # one chunk, V not a multiple of 8
    (torch.bfloat16, (2, 256, 128, 32000), 192),  # LM-head vocab
])
def test_chunked_cross_entropy(cuda, dtype, shape, chunk):
    from hydra_amd.kernels import fused_chunked_cross_entropy

    h, w, t = _case(*shape, dtype, seed=sum(shape))
    hd, wd = h.to(cuda).requires_grad_(), w.to(cuda).requires_grad_()
    loss = fused_chunked_cross_entropy(hd, wd, t.to(cuda), chunk_size=chunk)
    loss.backward(torch.tensor(0.5, device=cuda, dtype=dtype))
    ref, gh, gw = ofo.chunked_cross_entropy(h, w, t, grad_output=0.5)
    tol = 1e-5 if dtype == torch.float32 else 2e-2
    assert loss.dtype == dtype
    assert abs(loss.item() - ref.item()) / abs(ref.item()) < tol
    assert max_rel_err(hd.grad.cpu(), gh) < tol
    assert max_rel_err(wd.grad.cpu(), gw) < tol


def test_chunked_cross_entropy_edge_targets(cuda):
    """All targets ignored: loss 0, zero gradients.  Out-of-range targets are
    clamped into [0, V) (fused_ops.py:1407-1422)."""
    from hydra_amd.kernels import chunked_cross_entropy

    h, w, t = _case(1, 40, 32, 100, torch.float32, seed=2)
    hd, wd = h.to(cuda).requires_grad_(), w.to(cuda).requires_grad_()
    loss = chunked_cross_entropy(hd, wd, torch.full_like(t, -100).to(cuda), chunk_size=16)
    loss.backward()
    assert loss.item() == 0 and hd.grad.abs().max() == 0 and wd.grad.abs().max() == 0
    t[0, 3], t[0, 9] = 150, -5
    hd.grad = wd.grad = None
    loss = chunked_cross_entropy(hd, wd, t.to(cuda), chunk_size=16)
    loss.backward()
    ref, gh, gw = ofo.chunked_cross_entropy(h, w, t)
    assert abs(loss.item() - ref.item()) / abs(ref.item()) < 1e-5
    assert max_rel_err(hd.grad.cpu(), gh) < 1e-5 and max_rel_err(wd.grad.cpu(), gw) < 1e-5


@pytest.mark.parametrize("oob", [False, True])
def test_token_losses_from_hidden(cuda, oob):
    """compute_token_losses_from_hidden (loop.py:28-89) against the oracle,
    fp32 throughout (1e-5), token chunks with a ragged tail."""
    from hydra_amd.training import compute_token_losses_from_hidden

    h, w, t = _case(2, 150, 64, 3000, torch.bfloat16, seed=21)
    if oob:
        t[1, 7] = 3005
    got = compute_token_losses_from_hidden(h.to(cuda), w.to(cuda), t.to(cuda), token_chunk_size=128)
    ref = ofo.token_losses_from_hidden(h.float(), w.float(), t)
    assert got.dtype == torch.float32 and got.shape == (2, 150)
    assert max_rel_err(got.cpu(), ref) < 1e-5
    assert (got.cpu()[ref == 0] == 0).all()


@pytest.mark.parametrize("V", [1000, 1001, 32000])
@pytest.mark.parametrize("with_grad", [False, True])
def test_ce_rows_masked_logits(cuda, V, with_grad):
    """hydra_ce_rows on logits holding -inf (masked vocabulary entries): whole
    16-byte chunks and single entries.  Loss and gradient must be those of
    F.cross_entropy in fp64 (finite; masked entries get zero gradient)."""
    from hydra_amd import _lib

    rows = 6
    g = torch.Generator().manual_seed(V)
    x = torch.randn(rows, V, generator=g)
    x[0, :64] = -float("inf")          # leading chunks fully masked
    x[1, 8:16] = -float("inf")         # one 16-byte chunk (fp32: two)
    x[2, torch.randperm(V, generator=g)[: V // 3]] = -float("inf")
    x[3, V - 5:] = -float("inf")       # ragged tail
    t = torch.randint(0, V, (rows,), generator=g)
    for r in range(4):
        while torch.isinf(x[r, t[r]]):
            t[r] = (t[r] + 1) % V
    t[5] = -100
    xd, td = x.to(cuda), t.to(cuda)
    loss = torch.empty(rows, device=cuda)
    grad = torch.empty_like(xd) if with_grad else None
    scale = torch.full((1,), 0.25, device=cuda)
    _lib.call("hydra_ce_rows", xd.data_ptr(), rows, V, V, td.data_ptr(), -100, loss.data_ptr(), None,
              grad.data_ptr() if with_grad else None, V, scale.data_ptr() if with_grad else None,
              _lib.dtype_code(xd), _lib.stream(xd))
    x64 = x.double()
    ref = torch.nn.functional.cross_entropy(x64, t, ignore_index=-100, reduction="none")
    assert torch.isfinite(loss.cpu()).all()
    assert max_rel_err(loss.cpu(), ref) < 1e-5
    if with_grad:
        p = torch.softmax(x64, -1)
        gr = p.clone()
        valid = t != -100
        gr[valid, t[valid]] -= 1
        gr[~valid] = 0
        gr *= 0.25
        gc = grad.cpu()
        assert torch.isfinite(gc).all()
        assert max_rel_err(gc, gr) < 1e-5
        assert (gc[torch.isinf(x)] == 0).all()


@pytest.mark.parametrize("rows,V", [(3, 1), (5, 7), (4, 1000), (2, 8191), (3, 8192), (3, 16392), (2, 32768),
                                    (2, 40008), (3, 50257)])
def test_ce_grad_planes(cuda, rows, V):
    """hydra_ce_grad_planes at the edges of its row forms (registers, read
    twice, unaligned): both planes' sum against the fp64 gradient.  The planes
    carry 16 significant bits (2^-17 per value) of an fp32 value whose exponent
    argument is rounded at |x| 2^-24 (|x| <= 60 here): 2^-16 covers both."""
    from hydra_amd.kernels.fused_ops import _ce_grad_planes

    g = torch.Generator().manual_seed(V)
    x = torch.randn(rows, V, generator=g) * 5
    x[0, 0] = -float("inf") if V > 1 else 0.0
    t = torch.randint(0, V, (rows,), generator=g)
    t[-1] = -100
    scale = torch.tensor([0.37])
    got = _ce_grad_planes(x.to(cuda), t.to(cuda), -100, scale.to(cuda)).double().cpu()
    ref = torch.softmax(x.double(), 1)
    ref[torch.arange(rows), t.clamp(0)] -= 1
    ref = ref * 0.37
    ref[-1] = 0
    got = got[:rows] + got[rows:]
    assert got[-1].abs().max() == 0
    if V > 1:
        assert float((got - ref).norm() / ref.norm()) < 2.0 ** -16
    else:
        assert got.abs().max() < 1e-6


@pytest.mark.parametrize("rows,V", [(3, 1), (5, 7), (4, 1000), (2, 4099), (2, 8191), (3, 8193), (2, 16392), (2, 32767),
                                    (2, 32768)])
def test_ce_grad_planes_in_place(cuda, rows, V):
    """The planes in the logits' own memory, rows of whole 8-column pieces and
    ragged ones (whose padding holds NaNs beforehand); bound as above."""
    from hydra_amd.kernels.fused_ops import _ce_grad_planes_in_place

    g = torch.Generator().manual_seed(V)
    x = torch.randn(rows, V, generator=g) * 5
    t = torch.randint(0, V, (rows,), generator=g)
    t[-1] = -100
    logits = torch.full((rows, (V + 7) // 8 * 8), float("nan"), device=cuda)
    logits[:, :V] = x.to(cuda)
    got = _ce_grad_planes_in_place(logits, V, t.to(cuda), -100, torch.tensor([0.37], device=cuda)).double().cpu()
    ref = torch.softmax(x.double(), 1)
    ref[torch.arange(rows), t.clamp(0)] -= 1
    ref = ref * 0.37
    ref[-1] = 0
    got = got[0::2] + got[1::2]
    assert got[-1].abs().max() == 0
    if V > 1:
        assert float((got - ref).norm() / ref.norm()) < 2.0 ** -16
    else:
        assert got.abs().max() < 1e-6


@pytest.mark.parametrize("V", [1000, 1003])
def test_ce_grad_planes_of_infinite_gradients(cuda, V):
    """An infinite gradient is its first plane; inf - inf beside it would make
    NaN of the sum."""
    from hydra_amd.kernels.fused_ops import _ce_grad_planes

    x = torch.randn(2, V, generator=torch.Generator().manual_seed(1)).to(cuda)
    t = torch.tensor([3, 5], device=cuda)
    got = _ce_grad_planes(x, t, -100, torch.tensor([float("inf")], device=cuda)).float()
    want = torch.full((2, V), float("inf"), device=cuda)
    want[torch.arange(2, device=cuda), t] = -float("inf")
    assert torch.equal(got[:2] + got[2:], want)


@pytest.mark.parametrize("n,dim,V", [(70, 64, 33000), (33, 8, 4099), (1, 64, 40)])
def test_backward_of_odd_sizes(cuda, n, dim, V):
    """bf16 gradients over several chunks, rows longer than registers hold and
    ragged vocabularies, against fp64 of the same inputs: half an ulp of
    bf16, 2^-9, and the fp32 sums' rounding beside it."""
    from hydra_amd.kernels import chunked_cross_entropy

    g = torch.Generator().manual_seed(n)
    h, w = torch.randn(n, dim, generator=g).to(torch.bfloat16), (torch.randn(V, dim, generator=g) * 0.3).to(torch.bfloat16)
    t = torch.randint(0, V, (n,), generator=g)
    hd, wd = h.to(cuda).requires_grad_(), w.to(cuda).requires_grad_()
    chunked_cross_entropy(hd, wd, t.to(cuda), chunk_size=32).backward()
    h64, w64 = h.double().requires_grad_(), w.double().requires_grad_()
    torch.nn.functional.cross_entropy(h64 @ w64.t(), t).backward()
    for a, r in ((hd.grad, h64.grad), (wd.grad, w64.grad)):
        assert a.shape == r.shape
        assert float((a.double().cpu() - r).norm() / r.norm()) < 2.0 ** -8


@pytest.mark.parametrize("V", [32000, 4099, 40000])
def test_backward_holds_one_chunk_of_logits(cuda, V):
    """The bf16 backward's scratch at its peak: one chunk of fp32 logits (the
    gradient's planes in the same memory), the fp32 gradients and the product
    that is added to one of them, 16 bytes of [rows, dim] and 8 of [V, dim], and
    the returned gradients."""
    from hydra_amd.kernels import chunked_cross_entropy

    n, dim = 2048, 64
    g = torch.Generator(device=cuda).manual_seed(V)
    h = torch.randn(n, dim, device=cuda, generator=g).to(torch.bfloat16).requires_grad_()
    w = (torch.randn(V, dim, device=cuda, generator=g) * 0.05).to(torch.bfloat16).requires_grad_()
    t = torch.randint(0, V, (n,), device=cuda, generator=g)
    for _ in range(2):  # the GEMM library's own workspace comes with the first pass
        h.grad = w.grad = None
        loss = chunked_cross_entropy(h, w, t)
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        loss.backward()
        peak = torch.cuda.max_memory_allocated() - before
    logits = n * ((V + 7) // 8 * 8) * 4
    assert peak <= logits + 32 * n * dim + 10 * V * dim + (4 << 20), f"{peak / logits:.2f} chunks of logits"
