"""residual_norm at the widths where its lane split changes: rows of 1 to 513
16-byte chunks, which divide evenly over 4 to 64 lanes or do not, the widest a
wave holds (512) and the first past it, with row counts off the workgroups'.

h is exact (torch's own rounded adds).  y is one rounding of an fp32 value whose
relative error is at most (log2 dim + 8) 2^-24: half an ulp is 2^-9 of bf16
values and 2^-24 of fp32's, so 2^-8 and 2^-19 bound both."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("chunks", [1, 4, 5, 13, 17, 20, 33, 65, 96, 160, 192, 224, 257, 320, 512, 513])
def test_residual_norm_widths(cuda, chunks, dtype):
    from hydra_amd import _lib
    from hydra_amd.layers import residual_norm

    dim = chunks * (4 if dtype == torch.float32 else 8)
    g = torch.Generator().manual_seed(dim)
    for rows in (1, 13, 70):
        x, r = (torch.randn(rows, dim, generator=g).to(dtype).to(cuda) for _ in range(2))
        b1, b2 = ((0.1 * torch.randn(dim, generator=g)).to(dtype).to(cuda) for _ in range(2))
        w = (1 + 0.1 * torch.randn(dim, generator=g)).to(dtype).to(cuda)
        h, y = residual_norm(x, r=r, b1=b1, b2=b2, alpha=0.5, weight=w, norm=_lib.NORM_RMS, want_h=True)
        want = x + 0.5 * r + b1 + b2
        assert torch.equal(h, want)
        v = want.double()
        ref = v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + 1e-6) * w.double()
        u = 2.0 ** -19 if dtype == torch.float32 else 2.0 ** -8
        assert ((y.double() - ref).abs() <= u * ref.abs() + 2.0 ** -24).all(), rows
        _, a = residual_norm(x, r=r, b1=b1, b2=b2, alpha=0.5, weight=w, norm=_lib.NORM_ADA)
        # AdaRMSNorm in the input dtype: five roundings of half an ulp more
        assert ((a.double() - ref).abs() <= 6 * u * ref.abs() + 2.0 ** -24).all(), rows
