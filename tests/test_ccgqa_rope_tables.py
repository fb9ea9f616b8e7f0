"""Which RoPE tables the CCGQA prep kernel reads in place: whole rows one
after the other.  Every other form is converted to that first."""
from __future__ import annotations

import pytest
import torch


@pytest.mark.parametrize("form", ["whole", "batched", "bf16", "expanded", "slice", "transposed", "fp16"])
def test_tables_reach_the_kernel_as_whole_rows(form):
    from hydra_amd.attention.backends.ccgqa.ops import _rope_tables

    S, width = 5, 8
    full = torch.arange(2 * 16 * width, dtype=torch.float32).reshape(2, 16, width)
    cos, sin = full[0], full[1]
    if form == "batched":
        cos, sin = cos[None, None], sin[None, None]
    elif form in ("bf16", "fp16"):
        cos, sin = (t.to(torch.bfloat16 if form == "bf16" else torch.float16) for t in (cos, sin))
    elif form == "expanded":
        cos, sin = cos[:1].expand(16, width), sin[:1].expand(16, width)
    elif form == "slice":
        cos, sin = cos[:, :4], sin[:, :4]
    elif form == "transposed":
        cos, sin = cos.t().contiguous().t(), sin.t().contiguous().t()
    c, s, stride, flag = _rope_tables(cos, sin, S, True)
    in_place = form in ("whole", "batched", "bf16")
    assert (c.data_ptr() == cos.data_ptr()) == (s.data_ptr() == sin.data_ptr()) == in_place
    assert (flag != 0) == (form == "bf16")
    w = cos.shape[-1]
    assert stride == w and c.stride(-1) == 1 and c.stride(-2) == w
    assert c.dtype == (torch.bfloat16 if form == "bf16" else torch.float32)
    for got, want in ((c, cos), (s, sin)):
        got, want = got.reshape(-1, w)[:S], want.reshape(-1, w)[:S]
        assert torch.equal(got.float(), want.float())


@pytest.mark.parametrize("shape", [(4, 8), (1, 16, 8), (1, 1, 4, 8)])
def test_tables_that_do_not_cover_the_sequence_are_refused(shape):
    from hydra_amd.attention.backends.ccgqa.ops import _rope_tables

    with pytest.raises(ValueError, match="RoPE cache"):
        _rope_tables(torch.zeros(shape), torch.zeros(shape), 5, True)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("batched", [False, True])
def test_sine_tables_apart_from_the_cosines(dtype, batched):
    """The kernel walks both tables by one row stride: a sine table with too
    few rows or another width is refused, one with more rows is not."""
    from hydra_amd.attention.backends.ccgqa.ops import _rope_tables

    tables = [torch.zeros(n, w, dtype=dtype) for n, w in ((6, 8), (4, 8), (6, 4), (9, 8))]
    cos, short, narrow, longer = (t[None, None] if batched else t for t in tables)
    for sin in (short, narrow):
        with pytest.raises(ValueError, match="RoPE"):
            _rope_tables(cos, sin, 5, True)
    _rope_tables(cos, longer, 5, True)
