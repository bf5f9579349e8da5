"""Attention logits of several heads (gr_gat_scores) in every row layout: rows
side by side in a wavefront, one row of one to four chunks, heads of one lane to a
whole wavefront, and the widths that keep the loop over the heads, against
float64, with rows and destinations around the steps' edges."""

from __future__ import annotations

import pytest
import torch

from grinnder_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,C", [(2, 4), (3, 8), (8, 8), (16, 4), (3, 32), (8, 32), (5, 64),
                                 (2, 128), (2, 256), (3, 256), (16, 64), (4, 12), (2, 512)])
@pytest.mark.parametrize("rows,dst", [(1, 0), (3, 3), (17, 16), (1031, 517)])
@pytest.mark.parametrize("pad,offset", [(0, 0), (4, 0), (3, 0), (0, 1)])
def test_scores_match_float64(gpu, H, C, rows, dst, pad, offset):
    """pad: floats between rows; offset: floats past 16-byte alignment."""
    g = torch.Generator().manual_seed(H * 1000 + C + rows)
    ld = H * C + pad
    buf = torch.full((offset + rows * ld,), float("nan"))
    hs = torch.as_strided(buf, (rows, H * C), (ld, 1), offset)
    hs.copy_(torch.randn(rows, H * C, generator=g))
    a_s, a_d = (torch.randn(H, C, generator=g) for _ in range(2))
    dev = buf.to(gpu)
    as_d, ad_d = a_s.to(gpu), a_d.to(gpu)
    s = torch.full((rows + 1, H), 7.0, device=gpu)
    d = torch.full((dst + 1, H), 7.0, device=gpu)
    _lib.call("gr_gat_scores", dev.data_ptr() + 4 * offset, ld, rows, dst, H, C, as_d.data_ptr(),
              ad_d.data_ptr(), s.data_ptr(), d.data_ptr(), _lib.stream_handle())
    x = hs.double().view(rows, H, C)
    for got, a, n in ((s, a_s, rows), (d, a_d, dst)):
        # A sum of C products in any order is within C roundings of their magnitudes.
        bound = C * 2.0 ** -24 * (x[:n] * a.double()).abs().sum(2)
        err = (got[:n].cpu().double() - (x[:n] * a.double()).sum(2)).abs()
        assert bool((err <= bound).all())
        assert bool((got[n] == 7.0).all())  # nothing past the last row
