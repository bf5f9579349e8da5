"""Forward products of few rows (gr_gemm_nt's 64-row tiles): every column range and
alignment at the tile edges, against float64, and bit for bit the rows of a call
large enough for the large tiles."""

from __future__ import annotations

import pytest
import torch

from grinnder_amd.dense import gemm_nt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 16, 17, 33, 48, 49, 64, 65, 256])
@pytest.mark.parametrize("k", [3, 64, 100, 272])
@pytest.mark.parametrize("rows", [1, 64, 65, 1000])
def test_few_rows_match_float64_and_large_tiles(gpu, n, k, rows):
    g = torch.Generator().manual_seed(n * 1000 + k)
    a, b = torch.randn(65601, k, generator=g), torch.randn(n, k, generator=g)
    bias = torch.randn(n, generator=g)
    a_d, b_d, bias_d = a.to(gpu), b.to(gpu), bias.to(gpu)
    buf = torch.full((rows + 1, n), 7.0, device=gpu)
    out = gemm_nt(a_d[:rows], b_d, bias_d, out=buf[:rows])
    assert bool((buf[rows] == 7.0).all())
    x, w = a[:rows].double(), b.double()
    # k products and the bias summed in fp32, in any order.
    bound = (k + 1) * 2.0 ** -24 * (x.abs() @ w.abs().t() + bias.abs())
    assert bool(((out.cpu().double() - (x @ w.t() + bias)).abs() <= bound).all())
    if not (k % 32 == 0 and k <= 256 and n > 32 and n % 4 == 0):  # else the resident form
        assert torch.equal(gemm_nt(a_d, b_d, bias_d)[:rows], out)
