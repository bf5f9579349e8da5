"""The dense products on split operands (csrc/gemm_bf3.h): every tile shape at
its edges, unaligned and strided operands, infinities and NaN, and the error
and bias against float64."""

from __future__ import annotations

import pytest
import torch

from grinnder_amd import _lib
from grinnder_amd.dense import gemm_split, gemm_tn, pad_columns, pad_layer, pad_layer_grad

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    return torch.device("cuda", 0)


def _randn(*shape, seed, dev):
    g = torch.Generator(device=dev).manual_seed(seed)
    return torch.randn(*shape, device=dev, generator=g)


def gemm_nt_split(a, b, bias=None, out=None, rows_k=False):
    """gr_gemm_nt_split with a bias and a strided output."""
    n = b.size(1 if rows_k else 0)
    if out is None:
        out = torch.empty(a.size(0), n, device=a.device)
    _lib.call("gr_gemm_nt_split", a.data_ptr(), a.stride(0), b.data_ptr(), b.stride(0),
              int(rows_k), a.size(0), n, a.size(1), _lib.ptr(bias), out.data_ptr(),
              out.stride(0), _lib.stream_handle())
    return out


def _rel(c, ref):
    return float((c.double() - ref).norm() / ref.norm())


def _bound(k):
    """Relative 2-norm error of a product over k: a rounding of 2^-24 at each
    of at most k additions, random in sign, is at most 2^-24 sqrt(k) of the
    result; the dropped piece products are 2^-26 of each product."""
    return 2.0 ** -24 * (k ** 0.5 + 2)


# Rows and columns around each tile (128 x 32, 128 x 64, 128 x 128, 128 x 256,
# 256 x 256, and 64 x 32 / 64 x 64 for few rows), K around the 16-k chunk.
@pytest.mark.parametrize("m,n,k", [
    (63, 31, 15), (64, 32, 16), (65, 33, 17), (1, 1, 4), (32767, 32, 48), (32897, 20, 100),
    (32897, 47, 33), (33000, 64, 16), (33000, 65, 64), (33100, 129, 31), (5000, 128, 300),
    (66000, 256, 512), (131073, 257, 528), (262145, 256, 128), (262145, 132, 140), (300, 500, 1)])
@pytest.mark.parametrize("pad", [0, 1])
def test_gemm_nt_split_tiles_match_fp64(gpu, m, n, k, pad):
    """pad = 1: rows of A and B one float apart from 16-byte alignment."""
    a = _randn(m, k + pad, seed=1, dev=gpu)[:, pad:]
    b = _randn(n, k + pad, seed=2, dev=gpu)[:, pad:]
    bias = _randn(n, seed=3, dev=gpu)
    out = torch.full((m + 1, n + 2 * pad), 7.0, device=gpu)
    c = gemm_nt_split(a, b, bias, out=out[:m, pad:pad + n])
    ref = a.double() @ b.double().t() + bias.double()
    assert _rel(c, ref) <= _bound(k)
    # B as [K, N] gives the same sums in the same order.
    bt = torch.zeros(k, n + pad, device=gpu)[:, pad:]
    bt.copy_(b.t())
    assert torch.equal(gemm_nt_split(a, bt, bias, rows_k=True), c)
    assert torch.equal(gemm_split(a, bt) + bias, c)
    assert bool((out[m] == 7.0).all())  # no row past the last
    if pad:
        assert bool((out[:, 0] == 7.0).all()) and bool((out[:, -1] == 7.0).all())


@pytest.mark.parametrize("m,n,k", [
    (256, 256, 40_000), (255, 257, 33_001), (100, 256, 30_000), (129, 128, 33_007),
    (300, 64, 66_000), (47, 256, 40_001), (20, 300, 50_000), (32, 32, 20_000), (64, 128, 1000),
    (1, 1, 17), (5, 3, 1), (256, 1024, 20_000)])
@pytest.mark.parametrize("pad", [0, 3])
def test_gemm_tn_tiles_match_fp64(gpu, m, n, k, pad):
    a = _randn(k, m + pad, seed=4, dev=gpu)[:, pad:]
    b = _randn(k, n + pad, seed=5, dev=gpu)[:, pad:]
    c = gemm_tn(a, b)
    ref = a.double().t() @ b.double()
    assert _rel(c, ref) <= _bound(k)


@pytest.mark.parametrize("shape", [(300, 70, 40), (40_000, 256, 64), (70, 20, 256)])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3.4e38])
def test_products_keep_infinities_and_nan(gpu, shape, value):
    """An infinite, NaN or nearly largest operand gives what fp32 arithmetic
    gives: the rows (columns) it meets are inf, NaN or finite as in torch, and
    every other output is untouched by it."""
    m, n, k = shape
    a, b = _randn(m, k, seed=6, dev=gpu), _randn(n, k, seed=7, dev=gpu) * 0.01
    clean = gemm_nt_split(a, b)
    a[m // 2, k // 3] = value
    c, ref = gemm_nt_split(a, b), a.double() @ b.double().t()
    row = torch.zeros(m, dtype=torch.bool, device=gpu)
    row[m // 2] = True
    assert _rel(c[~row], ref[~row]) <= _bound(k) and _rel(clean[~row], ref[~row]) <= _bound(k)
    got, want = c[row].double(), ref[row].float().double()
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.isinf(), want.isinf())
    fin = want.isfinite()
    assert torch.allclose(got[fin], want[fin], rtol=1e-5)
    assert torch.equal(got[want.isinf()], want[want.isinf()])
    # The weight gradient's product of the same operands.
    x = a.t().contiguous()  # [k, m]: the value sits in one row and column
    w = _randn(k, n, seed=8, dev=gpu) * 0.01
    ct, rt = gemm_tn(x, w), x.double().t() @ w.double()
    assert _rel(ct[~row], rt[~row]) <= _bound(k)
    want = rt[row].float()
    assert torch.equal(ct[row].isnan(), want.isnan())
    assert torch.equal(ct[row][want.isinf()], want[want.isinf()])


def test_products_hold_small_and_large_magnitudes(gpu):
    """Scaling the operands by powers of two scales the result: the pieces
    keep all 24 bits from 1e-30 to 1e30."""
    a, b = _randn(500, 96, seed=9, dev=gpu), _randn(80, 96, seed=10, dev=gpu)
    base = gemm_nt_split(a, b)
    for e in (-100, -60, 60, 100):
        got = gemm_nt_split(a * 2.0 ** e, b * 2.0 ** (-e // 2))
        assert torch.equal(got, base * 2.0 ** (e + -e // 2))


@pytest.mark.parametrize("e", [-109, -112, -118, -125])
def test_products_of_operands_below_the_exact_range(gpu, e):
    """Operands below 2^-109 keep fewer than 24 bits: a bf16 piece ends at
    2^-133, so each operand is off by at most 2^-134 and a sum over k by
    2^-134 times the other operand's magnitudes (and its own rounding)."""
    k = 96
    a, b = _randn(300, k, seed=15, dev=gpu) * 2.0 ** e, _randn(70, k, seed=16, dev=gpu) * 2.0 ** 60
    ref = a.double() @ b.double().t()
    allowed = 2.0 ** -134 * b.double().abs().sum(1) + _bound(k) * ref.norm() / ref.numel() ** 0.5 * 8
    assert bool(((gemm_nt_split(a, b).double() - ref).abs() <= allowed).all())
    x, w = a.t().contiguous(), b.t().contiguous()
    assert bool(((gemm_tn(x, w).double() - ref).abs() <= allowed).all())


def test_products_error_and_bias_against_fp64(gpu):
    """No further from float64 than torch's fp32 product, and without the
    matrix core's bias: the mean error is far below the rms error, so sums
    over rows do not collect it."""
    a, b = _randn(40_000, 256, seed=11, dev=gpu), _randn(256, 256, seed=12, dev=gpu)
    ref = a.double() @ b.double().t()
    e = gemm_nt_split(a, b).double() - ref
    torch_rms = float(((a @ b.t()).double() - ref).pow(2).mean().sqrt())
    rms = float(e.pow(2).mean().sqrt())
    assert rms <= 1.05 * torch_rms
    # 10M errors: a random mean is below 1e-3 of their rms.
    assert abs(float(e.mean())) <= 3e-3 * rms
    x, w = _randn(400_000, 128, seed=13, dev=gpu), _randn(400_000, 64, seed=14, dev=gpu)
    ref = x.double().t() @ w.double()
    e = gemm_tn(x, w).double() - ref
    assert float(e.norm() / ref.norm()) <= 1.05 * _rel(x.t() @ w, ref)


@pytest.mark.parametrize("rows,cols,width", [(1, 1, 4), (3, 47, 48), (5000, 19, 20), (70, 64, 64),
                                             (0, 5, 8), (2, 3, 16)])
def test_pad_columns(gpu, rows, cols, width):
    """Zero-padded copies equal torch's, strided rows included, and the padded
    parameters' gradients are the slices."""
    a = _randn(rows, cols + 3, seed=21, dev=gpu)[:, 1:1 + cols]
    v = _randn(1, 1, cols, seed=22, dev=gpu)
    assert torch.equal(pad_columns(a, width), torch.nn.functional.pad(a, (0, width - cols)))
    assert torch.equal(pad_layer(None, width, v)[0],
                       torch.nn.functional.pad(v, (0, width - cols)))
    w = _randn(cols, 7, seed=23, dev=gpu).requires_grad_(True)
    b = _randn(cols, seed=24, dev=gpu).requires_grad_(True)
    wp, none, bp = pad_layer_grad(w, width, None, b)
    assert none is None and torch.equal(wp[:cols], w) and not bool(wp[cols:].any())
    assert torch.equal(bp[:cols], b) and not bool(bp[cols:].any())
    g = _randn(width, 7, seed=25, dev=gpu)
    (wp * g).sum().backward()
    assert torch.equal(w.grad, g[:cols]) and (b.grad is None or not bool(b.grad.any()))
