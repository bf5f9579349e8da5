"""The masked loss's gradient at the edges of its kernels: class counts around
the narrow form's limits and its 16-byte pieces, rows around a workgroup's 256,
no, some and only train rows, and the mean's and sum's scale; a mask changed
before the backward, a batched and a twice differentiated scale."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from grinnder_amd import _lib
from grinnder_amd.loss import mask_codes, masked_cross_entropy
from tests.graphs import TOL, max_abs_norm_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("classes", [1, 2, 3, 4, 5, 10, 16, 17, 33, 47, 49, 61, 63, 64, 65, 130, 1000])
@pytest.mark.parametrize("rows", [1, 255, 257, 1500])
@pytest.mark.parametrize("share", [0.0, 0.5, 1.0])
def test_masked_loss_gradient(gpu, rows, classes, share):
    g = torch.Generator(device=gpu).manual_seed(rows + classes)
    x = (3 * torch.randn(rows, classes, device=gpu, generator=g)).requires_grad_(True)
    y = torch.randint(0, classes, (rows,), device=gpu, generator=g)
    train = torch.rand(rows, device=gpu, generator=g) < share
    codes = mask_codes(train, ~train)
    # A buffer of NaN where the gradient will be allocated: unwritten rows show.
    torch.full((rows, classes), float("nan"), device=gpu)
    for reduction, scale in (("mean", 1.0), ("sum", 0.25)):
        loss, stats = masked_cross_entropy(x, y, codes, reduction)
        (got,) = torch.autograd.grad(loss * scale, x)
        ref = x.detach().double().requires_grad_(True)
        n = int(train.sum())
        want = torch.zeros_like(ref)
        if n:
            out = F.cross_entropy(ref[train], y[train], reduction=reduction) * scale
            (want,) = torch.autograd.grad(out, ref)
        assert max_abs_norm_err(got, want) <= TOL
        assert not bool(got[~train].any()) and int(stats[0]) == n


def test_backward_of_a_changed_mask_and_other_scales(gpu):
    x = torch.randn(300, 47, device=gpu, requires_grad=True)
    y = torch.randint(0, 47, (300,), device=gpu)
    train = torch.arange(300, device=gpu) % 3 == 0
    codes = mask_codes(train)
    loss, _ = masked_cross_entropy(x, y, codes, "mean")
    codes.zero_()
    (want,) = torch.autograd.grad(F.cross_entropy(x[train], y[train]), x)
    (got,) = torch.autograd.grad(loss, x, retain_graph=True)
    assert max_abs_norm_err(got, want) <= TOL
    (got,) = torch.autograd.grad(loss, x, torch.tensor([1.0, -2.0], device=gpu),
                                 is_grads_batched=True, retain_graph=True)
    assert max_abs_norm_err(got, torch.stack((want, -2 * want))) <= TOL
    a = torch.tensor(3.0, device=gpu, requires_grad=True)
    (got,) = torch.autograd.grad(loss * a, x, create_graph=True)
    (da,) = torch.autograd.grad(got.sum(1)[0] + got[0, 0], a)  # d(a * g)/da = g
    assert max_abs_norm_err(da, want.sum(1)[0] + want[0, 0]) <= TOL


@pytest.mark.parametrize("classes", [1, 3, 4, 16, 19, 33, 47, 64, 65, 300])
@pytest.mark.parametrize("extra", [0, 4])
def test_forward_entry_writes_every_gradient_row(gpu, classes, extra):
    """gr_xent_forward, the entry for a caller that scales the gradient itself,
    writes 0 on rows outside the train set (and on train rows of a label out
    of range) whatever the workspace's size past the 7 doubles a workgroup
    that it asks for; gr_xent_forward_train leaves those rows alone and gives
    the same values on the others."""
    rows, ldg, nan = 700, classes + 1, float("nan")
    x = torch.randn(rows, classes, device=gpu)
    y = torch.randint(0, classes, (rows,), device=gpu)
    train = torch.rand(rows, device=gpu) < 0.5
    y[::50] = classes  # out of range
    codes = mask_codes(train, ~train)
    n = (rows + 255) // 256
    ws = torch.empty(n * (7 + extra), dtype=torch.float64, device=gpu)
    loss, stats = torch.empty((), device=gpu), torch.empty(6, dtype=torch.int64, device=gpu)
    lse = torch.empty(rows, device=gpu)
    grad, part = (torch.full((rows, ldg), nan, device=gpu) for _ in range(2))
    _lib.call("gr_xent_forward", x.data_ptr(), classes, rows, classes, y.data_ptr(),
              codes.data_ptr(), 0, lse.data_ptr(), grad.data_ptr(), ldg, loss.data_ptr(),
              stats.data_ptr(), ws.data_ptr(), ws.numel(), _lib.stream_handle())
    ok = train & (y < classes)
    want = torch.softmax(x.double(), 1)
    want[ok] -= F.one_hot(y[ok], classes).double()
    want[~ok] = 0.0
    got = grad[:, :classes]
    assert max_abs_norm_err(got, want) <= TOL
    assert not bool(got[~ok].any()) and bool(grad[:, classes].isnan().all())
    assert max_abs_norm_err(lse, torch.logsumexp(x.double(), 1)) <= TOL
    bits = torch.zeros(4 * n, dtype=torch.int64, device=gpu)
    _lib.call("gr_xent_forward_train", x.data_ptr(), classes, rows, classes, y.data_ptr(),
              codes.data_ptr(), 0, part.data_ptr(), ldg, bits.data_ptr(), loss.data_ptr(),
              stats.data_ptr(), ws.data_ptr(), 7 * n, _lib.stream_handle())
    assert torch.equal(part[train, :classes], got[train]) and bool(part[~train].isnan().all())
    r = torch.arange(rows, device=gpu)
    assert torch.equal((bits[r // 64] >> (r % 64)) & 1, train.long())
