"""Several attention heads in one pass (csrc/gat_heads.hip) against the oracle:
every lane layout (heads and channels around powers of two, rows at any 4-byte
boundary, one to eight chunks a row, edge slots), split and empty rows, and the
forward without a backward."""

from __future__ import annotations

import pytest
import torch

import oracle
from grinnder_amd.aggregation import _gat_heads_ok, gat_attention, gat_scores
from grinnder_amd.data.adjacency import Adjacency
from grinnder_amd.nn import GAT
from tests.graphs import TOL, max_abs_norm_err, random_bipartite

pytestmark = pytest.mark.gpu

CASES = [
    # (heads, channels, one-pass kernels)
    (2, 1, True), (16, 1, True), (2, 2, True), (3, 5, True), (5, 16, True), (7, 12, True),
    (8, 8, True), (8, 23, True), (8, 32, True), (2, 116, True), (2, 69, True), (4, 49, True),
    (2, 256, True), (2, 512, True), (2, 129, True), (4, 130, True), (16, 64, True),
    (15, 68, True), (6, 6, True), (3, 257, True), (2, 511, True), (5, 3, True), (16, 63, True),
    # one head: 36..64 channels
    (1, 32, False), (1, 36, True), (1, 48, True), (1, 64, True), (1, 68, False),
]


def _inputs(H, C, concat, rows=260, sources=400, seg_len=64):
    rowptr, col, val = random_bipartite(rows, sources, 9, seed=H * 7 + C, long_rows=2,
                                        long_len=300)
    adj = Adjacency(rowptr, col, val, (rows, sources), seg_len=seg_len)
    g = torch.Generator().manual_seed(H * 100 + C)
    hs = torch.randn(sources, H * C, generator=g)
    att_src = torch.randn(1, H, C, generator=g) * C ** -0.5
    att_dst = torch.randn(1, H, C, generator=g) * C ** -0.5
    width = H * C if concat else C
    return rowptr, col, adj, hs, att_src, att_dst, torch.randn(width, generator=g), \
        torch.randn(rows, width, generator=g)


@pytest.mark.parametrize("H,C,one_pass", CASES)
@pytest.mark.parametrize("concat,offset", [(True, 0), (True, 1), (True, 2), (False, 0)])
def test_heads_match_oracle(gpu, H, C, one_pass, concat, offset):
    """offset: hs starts that many floats past 16-byte alignment."""
    rowptr, col, adj, hs, a_s, a_d, bias, gy = _inputs(H, C, concat)
    buf = torch.empty(hs.numel() + offset, device=gpu)
    hs_d = buf[offset:].view(hs.shape)
    hs_d.copy_(hs)
    if offset == 0:
        assert _gat_heads_ok(hs_d, H, C) == one_pass
    hs_d = hs_d.detach().requires_grad_(True)
    as_d, ad_d, b_d = (t.to(gpu).requires_grad_(True) for t in (a_s, a_d, bias))
    y = gat_attention(hs_d, adj, as_d, ad_d, b_d, H, C, concat)
    y.backward(gy.to(gpu))
    ref, alpha, tpre = oracle.gat_forward(rowptr, col, hs, H, C, a_s, a_d, bias, concat)
    dhs, das, dad, db = oracle.gat_backward(rowptr, col, hs, H, C, a_s, a_d, concat, alpha, tpre,
                                            gy)
    assert max_abs_norm_err(y, ref) <= TOL
    assert max_abs_norm_err(hs_d.grad, dhs) <= TOL
    assert max_abs_norm_err(as_d.grad.reshape(-1), torch.as_tensor(das).reshape(-1)) <= TOL
    assert max_abs_norm_err(ad_d.grad.reshape(-1), torch.as_tensor(dad).reshape(-1)) <= TOL
    assert max_abs_norm_err(b_d.grad, db) <= TOL
    with torch.no_grad():
        again = gat_attention(hs_d, adj, as_d, ad_d, b_d, H, C, concat)
    if one_pass and offset == 0:  # the same kernel without the backward's state
        assert torch.equal(again, y.detach())
    else:
        assert max_abs_norm_err(again, y.detach()) <= TOL


@pytest.mark.parametrize("H,C", [(8, 8), (2, 64), (4, 130)])
def test_heads_extreme_logits(gpu, H, C):
    """Logits of several hundred keep the softmax finite (the running maximum
    is taken off before the exponential), rows without edges give the bias,
    and a NaN source reaches only the rows that read it."""
    rowptr, col, adj, hs, a_s, a_d, bias, _ = _inputs(H, C, True)
    out = gat_attention((hs * 200).to(gpu), adj, a_s.to(gpu), a_d.to(gpu), bias.to(gpu), H, C)
    ref = oracle.gat_forward(rowptr, col, hs * 200, H, C, a_s, a_d, bias, True)[0]
    assert max_abs_norm_err(out, ref) <= 1e-4  # a logit of 1e3 has 6e-5 of rounding in it
    empty = rowptr[1:] == rowptr[:-1]
    assert bool(empty.any())
    assert torch.equal(out.cpu()[empty], bias.expand(int(empty.sum()), -1))
    bad = hs.clone()
    bad[399] = float("nan")
    reads = torch.zeros(260, dtype=torch.bool)
    rows = torch.repeat_interleave(torch.arange(260), rowptr[1:] - rowptr[:-1])
    reads[rows[col == 399]] = True
    got = gat_attention(bad.to(gpu), adj, a_s.to(gpu), a_d.to(gpu), bias.to(gpu), H, C).cpu()
    assert bool(got[~reads].isfinite().all()) and bool(got[reads].isnan().all())


@pytest.mark.parametrize("H,C", [(3, 12), (7, 20), (8, 27), (4, 36), (2, 69), (5, 3), (3, 5),
                                 (4, 130), (3, 341), (8, 8)])
@pytest.mark.parametrize("head", [0, -1])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
def test_a_nonfinite_gradient_stays_in_its_head(gpu, H, C, head, value):
    """An infinite or NaN output gradient of one head leaves the other heads'
    gradients as they were, bit for bit, also where lanes of a head hold
    nothing (they read head 0's first vector) or share features with a
    neighbour; in its own head NaN appears where float64 gives it."""
    rows = 260
    rowptr, col, adj, hs, a_s, a_d, _, gy = _inputs(H, C, True)
    head = head % H
    bad = gy.view(rows, H, C).clone()
    if head == 0:
        bad[::9, 0, 0] = value
    else:
        bad[::9, head, C - 1] = value  # a shared vector's part when C % 4 != 0
    bad = bad.view(rows, H * C)

    def grads(g):
        t = [x.to(gpu).requires_grad_(True) for x in (hs, a_s, a_d)]
        y = gat_attention(t[0], adj, t[1], t[2], None, H, C, True)
        return [x.reshape(-1, H, C).cpu() for x in torch.autograd.grad(y, t, g.to(gpu))]

    clean, got = grads(gy), grads(bad)
    others = [h for h in range(H) if h != head]
    for a, b in zip(got, clean):
        assert torch.equal(a[:, others], b[:, others])
    # The head itself, in float64 and the kernels' order: c = <G, O>, edge
    # gradients alpha (<G, Hs> - c).  Rows past the destinations, which get no
    # part from a destination's own logit.
    o, alpha, tpre = oracle.gat_forward(rowptr, col, hs, H, C, a_s, a_d, None, True)
    row = torch.repeat_interleave(torch.arange(rows), rowptr[1:] - rowptr[:-1])
    g = bad.view(rows, H, C)[:, head].double()
    h64 = hs.view(-1, H, C)[:, head].double()
    c = (g * torch.as_tensor(o).view(rows, H, C)[:, head]).sum(1)
    alpha, slope = (torch.as_tensor(t)[:, head] for t in (alpha, tpre))
    ge = alpha * ((g[row] * h64[col]).sum(1) - c[row])
    ds = torch.zeros(hs.size(0), dtype=torch.float64)
    ds.index_add_(0, col, torch.where(slope > 0, ge, 0.2 * ge))
    want = torch.zeros_like(h64).index_add_(0, col, alpha[:, None] * g[row])
    want += ds[:, None] * a_s[0, head].double()
    assert torch.equal(got[0][rows:, head].isnan(), want[rows:].isnan())
    assert bool(want[rows:].isnan().any()) and not bool(want[rows:].isnan().all())


@pytest.mark.parametrize("H,C", [(8, 8), (2, 256), (1, 48)])
def test_backward_when_only_the_scores_ask_for_a_gradient(gpu, H, C):
    """Frozen rows and parameters with precomputed scores that require a
    gradient: the backward runs and gives the scores none, and the gradients
    of a row leaf beside such scores are those with detached ones."""
    _, _, adj, hs, a_s, a_d, _, gy = (t if not torch.is_tensor(t) else t.to(gpu)
                                      for t in _inputs(H, C, True))
    s, d = gat_scores(hs, a_s, a_d, H, C, gy.size(0))
    s, d = s.requires_grad_(True), d.requires_grad_(True)
    y = gat_attention(hs, adj, a_s, a_d, None, H, C, scores=(s, d))
    assert y.requires_grad
    y.backward(gy)
    assert s.grad is None and d.grad is None
    leaf = hs.clone().requires_grad_(True)
    got = [torch.autograd.grad(gat_attention(leaf, adj, a_s, a_d, None, H, C, scores=sc), leaf,
                               gy)[0] for sc in ((s, d), (s.detach(), d.detach()))]
    assert torch.equal(got[0], got[1])


@pytest.mark.parametrize("heads,C,norm,last", [
    (8, 32, False, False), (8, 32, True, False), (1, 48, True, False), (1, 47, False, True),
    (1, 256, True, False), (1, 100, False, False), (1, 100, True, False), (1, 20, False, True),
    (16, 8, False, False)])
def test_kept_floats_covers_what_a_layers_graph_holds(gpu, heads, C, norm, last):
    """The floats that a trainer counts for a kept forward graph against the
    device memory it holds: never less, beyond the allocator's rounding, and
    not a third more."""
    E, B = 200_000, 160_000
    g = torch.Generator().manual_seed(C)
    adj = Adjacency(torch.arange(B + 1) * 4, torch.randint(0, E, (4 * B,), generator=g), None,
                    (B, E))
    model = (GAT(4, 16, C, 2, heads=1, dropout=0.0) if last else
             GAT(8, C, 4, 2, heads=heads, dropout=0.0, norm=norm)).to(gpu).train()
    layer = int(last)
    z = torch.randn(E, model.projected_width(layer), device=gpu)
    z[:, heads * C:] = 0.0
    s, d = model.projected_scores(layer, z)
    z.requires_grad_(True)
    model.forward_projected(layer, z, adj, scores=(s, d[:B]))  # builds the plan
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    out = model.forward_projected(layer, z, adj, scores=(s, d[:B]))
    held = torch.cuda.memory_allocated() - before + 4 * (z.numel() + s.numel())
    assert out.requires_grad
    per_row, per_out, per_edge = model.kept_floats(layer)
    count = 4 * (E * per_row + B * per_out + 4 * B * per_edge)
    print(f"held {held / 1e6:.1f} MB, counted {count / 1e6:.1f} MB", flush=True)
    assert held <= count + (8 << 20)  # the allocator leaves up to 1 MB at a large tensor's end
    assert count <= 4 / 3 * held
