"""The work this framework does for its users, as cases that can be timed and checked.

Every case goes through the public entry points: a model's layer (forward_layer) forward
and backward on one partition's adjacency, a whole model's inference, the masked loss,
or a Trainer epoch.  Graphs are seeded power-law graphs (a few hub rows and columns, most
rows short), features are what a layer meets: normal inputs whose columns have their own means,
ReLU- or ELU-shaped hidden activations, output gradients with column means (as a loss
gives).  All arithmetic is fp32, the framework's only feature type.

- listed(): the fixed cases; draw(rng): one more of the same ranges.
- prepare(case, seed): model, graph plans and inputs on the GPU; run(state): one pass.
- work(case): the bytes and operations a pass cannot do without.
- tolerance(case), exact(case, seed): how far two correct fp32 results may differ, and the
  result in 64 bits by plain torch.
"""

import torch
import torch.nn.functional as F

from grinnder_amd.config import GriNNderConfig
from grinnder_amd.data.adjacency import Adjacency
from grinnder_amd.data.partition import build_partitioned_graph
from grinnder_amd.engine.trainer import Trainer
from grinnder_amd.loss import mask_codes, masked_cross_entropy
from grinnder_amd.nn import GAT, GCN

DEV = "cuda:0"


# ------------------------------------------------------------------- the cases


def listed():
    return [
        # The smallest training step: the plumbing configuration (10k nodes, 128 -> 64 -> 10,
        # two partitions).  Launches and host work set its time.
        dict(name="epoch_gcn_10k_p2", kind="epoch", flow="auto", nodes=10_000, edges=50_000,
             parts=2, din=128, hidden=64, classes=10, layers=2),
        # The headline model (3-layer GCN, 100 -> 256 -> 256 -> 47, LayerNorm) on one
        # partition of a mid-size graph that stays in HBM.
        dict(name="epoch_gcn_150k", kind="epoch", flow="auto", nodes=150_000,
             edges=1_500_000, parts=1, din=100, hidden=256, classes=47, layers=3),
        # The same model trained the way the reference does it: features and gradients in
        # pinned host memory, halo rows gathered and gradients scattered over the host link.
        dict(name="epoch_gcn_30k_p4_host", kind="epoch", flow="off", nodes=30_000,
             edges=300_000, parts=4, din=100, hidden=256, classes=47, layers=3),
        # A hidden GCN layer with LayerNorm, forward and backward, on one partition and its
        # halo: the layer most of a training run is spent in.
        dict(name="gcn_hidden_norm", kind="gcn", rows=400_000, sources=1_000_000,
             edges=16_000_000, din=256, dout=256, last=False, norm=True, xgrad=True),
        # A wide input layer without LayerNorm (the model's default), whose input is data
        # and takes no gradient: the dense products outweigh the aggregation.
        dict(name="gcn_wide_input", kind="gcn", rows=100_000, sources=250_000,
             edges=2_000_000, din=1024, dout=256, last=False, norm=False, xgrad=False),
        # The output layer: 47 classes, an odd width, from 256 channels.
        dict(name="gcn_output_47", kind="gcn", rows=200_000, sources=200_000,
             edges=5_000_000, din=256, dout=47, last=True, norm=True, xgrad=True),
        # A hidden GAT layer with the model's default of 8 heads, no norm.
        dict(name="gat_8heads", kind="gat", rows=100_000, sources=200_000,
             edges=4_000_000, din=256, heads=8, channels=32, last=False, norm=False,
             xgrad=True),
        # A hidden GAT layer of one 256-wide head with LayerNorm (the 10M-node benchmark's
        # layer) on a partition with a large halo.
        dict(name="gat_1head_norm", kind="gat", rows=60_000, sources=250_000,
             edges=2_000_000, din=256, heads=1, channels=256, last=False, norm=True,
             xgrad=True),
        # The GAT output layer after 8 heads of 32: 47 classes, one head.
        dict(name="gat_output_47", kind="gat", rows=100_000, sources=100_000,
             edges=2_000_000, din=256, heads=1, channels=47, last=True, norm=False,
             xgrad=True),
        # Inference with the plumbing configuration: a handful of short launches.
        dict(name="infer_gcn_10k", kind="infer", model="gcn", nodes=10_000, edges=110_000,
             din=128, hidden=64, heads=1, classes=10, layers=2, norm=True),
        # Inference with the default GAT (8 heads of 8) on a small graph.
        dict(name="infer_gat_50k", kind="infer", model="gat", nodes=50_000, edges=1_000_000,
             din=256, hidden=8, heads=8, classes=10, layers=2, norm=False),
        # The loss of a large graph's logits: masked cross entropy, accuracy counts and the
        # logits' gradient.
        dict(name="loss_1m_47", kind="loss", rows=1_000_000, classes=47),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["epoch", "gcn", "gcn", "gcn", "gat", "gat", "gat", "gat", "infer",
                       "infer", "loss"])
    if kind == "epoch":
        flow = rng.choice(["auto", "auto", "off"])
        n = _log(rng, 3_000, 60_000 if flow == "auto" else 20_000)
        return dict(kind=kind, flow=flow, nodes=n, edges=n * rng.randint(3, 10),
                    parts=rng.choice([1, 2, 3, 4]) if flow == "auto" else rng.randint(2, 4),
                    din=_log(rng, 30, 300), hidden=rng.choice([32, 64, 100, 128, 256]),
                    classes=_log(rng, 3, 60), layers=rng.randint(2, 3))
    if kind == "loss":
        return dict(kind=kind, rows=_log(rng, 500, 900_000), classes=_log(rng, 2, 50))
    if kind == "infer":
        model = rng.choice(["gcn", "gat"])
        n = _log(rng, 1_000, 40_000)
        return dict(kind=kind, model=model, nodes=n, edges=n * rng.randint(4, 20),
                    din=_log(rng, 30, 500), hidden=rng.randint(4, 32) if model == "gat"
                    else rng.choice([16, 64, 100, 128, 256]),
                    heads=rng.choice([1, 2, 4, 8]) if model == "gat" else 1,
                    classes=_log(rng, 3, 60), layers=rng.randint(2, 3),
                    norm=rng.random() < 0.5)
    rows = _log(rng, 1_000, 90_000)
    case = dict(kind=kind, rows=rows, sources=int(rows * rng.uniform(1.0, 2.2)),
                edges=rows * rng.randint(6, 38), din=_log(rng, 30, 512))
    last = rng.random() < 0.3
    if kind == "gcn":
        case["dout"] = _log(rng, 3, 60) if last else rng.choice([16, 64, 100, 128, 200, 256])
    else:
        case["heads"] = 1 if last else rng.choice([1, 2, 4, 8, 8])
        case["channels"] = (_log(rng, 3, 60) if last else rng.randint(32, 256)
                            if case["heads"] == 1 else rng.randint(4, 256 // case["heads"]))
    case.update(last=last, norm=rng.random() < 0.5, xgrad=rng.random() < 0.8)
    return case


# ------------------------------------------------------------------ the inputs


def _generator(seed, offset=0):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 8 + offset)


def _features(rows, columns, g):
    """N(mean of the column, 1) rows."""
    mean = torch.randn(columns, generator=g, device=DEV) * 0.5
    return torch.randn(rows, columns, generator=g, device=DEV).add_(mean)


def _power_law(n, count, g):
    """`count` ids below n with a power-law frequency, hubs at shuffled places."""
    u = torch.rand(count, generator=g, device=DEV, dtype=torch.float64)
    return torch.randperm(n, generator=g, device=DEV)[(u * u * n).long().clamp_(max=n - 1)]


def _adjacency(rows, sources, edges, seed):
    """CSR of distinct edges and a self loop per row, with symmetric-normalised weights."""
    g = _generator(seed)
    extra = max(edges - rows, 0)
    key = _power_law(rows, extra, g) * sources + _power_law(sources, extra, g)
    loop = torch.arange(rows, device=DEV)
    key = torch.unique(torch.cat([key, loop * sources + loop]))
    row, col = key // sources, key % sources
    out_deg = torch.bincount(row, minlength=rows)
    in_deg = torch.bincount(col, minlength=sources)
    val = (out_deg[row].float() * in_deg[col].float()).rsqrt()
    rowptr = torch.zeros(rows + 1, dtype=torch.int64, device=DEV)
    rowptr[1:] = out_deg.cumsum(0)
    return row, col, val, rowptr


def _weights(case, seed):
    """The model with seeded weights (biases and norms as after some training)."""
    k = case["kind"]
    torch.manual_seed(int(seed))
    if k == "epoch":
        model = GCN(case["din"], case["hidden"], case["classes"], case["layers"], dropout=0.0,
                    norm=True)
    elif k == "infer" and case["model"] == "gcn":
        model = GCN(case["din"], case["hidden"], case["classes"], case["layers"], dropout=0.5,
                    norm=case["norm"])
    elif k == "infer":
        model = GAT(case["din"], case["hidden"], case["classes"], case["layers"],
                    heads=case["heads"], dropout=0.6, norm=case["norm"])
    elif k == "gcn":
        # Two layers, of which one runs: the first, or the last.
        model = (GCN(4, case["din"], case["dout"], 2, dropout=0.0, norm=case["norm"])
                 if case["last"] else
                 GCN(case["din"], case["dout"], 4, 2, dropout=0.0, norm=case["norm"]))
    else:
        model = (GAT(4, case["din"], case["channels"], 2, heads=1, dropout=0.0,
                     norm=case["norm"])
                 if case["last"] else
                 GAT(case["din"], case["channels"], 4, 2, heads=case["heads"], dropout=0.0,
                     norm=case["norm"]))
    with torch.no_grad():
        for name, p in model.named_parameters():
            if p.dim() == 1:
                p.add_(torch.randn(p.shape) * 0.1)
    return model.to(DEV)


def _layer_inputs(case, seed):
    g = _generator(seed, 1)
    x = _features(case["sources"], case["din"], g)
    if case["last"]:
        x = F.relu(x) if case["kind"] == "gcn" else F.elu(x)
    width = case["dout"] if case["kind"] == "gcn" else case["heads"] * case["channels"]
    gy = _features(case["rows"], width, g)
    return x, gy


def _epoch_inputs(case, seed):
    g = _generator(seed)
    n, m = case["nodes"], case["edges"]
    u, v = _power_law(n, m, g), _power_law(n, m, g)
    keep = u != v
    lo, hi = torch.minimum(u, v)[keep], torch.maximum(u, v)[keep]
    key = torch.unique(lo * n + hi)
    a, b = key // n, key % n
    ei = torch.stack([torch.cat([a, b]), torch.cat([b, a])])
    x = _features(n, case["din"], g)
    y = torch.randint(0, case["classes"], (n,), generator=g, device=DEV)
    split = torch.rand(n, generator=g, device=DEV)
    return ei, x, y, split < 0.6, (split >= 0.6) & (split < 0.8), split >= 0.8


def _loss_inputs(case, seed):
    g = _generator(seed)
    rows, classes = case["rows"], case["classes"]
    logits = torch.randn(rows, classes, generator=g, device=DEV) * 2
    y = torch.randint(0, classes, (rows,), generator=g, device=DEV)
    split = torch.rand(rows, generator=g, device=DEV)
    return logits, y, split < 0.6, (split >= 0.6) & (split < 0.8), split >= 0.8


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case}
    if kind == "loss":
        logits, y, train, val, test = _loss_inputs(case, seed)
        state.update(logits=logits.requires_grad_(True), y=y,
                     codes=mask_codes(train, val, test))
        return state
    if kind == "epoch":
        inputs = [t.cpu() for t in _epoch_inputs(case, seed)]
        config = GriNNderConfig(num_parts=case["parts"], device=DEV,
                                project_first=case["flow"],
                                input_residency="resident" if case["flow"] == "auto"
                                else "stream")
        model = _weights(case, seed)
        trainer = Trainer(model, build_partitioned_graph(*inputs, config), config)
        # A learning rate of 0 keeps the weights, so that every pass is the same step; the
        # optimizer's own work is done in full.
        optimizer = torch.optim.Adam(model.parameters(), lr=0.0, weight_decay=5e-4)
        state.update(model=model, trainer=trainer, optimizer=optimizer,
                     criterion=torch.nn.CrossEntropyLoss())
        # The first epoch builds the adjacency plans and uploads what stays resident.
        trainer.train_epoch(optimizer, state["criterion"])
        return state
    model = _weights(case, seed)
    if kind == "infer":
        n = case["nodes"]
        row, col, val, rowptr = _adjacency(n, n, case["edges"], seed)
        adj = Adjacency(rowptr.cpu(), col.cpu(), val.cpu(), (n, n))
        adj.device_plan(DEV)
        x = _features(n, case["din"], _generator(seed, 1))
        state.update(model=model.eval(), adj=adj, x=x)
        return state
    row, col, val, rowptr = _adjacency(case["rows"], case["sources"], case["edges"], seed)
    adj = Adjacency(rowptr.cpu(), col.cpu(), val.cpu(), (case["rows"], case["sources"]))
    adj.device_plan(DEV)
    x, gy = _layer_inputs(case, seed)
    layer = 1 if case["last"] else 0
    params = list(model.convs[layer].parameters())
    if case["norm"] and not case["last"]:
        params += list(model.norms[0].parameters())
    state.update(model=model.train(), adj=adj, x=x.requires_grad_(case["xgrad"]), gy=gy,
                 layer=layer, params=params)
    return state


# -------------------------------------------------------------------- the pass


def run(state):
    kind = state["case"]["kind"]
    if kind == "loss":
        loss, stats = masked_cross_entropy(state["logits"], state["y"], state["codes"])
        (grad,) = torch.autograd.grad(loss, state["logits"])
        return {"loss": loss.detach(), "stats": stats, "grad": grad}
    if kind == "epoch":
        metrics = state["trainer"].train_epoch(state["optimizer"], state["criterion"])
        return {"loss": metrics["loss"], "grads": [p.grad for p in state["model"].parameters()]}
    if kind == "infer":
        model, h = state["model"], state["x"]
        with torch.no_grad():
            for layer in range(model.num_layers):
                h = model.forward_layer(layer, h, state["adj"])
        return h
    x = state["x"]
    y = state["model"].forward_layer(state["layer"], x, state["adj"])
    wanted = state["params"] + ([x] if x.requires_grad else [])
    return {"y": y.detach(), "grads": list(torch.autograd.grad(y, wanted, state["gy"]))}


# ------------------------------------------------------- work, tolerance, exact


def _layer_work(rows, sources, edges, din, width, out, backward, xgrad):
    """Bytes and operations of one layer: the adjacency, the input rows and the output;
    with `backward` also the output's gradient, the weight gradient and the input's."""
    nbytes = 8.0 * edges + 4.0 * (sources * din + rows * out + width * din)
    flops = 2.0 * sources * din * width + 2.0 * edges * width
    if backward:
        nbytes += 4.0 * (rows * out + width * din + (sources * din if xgrad else 0))
        flops += 2.0 * sources * din * width * (2 if xgrad else 1) + 2.0 * edges * width
    return nbytes, flops


def work(case):
    kind = case["kind"]
    if kind == "loss":
        return {"bytes": case["rows"] * (8.0 * case["classes"] + 9),
                "flops": 8.0 * case["rows"] * case["classes"]}
    if kind in ("gcn", "gat"):
        width = case["dout"] if kind == "gcn" else case["heads"] * case["channels"]
        b, f = _layer_work(case["rows"], case["sources"], case["edges"], case["din"], width,
                           width, True, case["xgrad"])
        return {"bytes": b, "flops": f}
    n, L = case["nodes"], case["layers"]
    train = kind == "epoch"
    # An epoch's graph is symmetrised and gets a self loop per node.
    edges = 2 * case["edges"] + n if train else case["edges"]
    heads = case.get("heads", 1)
    dims = [case["din"]] + [case["hidden"] * heads] * (L - 1) + [case["classes"]]
    nbytes = flops = 0.0
    for i in range(L):
        b, f = _layer_work(n, n, edges, dims[i], dims[i + 1], dims[i + 1], train, i > 0)
        nbytes, flops = nbytes + b, flops + f
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Measured against exact(), and stated about four times wider or more.

    Logits, the loss and the output layer's gradients are continuous: 1e-7 to 5e-7 was seen.
    A gradient through a ReLU (or GAT's LeakyReLU) also carries the few elements within
    rounding of the kink, where two correct fp32 results take different sides: up to 3e-5
    was seen at the large cases, and one such element weighs more in a small one.
    """
    if case["kind"] == "loss":
        return {"rel": 5e-7, "differ": 0.0}
    if case["kind"] == "infer" or (case["kind"] == "gcn" and case["last"]):
        return {"rel": 3e-6}
    return {"rel": 5e-4}


def _aggregate64(row, col, weight, x, rows):
    out = torch.zeros((rows, x.size(1)), dtype=torch.float64, device=DEV)
    return out.index_add(0, row, x.index_select(0, col) * weight[:, None])


def _gcn64(conv, row, col, val, x, rows):
    w, b = conv
    z = x @ w.t()
    return _aggregate64(row, col, val, z, rows) + b


def _gat64(conv, row, col, x, rows, heads, concat):
    w, a_s, a_d, b = conv
    hs = x @ w.t()
    channels = hs.size(1) // heads
    outs = []
    for h in range(heads):
        z = hs[:, h * channels:(h + 1) * channels]
        t = F.leaky_relu((z @ a_s[0, h])[col] + (z[:rows] @ a_d[0, h])[row], 0.2)
        top = torch.full((rows,), -float("inf"), dtype=torch.float64, device=DEV)
        top = top.scatter_reduce(0, row, t.detach(), "amax")
        ex = torch.exp(t - top[row])
        den = torch.zeros(rows, dtype=torch.float64, device=DEV).index_add(0, row, ex)
        outs.append(_aggregate64(row, col, ex / (den[row] + 1e-16), z, rows))
    o = torch.cat(outs, 1) if concat else torch.stack(outs).mean(0)
    return o + b


def _params64(model):
    return {k: v.detach().double().requires_grad_(True) for k, v in model.named_parameters()}


def _model_layer64(model, p, layer, x, row, col, val, rows):
    pre = "convs.%d." % layer
    last = layer == model.num_layers - 1
    if isinstance(model, GCN):
        h = _gcn64((p[pre + "lin.weight"], p[pre + "bias"]), row, col, val, x, rows)
    else:
        conv = model.convs[layer]
        h = _gat64((p[pre + "lin.weight"], p[pre + "att_src"], p[pre + "att_dst"],
                    p[pre + "bias"]), row, col, x, rows, conv.heads, conv.concat)
    if last:
        return h
    if model.norms is not None:
        h = F.layer_norm(h, (h.size(1),), p["norms.%d.weight" % layer],
                         p["norms.%d.bias" % layer], model.norms[layer].eps)
    return F.relu(h) if isinstance(model, GCN) else F.elu(h)


def exact(case, seed):
    kind = case["kind"]
    if kind == "loss":
        logits, y, train, val, test = _loss_inputs(case, seed)
        z = logits.double().requires_grad_(True)
        loss = F.cross_entropy(z[train], y[train])
        (grad,) = torch.autograd.grad(loss, z)
        hit = logits.argmax(1) == y
        stats = [train.sum(), (hit & val).sum(), val.sum(), (hit & test).sum(), test.sum()]
        return {"loss": loss.detach(), "stats": torch.stack(stats + [train.sum() * 0]),
                "grad": grad}
    model = _weights(case, seed)
    p = _params64(model)
    if kind == "epoch":
        ei, x, y, train, _, _ = _epoch_inputs(case, seed)
        n = case["nodes"]
        loop = torch.arange(n, device=DEV)
        row, col = torch.cat([ei[0], loop]), torch.cat([ei[1], loop])
        scale = torch.bincount(col, minlength=n).float().pow(-0.5)
        val = (scale[row] * scale[col]).double()
        h = x.double()
        for layer in range(model.num_layers):
            h = _model_layer64(model, p, layer, h, row, col, val, n)
        loss = F.cross_entropy(h[train], y[train])
        names = [k for k, _ in model.named_parameters()]
        grads = torch.autograd.grad(loss, [p[k] for k in names])
        return {"loss": float(loss.detach()), "grads": list(grads)}
    if kind == "infer":
        n = case["nodes"]
        row, col, val, _ = _adjacency(n, n, case["edges"], seed)
        h = _features(n, case["din"], _generator(seed, 1)).double()
        with torch.no_grad():
            for layer in range(model.num_layers):
                h = _model_layer64(model, p, layer, h, row, col, val.double(), n)
        return h
    row, col, val, _ = _adjacency(case["rows"], case["sources"], case["edges"], seed)
    x, gy = _layer_inputs(case, seed)
    x = x.double().requires_grad_(case["xgrad"])
    layer = 1 if case["last"] else 0
    y = _model_layer64(model, p, layer, x, row, col, val.double(), case["rows"])
    names = ["convs.%d.%s" % (layer, k) for k, _ in model.convs[layer].named_parameters()]
    if case["norm"] and not case["last"]:
        names += ["norms.0." + k for k, _ in model.norms[0].named_parameters()]
    wanted = [p[k] for k in names] + ([x] if case["xgrad"] else [])
    return {"y": y.detach(), "grads": list(torch.autograd.grad(y, wanted, gy.double()))}
