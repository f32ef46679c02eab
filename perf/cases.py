"""Performance cases: the work that a program using this package has it do.

Every case goes through the public entry points (BCSRGraph, core.spmm_tc,
BCSRGraphConv, GCN_BCSR, NeighborSampler, BCSRSampler) on seeded synthetic
graphs of the sizes the benchmark and the tests use:

  spmm      products A X (and A^T G) of a graph that is multiplied again and
            again (full-graph training and inference): `prepare` has made the
            graph's first two products, after which it holds its schedule and
            tile copies, as it does from a training program's second step on
  conv      one graph convolution, forward and backward
  gcn       a full-graph training step up to the gradients
  block     a mini-batch step: sampling, feature gather, forward, backward
  neighbor  the mini-batch producer alone: sampling, transposes, gather
  topk      the window top-K sampler's batch
  build     COO edges -> BCSR graph -> its transpose

Graphs are symmetric with symmetric GCN weights, so A^T = A in the 64-bit
results that `exact` gives.
"""
from __future__ import annotations

import math
import types

import torch
import torch.nn.functional as F

from graph_rws_amd import synth
from graph_rws_amd.core import spmm_tc
from graph_rws_amd.core.ops import gather_rows
from graph_rws_amd.data import BCSRGraph, aligned_rows
from graph_rws_amd.helper.engine import loss_and_metrics_rows
from graph_rws_amd.layers import BCSRGraphConv
from graph_rws_amd.models import GCN_BCSR
from graph_rws_amd.sampler import BCSRSampler, NeighborSampler

DEV = "cuda"
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
# loss scale of a GradScaler at its start: f16 gradients of a mean over
# 10^5 rows would be subnormal without it
SCALE = 65536.0


def listed():
    return [
        # the smallest product: a 2,708-node graph's hidden layer on the
        # default f32 values and 16x8 tiles; launch and host time count
        dict(name="spmm_tiny_f32", kind="spmm", family="powerlaw", n=2708, edges=10556, gamma=2.5, width=16,
             dtype="f32", tc=8, backward=False),
        # a citation-sized power-law graph, hidden width 128, forward and
        # backward product
        dict(name="spmm_mid_bf16", kind="spmm", family="powerlaw", n=169343, edges=2160657, gamma=2.1, width=128,
             dtype="bf16", tc=16, backward=True),
        # a ragged width on the drop-in call (spmm_tc) with the default
        # dtype and tile shape
        dict(name="spmm_mid_f32_tc8", kind="spmm", family="powerlaw", n=169343, edges=2160657, gamma=2.1, width=99,
             dtype="f32", tc=8, backward=False),
        # the benchmark's headline product: a community graph of 114.6M
        # non-zeros, 608 f16 feature columns
        dict(name="spmm_community_f16", kind="spmm", family="community", n=232965, edges=114367035, communities=50,
             width=608, dtype="f16", tc=16, backward=False),
        # a co-purchase-sized power-law graph (2.4M nodes, 123.7M
        # non-zeros), its 112 padded feature columns
        dict(name="spmm_large_bf16", kind="spmm", family="powerlaw", n=2449029, edges=121250971, gamma=2.0,
             width=112, dtype="bf16", tc=16, backward=False),
        # one convolution in the default precision, forward and backward
        # with the input's gradient (a hidden layer)
        dict(name="conv_f32", kind="conv", family="powerlaw", n=169343, edges=2160657, gamma=2.1, width=128, out=256,
             dtype="f32", tc=16),
        # the smallest training step: 1433 -> 16 -> 7, f32
        dict(name="gcn_tiny_f32", kind="gcn", family="powerlaw", n=2708, edges=10556, gamma=2.5, width=1433,
             hidden=16, classes=7, layers=2, dtype="f32", tc=16),
        # a full-graph training step on the community graph under f16
        # autocast: 608 -> 256 -> 256 -> 41
        dict(name="gcn_community_f16", kind="gcn", family="community", n=232965, edges=114367035, communities=50,
             width=608, hidden=256, classes=41, layers=3, dtype="f16", tc=16),
        # the mini-batch producer: 1,024 seeds, fanouts 15/10/5, blocks with
        # the transposes training needs, input features gathered
        dict(name="neighbor_1024", kind="neighbor", n=11100000, edges=160000000, batch=1024, fanouts="15,10,5",
             width=128, dtype="f16", tc=16),
        # a whole mini-batch step over such a batch
        dict(name="block_1024", kind="block", n=11100000, edges=160000000, batch=1024, fanouts="15,10,5",
             width=128, hidden=256, classes=172, dtype="f16", tc=16),
        # the window top-K sampler's batch on the citation-sized graph
        dict(name="topk_1024", kind="topk", family="powerlaw", n=169343, edges=2160657, gamma=2.1, batch=1024,
             fanouts="15,10,5", dtype="f32", tc=8),
        # graph preparation for training: unordered COO edges to BCSR and
        # the transpose of the backward pass
        dict(name="build_community_f16", kind="build", family="community", n=232965, edges=114367035,
             communities=50, dtype="f16", tc=16),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_graph(rng, most_edges):
    if rng.random() < 0.4:
        n = _log(rng, 5000, 232965)
        deg = min(_log(rng, 40, 490), n // 20, most_edges // n)
        return dict(family="community", n=n, edges=n * max(2, deg), communities=rng.randint(4, 50))
    n = _log(rng, 2708, 2449029)
    deg = min(_log(rng, 4, 50), most_edges // n)
    return dict(family="powerlaw", n=n, edges=n * max(2, deg), gamma=round(rng.uniform(2.0, 2.5), 2))


def draw(rng):
    kind = rng.choice(["spmm", "spmm", "spmm", "conv", "conv", "gcn", "neighbor", "block", "topk", "build"])
    dtype = rng.choice(["f32", "f16", "bf16"])
    tc = rng.choice([8, 16])
    if kind in ("neighbor", "block"):
        n = _log(rng, 100000, 11100000)
        hops = rng.randint(2, 3)
        c = dict(kind=kind, n=n, edges=n * rng.randint(4, 14), batch=_log(rng, 64, 1024),
                 fanouts=",".join(str(rng.randint(3, 15)) for _ in range(hops)), width=rng.choice([64, 100, 128]),
                 dtype=rng.choice(["f16", "bf16"]), tc=16)
        if kind == "block":
            c.update(hidden=rng.choice([64, 128, 256]), classes=rng.randint(7, 172))
        return c
    if kind == "topk":
        n = _log(rng, 2708, 169343)
        return dict(kind=kind, family="powerlaw", n=n, edges=n * rng.randint(4, 12), gamma=round(rng.uniform(2.1, 2.5), 2),
                    batch=min(n // 4, _log(rng, 64, 1024)), fanouts=",".join(str(rng.randint(3, 20)) for _ in range(3)),
                    dtype=dtype, tc=tc)
    if kind == "build":
        return dict(kind=kind, dtype=dtype, tc=tc, **_draw_graph(rng, 60000000))
    if kind == "gcn":
        return dict(kind=kind, width=_log(rng, 32, 608), hidden=rng.choice([16, 64, 128, 256]),
                    classes=rng.randint(7, 47), layers=rng.randint(2, 3), dtype=dtype, tc=tc,
                    **_draw_graph(rng, 30000000))
    if kind == "conv":
        return dict(kind=kind, width=_log(rng, 16, 300), out=_log(rng, 7, 256), dtype=dtype, tc=tc,
                    **_draw_graph(rng, 60000000))
    return dict(kind=kind, width=_log(rng, 7, 608), dtype=dtype, tc=tc, backward=rng.random() < 0.5,
                **_draw_graph(rng, 60000000))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _fanouts(case):
    return [int(f) for f in case["fanouts"].split(",")]


def _csr(case, seed):
    if case["family"] == "community":
        return synth.sbm(case["n"], case["communities"], 0.8, case["edges"], seed=seed, device=DEV)
    cap = 17000.0 if case["n"] > 1000000 else None
    return synth.chung_lu(case["n"], case["edges"], case["gamma"], seed=seed, max_degree=cap, device=DEV)


def _graph(case, g):
    return BCSRGraph.from_csr(g.row_ptr, g.col_idx, g.values, case["n"], case["n"], tile_cols=case["tc"],
                              device=torch.device(DEV), values_dtype=DTYPES[case["dtype"]])


def _normal(seed, *shape):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    return torch.randn(*shape, generator=gen, device=DEV)


def _relabel(case, g, seed):
    """Rows, columns and values of g with its nodes renamed by a permutation
    drawn from the seed that keeps each 16-row window together and inside
    its stretch of the id range (its community): other edges, with the same
    number of distinct columns in every window, so that a build's outputs
    have the same sizes for every seed."""
    n = case["n"]
    W = n // 16  # whole windows; a last partial one keeps its place
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    w = torch.arange(W, device=DEV)
    part = w * case.get("communities", 1) // max(1, W)
    order = torch.argsort(part + torch.rand(W, generator=gen, device=DEV, dtype=torch.float64))
    inside = torch.rand(W, 16, generator=gen, device=DEV).argsort(1)
    name = torch.arange(n, device=DEV)
    name[:16 * W] = (order[:, None] * 16 + inside).view(-1)
    rows = torch.repeat_interleave(torch.arange(n, device=DEV), g.row_ptr[1:] - g.row_ptr[:-1])
    return name[rows], name[g.col_idx.long()], g.values


def _features(case, seed):
    return _normal(seed, case["n"], case["width"]).to(DTYPES[case["dtype"]])


def prepare(case, seed):
    dt = DTYPES[case["dtype"]]
    dev = torch.device(DEV)
    kind = case["kind"]
    s = dict(case=case)
    if kind in ("spmm", "conv", "gcn"):
        s["csr"] = g = _csr(case, seed)
        s["graph"] = G = _graph(case, g)
    if kind == "spmm":
        # features are stored with the row pitch the package recommends
        s["x"] = aligned_rows(_features(case, seed + 1))
        if case["backward"]:
            s["g"] = _normal(seed + 2, 16 * G.num_windows, case["width"]).to(dt)
        for _ in range(2):
            run(s)
    elif kind == "conv":
        # parameters and input are f32; f16 and bf16 run under autocast
        torch.manual_seed(seed)
        s["conv"] = BCSRGraphConv(case["width"], case["out"]).to(dev)
        s["x"] = _normal(seed + 1, case["n"], case["width"]).to(dt).requires_grad_(True)
        s["g"] = _normal(seed + 2, case["n"], case["out"]).to(dt)
    elif kind == "gcn":
        torch.manual_seed(seed)
        s["model"] = GCN_BCSR(case["width"], case["hidden"], case["classes"], case["layers"], dropout=0.0,
                              use_checkpoint=False).to(dev).train()
        s["graphs"] = s["model"]._ensure_graph_list(G)
        s["x"] = _features(case, seed + 1)
        gen = torch.Generator(device=DEV)
        gen.manual_seed(seed + 2)
        s["labels"] = torch.randint(0, case["classes"], (case["n"],), generator=gen, device=DEV)
        s["idx"] = (torch.rand(case["n"], generator=gen, device=DEV) < 0.66).nonzero().view(-1)
        s["targets"] = s["labels"][s["idx"]]
    elif kind in ("neighbor", "block"):
        # the producer's outputs have the sizes of what it drew: `neighbor`
        # keeps one draw for every seed (its features vary), `block` draws
        # from the seed
        own = seed if kind == "block" else case["n"]
        s["csr"] = synth.powerlaw_csr(case["n"], case["edges"], seed=own, device=DEV)
        s["x"] = _normal(seed + 1, case["n"], case["width"]).to(dt)
        s["seeds"] = torch.sort(synth.distinct_seeds(case["n"], case["batch"], seed=own + 2, device=DEV)).values
        s["sampler"] = NeighborSampler(_fanouts(case), seed=own, tile_cols=case["tc"], values_dtype=dt)
        if kind == "block":
            torch.manual_seed(seed)
            s["model"] = GCN_BCSR(case["width"], case["hidden"], case["classes"], len(_fanouts(case)), dropout=0.0,
                                  use_checkpoint=False).to(dev).train()
            gen = torch.Generator(device=DEV)
            gen.manual_seed(seed + 3)
            s["targets"] = torch.randint(0, case["classes"], (case["batch"],), generator=gen, device=DEV)
    elif kind == "topk":
        # the sampler ranks columns by |value|: signs drawn from the seed
        # give other values and the same selection, so outputs of one size
        g = _csr(case, case["n"])
        sign = torch.sign(_normal(seed, g.nnz))
        s["csr"] = g = synth.CSRGraph(g.num_nodes, g.row_ptr, g.col_idx, g.values * torch.where(sign == 0, 1, sign))
        s["graph"] = _graph(case, g)
        s["seeds"] = synth.distinct_seeds(case["n"], case["batch"], seed=case["n"] + 1, device=DEV)
        s["sampler"] = BCSRSampler(_fanouts(case), tile_cols=case["tc"], verbose=False)
    else:
        rows, cols, values = _relabel(case, _csr(case, case["n"]), seed)
        gen = torch.Generator(device=DEV)
        gen.manual_seed(seed + 1)
        perm = torch.randperm(rows.numel(), generator=gen, device=DEV)
        src, dst, val = rows[perm], cols[perm], values[perm]
        # what a graph loader hands over: num_nodes(), edges(), edata, device
        s["loaded"] = types.SimpleNamespace(device=dev, num_nodes=lambda: case["n"], edges=lambda: (src, dst),
                                            edata={"weight": val})
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _autocast(case):
    dt = DTYPES[case["dtype"]]
    return torch.autocast("cuda", dtype=dt if dt != torch.float32 else torch.float16, enabled=dt != torch.float32)


def _scale(case):
    return SCALE if case["dtype"] == "f16" else 1.0


def _blocks(s):
    case = s["case"]
    # the first layer's input needs no gradient; its backward runs A^T only
    # where it does not aggregate first
    layers = len(_fanouts(case))
    blocks = s["sampler"].sample_layers(s["csr"].row_ptr, s["csr"].col_idx, s["seeds"],
                                        transposes=[l > 0 for l in range(layers)])
    return blocks, gather_rows(s["x"], blocks[0].src_nodes)


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "spmm":
        G = s["graph"]
        if case["tc"] == 8 and not case["backward"]:
            return [spmm_tc(G.window_offset, G.original_col_indices, G.values_condensed, s["x"], tile_cols=8)[0]]
        out = [G.spmm(s["x"])]
        if case["backward"]:
            out.append(G.spmm_transpose(s["g"]))
        return out
    if kind == "conv":
        conv = s["conv"]
        with _autocast(case):
            y = conv(s["graph"], s["x"], features_target=s["x"])
        return [y.detach()] + list(torch.autograd.grad(y, [s["x"], conv.weight_neigh, conv.weight_self], s["g"]))
    if kind == "gcn":
        with _autocast(case):
            logits = s["model"](s["graphs"], s["x"])
            loss, _, _ = loss_and_metrics_rows(logits, s["idx"], s["targets"])
        grads = torch.autograd.grad(loss * _scale(case), list(s["model"].parameters()))
        return [logits.detach(), loss.detach()] + list(grads)
    if kind == "neighbor":
        blocks, feats = _blocks(s)
        out = [feats]
        for l, b in enumerate(blocks):
            out += [b.src_nodes, b.window_offset, b.original_col_indices, b.values_condensed]
            if l > 0:
                t = b.transpose()
                out += [t.window_offset, t.original_col_indices, t.values_condensed]
        return out
    if kind == "block":
        blocks, feats = _blocks(s)
        with _autocast(case):
            logits = s["model"](blocks, feats)
            loss, _, _ = loss_and_metrics_rows(logits, None, s["targets"])
        grads = torch.autograd.grad(loss * _scale(case), list(s["model"].parameters()))
        return [logits.detach(), loss.detach()] + list(grads)
    if kind == "topk":
        out = []
        for g in s["sampler"].sample_layers(s["graph"], s["seeds"]):
            out += [g.window_offset, g.original_col_indices, g.values_condensed, g.active_windows, g.active_masks]
        return out
    G = BCSRGraph.from_dgl(s["loaded"], tile_cols=case["tc"], values_dtype=DTYPES[case["dtype"]])
    T = G.transpose()
    return [G.window_offset, G.original_col_indices, G.values_condensed,
            T.window_offset, T.original_col_indices, T.values_condensed]


# ---------------------------------------------------------------------------
# the least work, tolerances and 64-bit results
# ---------------------------------------------------------------------------
def work(case):
    """Bytes: every input once and every output once (a graph as CSR: a
    column index and a value per non-zero); flops: two per product term."""
    kind = case["kind"]
    e = 4 if case["dtype"] == "f32" else 2
    n = case["n"]
    nnz = case["edges"] + n
    graph = nnz * (4 + e) + 8 * n
    if kind == "spmm":
        k = 2 if case["backward"] else 1
        return {"bytes": k * (graph + 2 * n * case["width"] * e), "flops": k * 2 * nnz * case["width"]}
    if kind == "conv":
        i, o = case["width"], case["out"]
        w = min(i, o)
        return {"bytes": 2 * graph + n * e * (2 * i + 2 * o) + 16 * i * o,
                "flops": 2 * 2 * nnz * w + 3 * 2 * 2 * n * i * o}
    if kind == "gcn":
        dims = [case["width"]] + [case["hidden"]] * (case["layers"] - 1) + [case["classes"]]
        flops, act = 0, 0
        for l in range(case["layers"]):
            i, o = dims[l], dims[l + 1]
            flops += 2 * 2 * nnz * min(i, o) + (3 if l else 2) * 2 * 2 * n * i * o
            act += n * e * (i + o) * (2 if l else 1)
        return {"bytes": 2 * graph + act, "flops": flops}
    if kind in ("neighbor", "block"):
        # frontiers grow by the fanout, or by the graph's mean degree where
        # that is smaller; per edge an index and two degrees are read and a
        # column index and a value written
        f, edges, rows = case["batch"], 0, []
        for k in reversed(_fanouts(case)):
            rows.append(f)
            m = int(f * min(k, 0.5 * case["edges"] / n))
            edges += m
            f += m
        rows.append(f)
        b = edges * (4 + 16 + 4 + e) + 24 * sum(rows) + 2 * f * case["width"] * e
        if kind == "neighbor":
            return {"bytes": b, "flops": 0}
        dims = [case["width"]] + [case["hidden"]] * (len(rows) - 2) + [case["classes"]]
        flops = 0
        for l in range(len(rows) - 1):
            flops += 3 * 2 * 2 * rows[len(rows) - 2 - l] * dims[l] * dims[l + 1]
        return {"bytes": b + 3 * rows[-2] * case["hidden"] * e, "flops": flops}
    if kind == "topk":
        # each layer reads its active windows' columns and values and writes
        # the kept ones; a few hops reach every window of such a graph
        W, deg = n // 16 + 1, case["edges"] / n
        ids, b = case["batch"], 0
        for k in reversed(_fanouts(case)):
            a = W * (1 - math.exp(-ids / W))
            slots = 16 * deg
            keep = min(32 * math.ceil(k / 32), slots)
            b += int(a * (slots + keep) * (4 + 16 * e))
            ids = a * keep
        return {"bytes": b, "flops": 0}
    return {"bytes": nnz * (8 + 8 + 4) + 2 * graph, "flops": 0}


def tolerance(case):
    kind, dt = case["kind"], case["dtype"]
    if kind in ("neighbor", "topk", "build"):
        return "exact"
    # about four times the error measured against `exact` (f32 products
    # 4.5e-8, weight gradients over 169,343 rows 4.5e-6; f16 outputs 2.1e-4,
    # bf16 1.7e-3)
    if kind == "spmm":
        # one rounding of f32 sums to the output type
        return {"f32": {"rel": 5e-7, "max": 2e-5}, "f16": {"rel": 1e-3, "max": 2e-2},
                "bf16": {"rel": 7e-3, "max": 6e-2}}[dt]
    if kind == "conv":
        # two or three rounded products in a row
        return {"f32": {"rel": 2e-5, "max": 8e-4}, "f16": {"rel": 2e-3, "max": 8e-2},
                "bf16": {"rel": 1.5e-2, "max": 0.5}}[dt]
    # whole models: a rounding of one layer travels through the others (f16
    # gradients of the first layer are 2.7e-2 off the 64-bit ones)
    return {"f32": {"rel": 5e-5, "max": 5e-3}, "f16": {"rel": 3e-2, "max": 0.9}, "bf16": {"rel": 3e-2, "max": 0.9}}[dt]


class _Symmetric(torch.autograd.Function):
    """A x for a symmetric A in 64 bits (A^T g = A g)."""

    @staticmethod
    def forward(ctx, a, x):
        ctx.a = a
        return _mm(a, x)

    @staticmethod
    def backward(ctx, g):
        return None, _mm(ctx.a, g)


def _mm(a, x):
    out = torch.empty((a.shape[0], x.shape[1]), dtype=torch.float64, device=DEV)
    for c in range(0, x.shape[1], 64):
        out[:, c:c + 64] = torch.sparse.mm(a, x[:, c:c + 64].contiguous())
    return out


def _sparse(case, g):
    vals = g.values.to(DTYPES[case["dtype"]]).double()
    return torch.sparse_csr_tensor(g.row_ptr, g.col_idx.long(), vals, (case["n"], case["n"]),
                                   check_invariants=False)


def _model64(case, params, layers, product, x, rows_of):
    """Logits of the model in 64 bits; params in the model's own order."""
    p = list(params)
    convs, norms = p[:2 * layers], p[2 * layers:]
    h = x
    for l in range(layers):
        wn, ws = convs[2 * l], convs[2 * l + 1]
        t = rows_of(l, h)
        h = product(l, h @ wn) + t @ ws
        if l < layers - 1:
            h = F.layer_norm(F.relu(h), (h.shape[1],), norms[2 * l], norms[2 * l + 1], 1e-5)
    return h


def _block64(b):
    """Edges (rows, columns, values) of a sampled block's tiles."""
    tc = b.tile_cols
    win = torch.repeat_interleave(torch.arange(b.num_windows, device=DEV), b.window_offset[1:] - b.window_offset[:-1])
    v = b.values_condensed.view(-1, 16, tc)
    t, r, c = v.nonzero(as_tuple=True)
    return win[t] * 16 + r, b.original_col_indices.view(-1, tc)[t, c].long(), v[t, r, c].double()


def exact(case, seed):
    kind = case["kind"]
    if kind in ("neighbor", "topk", "build"):
        return None
    s = prepare(case, seed)
    if kind == "spmm":
        a = _sparse(case, s["csr"])
        pad = 16 * s["graph"].num_windows - case["n"]
        out = [F.pad(_mm(a, s["x"].double()), (0, 0, 0, pad))]
        if case["backward"]:
            out.append(_mm(a, s["g"][:case["n"]].double()))
        return out
    if kind == "conv":
        a = _sparse(case, s["csr"])
        x = s["x"].detach().double().requires_grad_(True)
        wn, ws = (w.detach().double().requires_grad_(True) for w in (s["conv"].weight_neigh, s["conv"].weight_self))
        y = _Symmetric.apply(a, x @ wn) + x @ ws
        return [y.detach()] + list(torch.autograd.grad(y, [x, wn, ws], s["g"].double()))
    params = [p.detach().double().requires_grad_(True) for p in s["model"].parameters()]
    if kind == "gcn":
        a = _sparse(case, s["csr"])
        logits = _model64(case, params, case["layers"], lambda l, t: _Symmetric.apply(a, t), s["x"].double(),
                          lambda l, h: h)
        loss = F.cross_entropy(logits[s["idx"]], s["targets"])
    else:
        blocks, feats = _blocks(s)
        edges = [_block64(b) for b in blocks]

        def product(l, t):
            r, c, v = edges[l]
            return torch.zeros(blocks[l].num_rows, t.shape[1], dtype=torch.float64, device=DEV).index_add(
                0, r, t[c] * v[:, None])

        logits = _model64(case, params, len(blocks), product, feats.double(), lambda l, h: h[:blocks[l].num_rows])
        loss = F.cross_entropy(logits, s["targets"])
    grads = torch.autograd.grad(loss * _scale(case), params)
    return [logits.detach(), loss.detach()] + list(grads)
