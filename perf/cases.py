"""The work that TinyGNN programs have this library do, as measurable cases.

A case names one call (or the short sequence of calls that a program makes
together) and its sizes:

* ``spmm``    -- ``tg.spmm`` / ``tg.spmm_epilogue`` over a kept row plan;
* ``csr``     -- ``tg.edge_list_to_csr`` of an edge list;
* ``norm``    -- ``tg.gcn_norm``;
* ``matmul``  -- ``tg.matmul`` with its fused bias and activation;
* ``sage``    -- ``tg.sage_forward`` over a kept row plan (mean or max);
* ``model``   -- ``Model.forward``: one GCN / SAGE / GAT layer, or a 2-layer
  stack, in both adjacency modes and both precisions;
* ``ingest``  -- CSV texts in device memory to a graph: ``parse_edges``,
  ``parse_features`` and ``edge_list_to_csr``.

Graphs are directed, with power-law out-degrees (exponent 2.1, clipped at
20,000 and at a tenth of the nodes) and uniform destinations, as
``tinygnn_amd.synth`` makes them for the benchmark; everything here is drawn on
the GPU from the seed.
"""
from __future__ import annotations

import math

import torch

import tinygnn_amd as tg

DEV = "cuda"
EPILOGUES = {"none": tg.EPI_NONE, "relu": tg.EPI_RELU, "elu": tg.EPI_ELU}


def listed():
    return [
        # One aggregation of a Cora-size citation graph at the hidden width
        # of its GCN (16): the smallest call, launch bound.
        dict(name="spmm_cora_f16", op="spmm", n=2708, edges=10858, f=16, weighted=True,
             precision="exact", epilogue="none"),
        # The headline benchmark: CSR SpMM of 1M nodes and 50M nonzeros.
        dict(name="spmm_1m_50m_f128", op="spmm", n=1_000_000, edges=50_000_000, f=128,
             weighted=True, precision="exact", epilogue="none"),
        # Building that graph's CSR from its unordered edge list.
        dict(name="csr_1m_50m", op="csr", n=1_000_000, edges=50_000_000, shuffled=True),
        # Normalising a graph with weighted edges, once per graph or per call.
        dict(name="norm_weighted_10m", op="norm", n=200_000, edges=10_000_000, weighted=True),
        # The dense transform of a GCN layer over Cora's bag-of-words features
        # (1,433 -> 16), and of one over a 602-feature social graph.
        dict(name="matmul_cora", op="matmul", m=2708, k=1433, n=16, data="bag", epilogue="none"),
        dict(name="matmul_233k_602_256", op="matmul", m=232_965, k=602, n=256, data="normal",
             epilogue="relu"),
        # A SAGE-Max layer on a 100K-node graph of mean degree 5 (256 -> 128),
        # the size at which the reference's layer timings are published, and a
        # GCN layer of odd widths on a weighted graph of that size, as a model
        # in its default mode: preprocessing on every call.
        dict(name="sage_max_100k", op="sage", n=100_000, edges=500_000, f_in=256, f_out=128,
             agg="max", precision="exact"),
        dict(name="gcn_layer_100k_odd", op="model", arch="gcn", n=100_003, edges=1_500_007,
             f_in=257, hidden=0, heads=1, classes=121, weighted=True, mode="reference",
             precision="fast", data="normal"),
        # One multi-head GAT layer (4 x 64, ELU) on the largest graph.
        dict(name="gat_layer_233k_115m", op="model", arch="gat", n=232_965, edges=114_615_892,
             f_in=602, hidden=0, heads=4, classes=64, weighted=False, mode="cached",
             precision="fast", data="normal"),
        # Whole 2-layer forwards: GAT on a Cora-size graph with a model fresh
        # to its graph's preprocessing on every call, and GCN serving the
        # 232,965-node graph with the preprocessing kept.
        dict(name="gat_cora_forward", op="model", arch="gat", n=2708, edges=10858, f_in=1433,
             hidden=8, heads=8, classes=7, weighted=False, mode="reference", precision="fast",
             data="bag"),
        dict(name="gcn_233k_115m_forward", op="model", arch="gcn", n=232_965,
             edges=114_615_892, f_in=602, hidden=256, heads=1, classes=41, weighted=False,
             mode="cached", precision="fast", data="normal"),
        # Loading a graph from its two CSV texts.
        dict(name="ingest_5m_edges", op="ingest", n=100_000, edges=5_000_000, f=100),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: an operation, and sizes log-uniform over its range."""
    op = rng.choice(["spmm", "spmm", "csr", "norm", "matmul", "matmul", "sage", "model", "model",
                     "model", "ingest"])
    if op == "matmul":
        m, k, n = _log(rng, 500, 500_000), _log(rng, 8, 1500), _log(rng, 2, 600)
        while m * k * n > 3.5e10 or m * max(k, n) > 2e8:
            m = max(500, m // 2)
        return dict(op=op, m=m, k=k, n=n, data=rng.choice(["normal", "bag"]),
                    epilogue=rng.choice(["none", "relu", "elu"]))
    n = _log(rng, 1000, 1_000_000)
    edges = min(int(n * math.exp(rng.uniform(math.log(2), math.log(300)))), 30_000_000)
    if op == "spmm":
        return dict(op=op, n=n, edges=edges, f=_log(rng, 3, 512 if n < 400_000 else 128),
                    weighted=rng.random() < 0.6, precision=rng.choice(["exact", "fast"]),
                    epilogue=rng.choice(["none", "none", "relu"]))
    if op == "csr":
        return dict(op=op, n=n, edges=edges, shuffled=rng.random() < 0.7)
    if op == "norm":
        return dict(op=op, n=n, edges=edges, weighted=rng.random() < 0.5)
    if op == "ingest":
        n = min(n, 200_000)
        return dict(op=op, n=n, edges=min(edges, 5_000_000), f=_log(rng, 3, 100))
    n = min(n, 250_000)
    f_in = _log(rng, 16, 700)
    if op == "sage":
        edges = min(edges, 5_000_000)
        return dict(op=op, n=n, edges=edges, f_in=f_in, f_out=_log(rng, 5, 256),
                    agg=rng.choice(["mean", "max"]), precision=rng.choice(["exact", "fast"]))
    arch = rng.choice(["gcn", "sage", "gat"])
    heads = rng.choice([1, 2, 4, 8]) if arch == "gat" else 1
    stack = rng.random() < 0.5
    precision = rng.choice(["fast", "fast", "fast", "exact"])
    case = dict(op="model", arch=arch, n=n,
                edges=min(edges, 20_000_000 if precision == "fast" else 3_000_000),
                f_in=f_in, hidden=max(4, _log(rng, 8, 256) // heads) if stack else 0,
                heads=heads, classes=_log(rng, 3, 64), weighted=rng.random() < 0.3,
                mode=rng.choice(["reference", "cached"]), precision=precision,
                data=rng.choice(["normal", "bag"]))
    if arch == "gat":
        case["concat"] = rng.random() < 0.7
    return case


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _degrees(n, edges, g):
    """Power-law out-degrees that sum to about ``edges``."""
    dmax = min(20_000, max(n // 10, 4 * edges // n))
    u = torch.rand(n, generator=g, device=DEV, dtype=torch.float64)
    tail = (1.0 - u).pow(-1.0 / 1.1)
    lo, hi = 0.0, float(dmax)
    for _ in range(40):
        mid = 0.5 * (lo + hi)
        if float((tail * mid).clamp(1, dmax).floor().sum()) < edges:
            lo = mid
        else:
            hi = mid
    return (tail * hi).clamp(1, dmax).floor().to(torch.int64)


def _edges(n, edges, g, shuffled=True):
    """``edges`` directed edges without self-loops, sources of power-law
    out-degree, in random order (or by source)."""
    src = torch.repeat_interleave(torch.arange(n, dtype=torch.int32, device=DEV),
                                  _degrees(n, edges, g))
    if src.numel() < edges:
        more = torch.randint(0, n, (edges - src.numel(),), generator=g, device=DEV,
                             dtype=torch.int32)
        src = torch.cat([src, more])
    src = src[torch.randperm(src.numel(), generator=g, device=DEV)[:edges]]
    if not shuffled:
        src = src.sort().values
    dst = torch.randint(0, n - 1, (edges,), generator=g, device=DEV, dtype=torch.int32)
    dst += (dst >= src).to(torch.int32)
    return src.contiguous(), dst


def _csr(src, dst, n):
    """(row_ptr, col_ind) int32 of an edge list: rows = sources, each row's
    destinations ascending."""
    key = (src.to(torch.int64) * n + dst).sort().values
    row_ptr = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    row_ptr[1:] = torch.bincount(src, minlength=n).cumsum(0)
    return row_ptr.to(torch.int32), (key % n).to(torch.int32)


def _graph(case, g):
    n, edges = case["n"], case["edges"]
    row_ptr, col_ind = _csr(*_edges(n, edges, g), n)
    if case.get("weighted"):
        val = torch.rand(edges, generator=g, device=DEV) + 0.1
    else:
        val = torch.ones(edges, device=DEV)
    return tg.DeviceCSR(n, n, row_ptr, col_ind, val)


def _features(rows, cols, data, g):
    """Standard-normal features, or a row-normalised bag of words."""
    if data == "normal":
        return torch.randn(rows, cols, generator=g, device=DEV)
    x = (torch.rand(rows, cols, generator=g, device=DEV) < max(0.013, 2.0 / cols)).float()
    return x / x.sum(dim=1, keepdim=True).clamp(min=1.0)


def _glorot(f_in, f_out, g, shape=None):
    a = math.sqrt(6.0 / (f_in + f_out))
    return (torch.rand(shape or (f_in, f_out), generator=g, device=DEV) * 2 - 1) * a


def _spec(case):
    """The model's layers: ``hidden`` 0 is one layer of ``classes`` outputs
    (per head), else a 2-layer stack with the hidden activation between."""
    arch, f_in, hid, heads, out = (case[k] for k in ("arch", "f_in", "hidden", "heads",
                                                     "classes"))
    if arch == "gat":
        first = dict(type="gat", out=hid or out, heads=heads, concat=case.get("concat", True),
                     slope=0.2, act=0, post=2)
        second = dict(type="gat", out=out, heads=1, concat=True, slope=0.2, act=0, post=0)
    else:
        first = dict(type=arch, out=hid or out, act=1, post=0)
        second = dict(type=arch, out=out, act=0, post=0)
    first["in"], second["in"] = f_in, hid * (heads if first.get("concat", True) else 1)
    return [first, second] if hid else [first]


def _model_weights(spec, g):
    w = {}
    for i, l in enumerate(spec):
        f_in, f_out = l["in"], l["out"]
        if l["type"] == "gcn":
            w[f"layer{i}.weight"] = _glorot(f_in, f_out, g)
        elif l["type"] == "sage":
            w[f"layer{i}.weight_neigh"] = _glorot(f_in, f_out, g)
            w[f"layer{i}.weight_self"] = _glorot(f_in, f_out, g)
        else:
            for h in range(l["heads"]):
                p = f"layer{i}.head{h}"
                w[p + ".weight"] = _glorot(f_in, f_out, g)
                w[p + ".attn_left"] = _glorot(f_out, 1, g, (1, f_out))
                w[p + ".attn_right"] = _glorot(f_out, 1, g, (1, f_out))
                w[p + ".bias"] = 0.1 * torch.randn(1, f_out, generator=g, device=DEV)
        if l["type"] != "gat":
            w[f"layer{i}.bias"] = 0.1 * torch.randn(1, f_out, generator=g, device=DEV)
    return w


def _texts(case, g):
    """Edge and feature CSV texts as device bytes, and the numbers in them:
    ids without padding, features '-d.dddddd' with rows in random order."""
    n, e, f = case["n"], case["edges"], case["f"]

    def digits(v, width, pad):
        p = torch.tensor([10 ** (width - 1 - i) for i in range(width)], device=DEV)
        d = (v.unsqueeze(-1) // p % 10 + 48).to(torch.uint8)
        if not pad:  # leading zeros become 0 bytes, dropped below
            d[(v.unsqueeze(-1) < p) & (p > 1)] = 0
        return d

    src, dst = _edges(n, e, g)
    w = len(str(n - 1))
    parts = []
    for lo in range(0, e, 4_000_000):
        s, d = src[lo:lo + 4_000_000].long(), dst[lo:lo + 4_000_000].long()
        comma = torch.full((s.numel(), 1), 44, dtype=torch.uint8, device=DEV)
        line = torch.cat([digits(s, w, False), comma, digits(d, w, False), comma - 34], 1)
        parts.append(line[line != 0])
    head = torch.tensor(list(b"src,dst\n"), dtype=torch.uint8, device=DEV)
    edges_text = torch.cat([head] + parts)

    k = torch.randint(-9_999_999, 10_000_000, (n, f), generator=g, device=DEV)
    ids = torch.randperm(n, generator=g, device=DEV)
    a = k[ids].abs()
    field = torch.empty((n, f, 10), dtype=torch.uint8, device=DEV)
    field[..., 0] = 44
    field[..., 1] = torch.where(k[ids] < 0, 45, 0)
    field[..., 2] = (a // 1_000_000 + 48).to(torch.uint8)
    field[..., 3] = 46
    field[..., 4:] = digits(a % 1_000_000, 6, True)
    line = torch.cat([digits(ids, w, False), field.reshape(n, f * 10),
                      torch.full((n, 1), 10, dtype=torch.uint8, device=DEV)], 1)
    names = "node_id," + ",".join(f"f{j}" for j in range(f)) + "\n"
    head = torch.tensor(list(names.encode()), dtype=torch.uint8, device=DEV)
    return edges_text, torch.cat([head, line[line != 0]]), src, dst, k


def _inputs(case, seed):
    """The case's inputs as a dict, from the seed alone."""
    g, op = _gen(seed), case["op"]
    if op == "matmul":
        return dict(a=_features(case["m"], case["k"], case["data"], g),
                    b=_glorot(case["k"], case["n"], g),
                    bias=(None if case["epilogue"] == "none" else
                          0.1 * torch.randn(1, case["n"], generator=g, device=DEV)))
    if op == "csr":
        return dict(zip(("src", "dst"), _edges(case["n"], case["edges"], g, case["shuffled"])))
    if op == "ingest":
        return dict(zip(("edges", "features", "src", "dst", "k"), _texts(case, g)))
    s = dict(adj=_graph(case, g))
    if op == "spmm":
        s["b"] = torch.randn(case["n"], case["f"], generator=g, device=DEV)
        if case["epilogue"] != "none":
            s["bias"] = 0.1 * torch.randn(1, case["f"], generator=g, device=DEV)
    elif op == "sage":
        s["x"] = torch.randn(case["n"], case["f_in"], generator=g, device=DEV)
        s["w_neigh"] = _glorot(case["f_in"], case["f_out"], g)
        s["w_self"] = _glorot(case["f_in"], case["f_out"], g)
        s["bias"] = 0.1 * torch.randn(1, case["f_out"], generator=g, device=DEV)
    elif op == "model":
        s["x"] = _features(case["n"], case["f_in"], case["data"], g)
        s["weights"] = _model_weights(_spec(case), g)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    op = case["op"]
    if op in ("spmm", "sage"):
        adj = s["adj"]
        s["plan"] = tg.SpmmPlan(adj.row_ptr, adj.n_rows, adj.nnz,
                                case["f"] if op == "spmm" else max(case["f_in"], case["f_out"]),
                                precision=(tg.PRECISION_EXACT if case["precision"] == "exact"
                                           else tg.PRECISION_FAST))
    elif op == "model":
        m = tg.Model.from_spec(_spec(case), {k: v.cpu().numpy()
                                             for k, v in s.pop("weights").items()})
        if case["precision"] == "exact":
            m.set_precision(tg.PRECISION_EXACT)
        s["model"] = m
    elif op == "ingest":
        s = {k: s[k] for k in ("case", "edges", "features")}
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(state):
    case = state["case"]
    op = case["op"]
    if op == "spmm":
        if "bias" in state:
            return tg.spmm_epilogue(state["adj"], state["b"], state["plan"], state["bias"],
                                    EPILOGUES[case["epilogue"]])
        return tg.spmm(state["adj"], state["b"], state["plan"])
    if op == "csr":
        a = tg.edge_list_to_csr(state["src"], state["dst"], case["n"])
        return a.row_ptr, a.col_ind, a.val
    if op == "norm":
        a, deg, dis = tg.gcn_norm(state["adj"], with_degrees=True)
        return a.row_ptr, a.col_ind, a.val, deg, dis
    if op == "matmul":
        return tg.matmul(state["a"], state["b"], state["bias"], EPILOGUES[case["epilogue"]])
    if op == "sage":
        return tg.sage_forward(state["plan"], state["adj"], state["x"], state["w_neigh"],
                               state["w_self"], state["bias"],
                               agg=tg.AGG_MAX if case["agg"] == "max" else tg.AGG_MEAN)
    if op == "model":
        return state["model"].forward(state["adj"], state["x"],
                                      tg.FORWARD_CACHED if case["mode"] == "cached"
                                      else tg.FORWARD_REFERENCE)
    te = tg.CsvText.from_device(state["edges"])
    src, dst, _ = te.parse_edges()
    te.close()
    tf = tg.CsvText.from_device(state["features"])
    x = tf.parse_features(case["n"])
    tf.close()
    a = tg.edge_list_to_csr(src, dst, case["n"])
    return a.row_ptr, a.col_ind, a.val, x


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    op = case["op"]
    if op == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        return dict(bytes=4.0 * (m * k + k * n + m * n), flops=2.0 * m * k * n)
    n, e = case["n"], case["edges"]
    csr = 4.0 * (n + 1) + 8.0 * e
    if op == "spmm":
        return dict(bytes=csr + 8.0 * n * case["f"], flops=2.0 * e * case["f"])
    if op == "csr":
        return dict(bytes=csr + 8.0 * e, flops=0.0)
    if op == "norm":
        return dict(bytes=2 * csr + 16.0 * n, flops=3.0 * e)
    if op == "ingest":
        w = len(str(n - 1))
        text = e * 2.0 * (w + 0.9) + n * (w + 9.5 * case["f"])
        return dict(bytes=text + csr + 4.0 * n * case["f"], flops=0.0)
    if op == "sage":
        fi, fo = case["f_in"], case["f_out"]
        return dict(bytes=csr - 4.0 * e + 4.0 * (n * fi + 2 * fi * fo + n * fo),
                    flops=4.0 * n * fi * fo + 1.0 * e * min(fi, fo))
    spec = _spec(case)
    out = spec[-1]["out"] * (spec[-1].get("heads", 1) if spec[-1].get("concat", True) else 1)
    byts, flops = csr + 4.0 * n * (spec[0]["in"] + out), 0.0
    for l in spec:
        wide = l["out"] * l.get("heads", 1)
        both = 2 if l["type"] == "sage" else 1
        byts += 4.0 * both * l["in"] * wide
        flops += 2.0 * both * n * l["in"] * wide + 2.0 * (e + n) * wide
    return dict(bytes=byts, flops=flops)


def tolerance(case):
    """Whole numbers, and copied or once-rounded values, are exact or within
    an ulp or two; sums are in fp32, with rows of up to 20,000 terms."""
    op = case["op"]
    if op == "csr":
        return "exact"
    if op == "ingest":  # correctly rounded decimals
        return {"rel": 1e-7, "max": 2e-7}
    # measured against 64 bits, times about four: degrees 1.8e-6 / 4.1e-6,
    # products 6.9e-7 / 5.4e-6, SpMM 1.3e-6 / 1.5e-4, layers 7.3e-7 / 1.8e-5
    if op == "norm":
        return {"rel": 7e-6, "max": 2e-5}
    if op == "matmul":
        return {"rel": 3e-6, "max": 2e-5}
    if op == "spmm":
        return {"rel": 5e-6, "max": 6e-4}
    return {"rel": 3e-6, "max": 1e-4}


# ---------------------------------------------------------------------------
# The same results in 64 bits, by torch alone
# ---------------------------------------------------------------------------
def _rows(row_ptr):
    n = row_ptr.numel() - 1
    return torch.repeat_interleave(torch.arange(n, device=DEV), row_ptr.diff().long())


def _row_reduce(row_ptr, how, part, width):
    """Reduces each row's entries ('sum', or 'max'; 0 for an empty row): entry
    rows lo..hi come from part(lo, hi), some 2**27 values at a time."""
    n, nnz = row_ptr.numel() - 1, int(row_ptr[-1])
    cuts = torch.searchsorted(row_ptr, torch.arange(0, nnz, max(1, (1 << 27) // width),
                                                    dtype=row_ptr.dtype, device=DEV))
    cuts = sorted({0, n, *cuts.tolist()})
    ends = row_ptr[torch.tensor(cuts, device=DEV)].tolist()
    out = []
    for r0, r1, lo, hi in zip(cuts, cuts[1:], ends, ends[1:]):
        lengths = row_ptr[r0:r1 + 1].diff().long()
        x = part(lo, hi)
        y = (torch.segment_reduce(x, how, lengths=lengths, axis=0) if hi > lo else
             torch.zeros((r1 - r0,) + tuple(x.shape[1:]), dtype=x.dtype, device=DEV))
        y[lengths == 0] = 0.0
        out.append(y)
    return torch.cat(out)


def _weighted_sum(row_ptr, col_ind, val, b):
    """out[i] = sum over row i of val * b[col], in fp64."""
    def part(lo, hi):
        x = b[col_ind[lo:hi].long()]
        return x if val is None else x.mul_(val[lo:hi, None])
    return _row_reduce(row_ptr, "sum", part, b.shape[1])


def _self_loops(adj):
    """A + I in fp64 for a graph without self-loops: (row_ptr, col, val)."""
    n = adj.n_rows
    eye = torch.arange(n, device=DEV)
    key = torch.cat([_rows(adj.row_ptr) * n + adj.col_ind, eye * n + eye])
    key, at = key.sort(stable=True)
    val = torch.cat([adj.val.double(), torch.ones(n, dtype=torch.float64, device=DEV)])[at]
    return adj.row_ptr + torch.arange(n + 1, device=DEV, dtype=torch.int32), \
        (key % n).to(torch.int32), val


def _norm(adj):
    rp, ci, v = _self_loops(adj)
    rows = _rows(rp)
    deg = _row_reduce(rp, "sum", lambda lo, hi: v[lo:hi], 1)
    dis = deg.rsqrt()
    return rp, ci, v * dis[rows] * dis[ci.long()], deg, dis


def _act(x, act, post):
    x = x.relu() if act == 1 else x
    return x.relu() if post == 1 else torch.nn.functional.elu(x) if post == 2 else x


def _sage64(adj, x, wn, ws, bias, agg, act):
    deg = adj.row_ptr.diff().clamp(min=1).double()[:, None]
    if agg == "max":
        t = _row_reduce(adj.row_ptr, "max", lambda lo, hi: x[adj.col_ind[lo:hi].long()],
                        x.shape[1]) @ wn
    elif wn.shape[1] < x.shape[1]:
        t = _weighted_sum(adj.row_ptr, adj.col_ind, None, x @ wn) / deg
    else:
        t = (_weighted_sum(adj.row_ptr, adj.col_ind, None, x) / deg) @ wn
    return _act(t + x @ ws + bias, act, 0)


def _gat64(rp, ci, x, w, al, ar, bias, slope, act):
    wh = x @ w
    rows, cols = _rows(rp), ci.long()
    e = (wh @ al.t()).squeeze(1)[rows] + (wh @ ar.t()).squeeze(1)[cols]
    e = torch.where(e >= 0, e, slope * e)
    e = (e - _row_reduce(rp, "max", lambda lo, hi: e[lo:hi], 1)[rows]).exp_()
    total = _row_reduce(rp, "sum", lambda lo, hi: e[lo:hi], 1)
    return _act(_weighted_sum(rp, ci, e / total[rows], wh) + bias, act, 0)


def exact(case, seed):
    s, op = _inputs(case, seed), case["op"]
    if op == "matmul":
        y = s["a"].double() @ s["b"].double()
        if s["bias"] is not None:
            y = y + s["bias"].double()
        return _act(y, *{"none": (0, 0), "relu": (1, 0), "elu": (0, 2)}[case["epilogue"]])
    if op in ("csr", "ingest"):
        rp, ci = _csr(s["src"], s["dst"], case["n"])
        out = (rp, ci, torch.ones(case["edges"], dtype=torch.float64, device=DEV))
        return out if op == "csr" else out + (s["k"].double() / 1e6,)
    adj = s["adj"]
    if op == "norm":
        return _norm(adj)
    if op == "spmm":
        y = _weighted_sum(adj.row_ptr, adj.col_ind, adj.val.double(), s["b"].double())
        if "bias" in s:
            y = y + s["bias"].double()
        return _act(y, int(case["epilogue"] == "relu"), 0)
    if op == "sage":
        return _sage64(adj, s["x"].double(), s["w_neigh"].double(), s["w_self"].double(),
                       s["bias"].double(), case["agg"], 1)
    x = s["x"].double()
    w = {k: v.double() for k, v in s["weights"].items()}
    sl = None if case["arch"] == "sage" else _norm(adj) if case["arch"] == "gcn" \
        else _self_loops(adj)
    for i, l in enumerate(_spec(case)):
        p = f"layer{i}"
        if l["type"] == "gcn":
            x = _weighted_sum(*sl[:3], x @ w[p + ".weight"]) + w[p + ".bias"]
            x = _act(x, l["act"], l["post"])
        elif l["type"] == "sage":
            x = _sage64(adj, x, w[p + ".weight_neigh"], w[p + ".weight_self"], w[p + ".bias"],
                        "mean", l["act"])
        else:
            y = [_gat64(sl[0], sl[1], x, *(w[f"{p}.head{h}.{k}"] for k in
                                           ("weight", "attn_left", "attn_right", "bias")),
                        l["slope"], l["act"]) for h in range(l["heads"])]
            x = _act(torch.cat(y, 1) if l["concat"] else torch.stack(y).mean(0), 0, l["post"])
    return x
