"""The work that is timed when a change is judged: one entry for each path that
a program reaches through the package's public functions, over its real range.

    listed()             the fixed cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  what a program holds before the call (inputs, plans)
    run(state)           one pass through the public entry points
    work(case)           bytes and operations one pass cannot do without
    exact(case, seed)    the same outputs from plain torch in 64 bits

A case is a dict of plain values; "kind" names the path:

    dist      gt.dist          all pairs of one point set, packed or full
    cross     gt.dist_cross    two point sets
    batched   Batch.run        many uneven point sets in one launch
    pdist     gt.pdist         forward and backward through autograd
    mds       gt.mds_stress    stress and its gradient
    clust     gt.dist + gt.hclust, the two stages of gpuDistClust
    pmcc      gt.pmcc          Pearson, both "use" modes
    kendall   gt.kendall
"""
import math

import numpy as np
import torch

import gputools_amd as gt
from gputools_amd.batched import Batch

METHODS = ("euclidean", "maximum", "manhattan", "canberra", "binary", "minkowski")
# operations per feature and pair: difference, power or magnitude, sum
FLOPS = {"euclidean": 3, "maximum": 2, "manhattan": 2, "canberra": 4, "binary": 2, "minkowski": 3}


def listed():
    return [
        # the reference's small example: one call whose launch and latency count
        {"name": "dist_small", "kind": "dist", "n": 1000, "k": 64, "method": "euclidean",
         "precision": "fp32", "layout": "packed", "data": "uniform"},
        # an ordinary gpuDist call, default method and precision
        {"name": "dist_ordinary", "kind": "dist", "n": 8192, "k": 256, "method": "euclidean",
         "precision": "fp32", "layout": "packed", "data": "normal"},
        # presence/absence tables (0/1 columns), a ragged size
        {"name": "dist_binary", "kind": "dist", "n": 30011, "k": 300, "method": "binary",
         "precision": "fp32", "layout": "packed", "data": "bernoulli"},
        # the headline: the largest size a 32-bit R vector takes, clustered
        # points whose near pairs cancel in the matrix-core form
        {"name": "dist_bf16_mixture", "kind": "dist", "n": 65536, "k": 512, "method": "euclidean",
         "precision": "bf16x3", "layout": "packed", "data": "mixture"},
        # the other split precision at a middle, ragged size
        {"name": "dist_fp16_ragged", "kind": "dist", "n": 9001, "k": 130, "method": "euclidean",
         "precision": "fp16x3", "layout": "packed", "data": "uniform"},
        # many uneven point sets at once
        {"name": "batched_1024", "kind": "batched", "sets": 1024, "method": "euclidean", "tile": 3},
        # a training step through the distances
        {"name": "pdist_backward", "kind": "pdist", "n": 16384, "k": 128, "method": "euclidean",
         "precision": "fp32"},
        # metric MDS to the plane: the usual embedding for a plot
        {"name": "mds_plane", "kind": "mds", "n": 16384, "q": 2},
        # gpuDistClust's two stages on the device
        {"name": "clust_average", "kind": "clust", "n": 8192, "k": 256, "method": "euclidean",
         "clust": "average"},
        # gpuCor(x): every variable against every other, no missing values
        {"name": "pmcc_everything", "kind": "pmcc", "na": 8192, "nb": 0, "dim": 1024,
         "use": "everything", "precision": "bf16x3", "missing": 0.0},
        # gpuCor(x, use = "pairwise.complete.obs") on a table with holes
        {"name": "pmcc_pairwise", "kind": "pmcc", "na": 4001, "nb": 0, "dim": 777,
         "use": "pairwise.complete.obs", "precision": "fp32", "missing": 0.1},
        # gpuCor(x, method = "kendall")
        {"name": "kendall_self", "kind": "kendall", "na": 1024, "nb": 0, "dim": 2048,
         "data": "normal"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("dist", "dist", "dist", "split", "split", "cross", "batched", "pdist",
                       "mds", "clust", "pmcc", "pmcc", "kendall"))
    if kind == "dist":
        method = rng.choice(METHODS)
        k = _log(rng, 2, 2000)
        n = _log(rng, 60, min(30000, int(math.sqrt(6e10 / k))))
        data = {"canberra": "shifted", "binary": "bernoulli"}.get(
            method, rng.choice(("normal", "uniform")))
        return {"kind": "dist", "n": n, "k": k, "method": method, "precision": "fp32",
                "layout": rng.choice(("packed", "packed", "full")), "data": data}
    if kind == "split":
        k = _log(rng, 8, 2000)
        n = _log(rng, 300, min(40000, int(math.sqrt(4e11 / k))))
        return {"kind": "dist", "n": n, "k": k, "method": "euclidean",
                "precision": rng.choice(("bf16x3", "fp16x3")), "layout": "packed",
                "data": rng.choice(("normal", "uniform", "mixture"))}
    if kind == "cross":
        k = _log(rng, 2, 1000)
        return {"kind": "cross", "na": _log(rng, 20, 8000), "nb": _log(rng, 20, 8000), "k": k,
                "method": rng.choice(METHODS)}
    if kind == "batched":
        return {"kind": "batched", "sets": _log(rng, 16, 1024),
                "method": rng.choice(("euclidean", "manhattan", "maximum")),
                "tile": rng.choice((1, 2, 3))}
    if kind == "pdist":
        k = _log(rng, 2, 400)
        n = _log(rng, 100, min(16384, int(math.sqrt(3e10 / k))))
        method = rng.choice(("euclidean", "euclidean", "minkowski"))
        return {"kind": "pdist", "n": n, "k": k, "method": method, "precision": "fp32"}
    if kind == "mds":
        return {"kind": "mds", "n": _log(rng, 200, 16384), "q": rng.choice((2, 2, 3, 5, 16, 32))}
    if kind == "clust":
        return {"kind": "clust", "n": _log(rng, 100, 6000), "k": _log(rng, 4, 300),
                "method": rng.choice(("euclidean", "manhattan", "maximum")),
                "clust": rng.choice(("single", "complete", "average", "ward"))}
    if kind == "pmcc":
        use = rng.choice(("everything", "pairwise.complete.obs"))
        pairwise = use != "everything"
        na = _log(rng, 50, 4500 if pairwise else 8000)
        return {"kind": "pmcc", "na": na, "nb": rng.choice((0, 0, _log(rng, 50, 4000))),
                "dim": _log(rng, 20, 800 if pairwise else 1500), "use": use,
                "precision": "fp32" if pairwise else rng.choice(("bf16x3", "fp16x3", "fp32")),
                "missing": rng.choice((0.02, 0.1, 0.3)) if pairwise else 0.0}
    n = _log(rng, 30, 2048)
    return {"kind": "kendall", "na": _log(rng, 20, 1024), "nb": rng.choice((0, _log(rng, 20, 700))),
            "dim": n, "data": rng.choice(("normal", "ordinal"))}


# ------------------------------- inputs ------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _points(data, n, k, g):
    if data == "uniform":
        return torch.rand((n, k), generator=g, device="cuda")
    if data == "bernoulli":
        return (torch.rand((n, k), generator=g, device="cuda") < 0.1).float()
    x = torch.randn((n, k), generator=g, device="cuda")
    if data == "shifted":      # positive data, as canberra is used on
        return x.abs_().add_(0.1)
    if data == "mixture":      # 64 centres, points 1e-3 around them
        c = torch.randn((64, k), generator=g, device="cuda")
        return x.mul_(1e-3).add_(c[torch.arange(n, device="cuda") % 64])
    if data == "ordinal":      # questionnaire answers: many ties
        return x.mul_(1.5).round_().clamp_(-3, 3)
    return x


def _variables(n, dim, missing, g):
    """Expression-like variables: each has its own level and spread, groups of
    them share a factor, and a share of the samples is missing."""
    factor = torch.randn((24, dim), generator=g, device="cuda")
    x = torch.randn((n, dim), generator=g, device="cuda")
    load = torch.rand((n, 1), generator=g, device="cuda") * 1.5
    x += load * factor[torch.randint(24, (n,), generator=g, device="cuda")]
    x *= 0.2 + torch.rand((n, 1), generator=g, device="cuda")
    x += torch.rand((n, 1), generator=g, device="cuda") * 8
    if missing:
        x[torch.rand((n, dim), generator=g, device="cuda") < missing] = float("nan")
    return x


def _sets(case, seed):
    # sizes and feature counts are the plan of the case, the same for each seed
    rng = np.random.default_rng(case["sets"])
    sizes = np.floor(np.exp(rng.uniform(np.log(32), np.log(2048), case["sets"]))).astype(np.int64)
    dims = rng.choice(np.asarray((16, 32, 64, 128), dtype=np.int64), case["sets"])
    x = torch.randn(int((sizes * dims).sum()), generator=_gen(seed), device="cuda")
    return sizes, dims, x


def _p(case):
    return 3.0 if case["method"] == "minkowski" else 2.0


def _pairs(n):
    return n * (n - 1) // 2


def prepare(case, seed):
    kind, g = case["kind"], _gen(seed)
    s = {"case": case}
    if kind == "dist":
        s["x"] = _points(case["data"], case["n"], case["k"], g)
    elif kind == "cross":
        data = {"canberra": "shifted", "binary": "bernoulli"}.get(case["method"], "normal")
        s["a"] = _points(data, case["na"], case["k"], g)
        s["b"] = _points(data, case["nb"], case["k"], g)
    elif kind == "batched":
        sizes, dims, x = _sets(case, seed)
        s["batch"] = Batch(x=x, sizes=sizes, dims=dims, method=case["method"])
        s["batch"].schedule(case["tile"])
    elif kind == "pdist":
        s["x"] = _points("normal", case["n"], case["k"], g)
        s["g"] = torch.randn(_pairs(case["n"]), generator=g, device="cuda")
    elif kind == "mds":
        # dissimilarities near, not at, the embedding's own distances
        s["y"] = _points("normal", case["n"], case["q"], g)
        s["delta"] = torch.rand(_pairs(case["n"]), generator=g, device="cuda") * (
            2.0 * math.sqrt(2.0 * case["q"]))
    elif kind == "clust":
        s["x"] = _points("normal", case["n"], case["k"], g)
    elif kind == "pmcc":
        s["a"] = _variables(case["na"], case["dim"], case["missing"], g)
        s["b"] = _variables(case["nb"], case["dim"], case["missing"], g) if case["nb"] else None
    else:
        s["a"] = _points(case["data"], case["na"], case["dim"], g)
        s["b"] = _points(case["data"], case["nb"], case["dim"], g) if case["nb"] else None
    return s


# ------------------------------- one pass ----------------------------------

def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "dist":
        return gt.dist(state["x"], c["method"], _p(c), precision=c["precision"],
                       layout=c["layout"])
    if kind == "cross":
        return gt.dist_cross(state["a"], state["b"], c["method"], _p(c))
    if kind == "batched":
        b = state["batch"]
        b.run(c["tile"])
        return b.out[:b.pairs]
    if kind == "pdist":
        x = state["x"].detach().requires_grad_(True)
        d = gt.pdist(x, c["method"], _p(c), precision=c["precision"])
        d.backward(state["g"])
        return d.detach(), x.grad
    if kind == "mds":
        y = state["y"].detach().requires_grad_(True)
        stress = gt.mds_stress(y, state["delta"])
        stress.backward()
        return stress.detach(), y.grad
    if kind == "clust":
        d = gt.dist(state["x"], c["method"], layout="full")
        return gt.hclust(d, c["clust"])
    if kind == "pmcc":
        return gt.pmcc(state["a"], state["b"], use=c["use"], precision=c["precision"])
    return gt.kendall(state["a"], state["b"])


def work(case):
    kind = case["kind"]
    if kind in ("dist", "clust", "pdist"):
        n, k = case["n"], case["k"]
        pairs = _pairs(n)
        dots = case.get("precision", "fp32") != "fp32" or case["method"] == "binary"
        flops = (2 if dots else FLOPS[case["method"]]) * k * pairs
        if kind == "dist":
            cells = pairs if case["layout"] == "packed" else n * n
            return {"bytes": 4 * (n * k + cells), "flops": flops}
        if kind == "pdist":   # forward, and both rows' gradients from each pair
            return {"bytes": 4 * (2 * n * k + 2 * pairs), "flops": flops + 4 * k * pairs}
        # about four operations per live cluster and round
        return {"bytes": 4 * (n * k + 3 * n), "flops": flops + 4 * pairs}
    if kind == "cross":
        na, nb, k = case["na"], case["nb"], case["k"]
        return {"bytes": 4 * ((na + nb) * k + na * nb), "flops": FLOPS[case["method"]] * k * na * nb}
    if kind == "batched":
        rng = np.random.default_rng(case["sets"])
        sizes = np.floor(np.exp(rng.uniform(np.log(32), np.log(2048), case["sets"])))
        dims = rng.choice(np.asarray((16, 32, 64, 128)), case["sets"])
        pairs = sizes * (sizes - 1) / 2
        return {"bytes": float(4 * ((sizes * dims).sum() + pairs.sum())),
                "flops": float(FLOPS[case["method"]] * (pairs * dims).sum())}
    if kind == "mds":
        n, q = case["n"], case["q"]
        return {"bytes": 4 * (_pairs(n) + 2 * n * q), "flops": 6 * q * _pairs(n)}
    na, nb, dim = case["na"], case["nb"], case["dim"]
    cells = na * (nb or na)
    unique = na * nb if nb else na * (na + 1) // 2
    if kind == "pmcc":
        per = 2 if case["use"] == "everything" else 12
        return {"bytes": 4 * (na + nb) * dim + 12 * cells, "flops": per * dim * unique}
    # Kendall: one sign product per sample pair and pair of variables
    return {"bytes": 4 * (na + nb) * dim + 8 * cells, "flops": dim * (dim - 1) * unique}


# ------------------------------- 64 bits -----------------------------------

def _block(a, b, method):
    """Distances of the rows of a to the rows of b (float64)."""
    if method == "euclidean":
        sq = (a * a).sum(1)[:, None] + (b * b).sum(1)[None, :] - 2.0 * (a @ b.T)
        return sq.clamp_(min=0.0).sqrt_()
    if method == "binary":
        x, y = (a != 0).double(), (b != 0).double()
        both = x @ y.T
        either = x.sum(1)[:, None] + y.sum(1)[None, :] - both
        return torch.where(either > 0, (either - both) / either.clamp(min=1.0), torch.zeros_like(both))
    acc = torch.zeros((a.shape[0], b.shape[0]), dtype=torch.float64, device=a.device)
    for f in range(a.shape[1]):
        u, v = a[:, f, None], b[None, :, f]
        d = (u - v).abs_()
        if method == "maximum":
            torch.maximum(acc, d, out=acc)
        elif method == "manhattan":
            acc += d
        elif method == "canberra":    # positive data: no 0/0 term
            acc += d.div_((u + v).abs_())
        else:                         # minkowski, p = 3
            acc += d.pow_(3)
    return acc.pow_(1.0 / 3.0) if method == "minkowski" else acc


def _all_pairs(x, method, layout="packed"):
    n = x.shape[0]
    x = x.double()
    if layout == "packed":
        out = torch.empty(_pairs(n), dtype=torch.float64, device=x.device)
    else:
        out = torch.empty((n, n), dtype=torch.float64, device=x.device)
    cols = torch.arange(n, device=x.device)
    at = 0
    step = max(1, min(n, (1 << 27) // max(n, 1)))
    for j in range(0, n, step):
        rows = cols[j:j + step]
        d = _block(x[j:j + step], x, method)
        if layout == "packed":        # column j of the triangle: rows j + 1 ..
            d = d[cols[None, :] > rows[:, None]]
            out[at:at + d.numel()] = d
            at += d.numel()
        else:
            d[rows - j, rows] = 0.0
            out[j:j + step] = d
    return out


def _unpack(v, n):
    m = torch.zeros((n, n), dtype=torch.float64, device=v.device)
    m[torch.ones((n, n), dtype=torch.bool, device=v.device).triu_(1)] = v.double()
    return m + m.T


def exact(case, seed):
    kind = case["kind"]
    if kind == "clust":    # merges follow the distances' last bits
        return None
    s = prepare(case, seed)
    if kind == "dist":
        return _all_pairs(s["x"], case["method"], case["layout"])
    if kind == "cross":
        return _block(s["b"].double(), s["a"].double(), case["method"])
    if kind == "batched":
        b = s["batch"]
        return torch.cat([_all_pairs(b.set_points(i), case["method"]) for i in range(b.nsets)])
    if kind == "pdist":
        x, n = s["x"].double(), case["n"]
        d = _all_pairs(s["x"], case["method"])
        full = _unpack(d, n)
        w = _unpack(s["g"], n)
        grad = torch.zeros_like(x)
        if case["method"] == "euclidean":
            w /= full.fill_diagonal_(1.0)
            grad = x * w.sum(1, keepdim=True) - w @ x
        else:                         # minkowski, p = 3
            w /= full.fill_diagonal_(1.0).square_()
            for f in range(x.shape[1]):
                diff = x[:, f, None] - x[None, :, f]
                grad[:, f] = (w * diff * diff.abs()).sum(1)
        return d, grad
    if kind == "mds":
        y, n = s["y"].double(), case["n"]
        d = torch.zeros((n, n), dtype=torch.float64, device="cuda")
        for f in range(case["q"]):
            d += (y[:, f, None] - y[None, :, f]).square_()
        d.sqrt_()
        r = d - _unpack(s["delta"], n)
        w = 2.0 * r / d.fill_diagonal_(1.0)
        w.fill_diagonal_(0.0)
        r.fill_diagonal_(0.0)
        return r.square_().sum() / 2.0, y * w.sum(1, keepdim=True) - w @ y
    if kind == "pmcc":
        a = s["a"].double()
        b = a if s["b"] is None else s["b"].double()
        c = a.nanmean(1, keepdim=True)
        ma, mb = (~a.isnan()).double(), (~b.isnan()).double()
        a = (a - c).nan_to_num_(nan=0.0)
        b = (b - b.nanmean(1, keepdim=True)).nan_to_num_(nan=0.0)
        n = ma @ mb.T
        sa, sb = a @ mb.T, ma @ b.T
        r = (a @ b.T - sa * sb / n) / (((a * a) @ mb.T - sa * sa / n) *
                                       (ma @ (b * b).T - sb * sb / n)).sqrt_()
        ts = torch.where(r >= 0.999, torch.full_like(r, 10000.0),
                         r * ((n - 2.0) / (1.0 - r * r).clamp(min=1e-9)).sqrt())
        return n, r, ts
    # Kendall: a sample pair tied in both variables counts as concordant
    a = s["a"]
    b = a if s["b"] is None else s["b"]
    dim, step = case["dim"], 32
    conc = torch.zeros((b.shape[0], a.shape[0]), dtype=torch.float64, device="cuda")
    idx = torch.arange(dim, device="cuda")
    for i in range(0, dim, step):
        later = (idx[None, :] > idx[i:i + step, None]).reshape(-1)
        sides = []
        for v in (a, b):
            sign = (v[:, None, :] - v[:, i:i + step, None]).sign_().reshape(v.shape[0], -1)
            sides.append([((sign == t) & later).double() for t in (1.0, -1.0, 0.0)])
        for u, v in zip(*sides):
            conc += v @ u.T
    total = dim * (dim - 1) / 2.0
    return (2.0 * conc - total) / total
