"""The calls this framework is measured on, from the smallest to the largest.

A case is a dict of plain values; ``op`` names the entry point and the rest its
sizes, types and options:

classify     KNeighborsClassifier.predict_proba on device queries (fit before)
knn          prims.knn_topk, f32 / f64, Euclidean / cosine, d > 16
selfknn      prims.knn_topk of few-column points against themselves
metric_knn   prims.knn_topk, Manhattan / Chebyshev
assign       prims.kmeans_assign, the step of KMeans.predict
fit          prims.kmeans_fit with k-means++ starts
graph        prims.knn_graph, UMAP's operand
radius       prims.radius_neighbors
pairwise     prims.pairwise_distance

Listed sizes are the benchmark's configurations (``mlrs_amd/synthetic.py``,
with the same distributions drawn on the device) or sizes of the same kind
that are not round: row widths that are no multiple of a vector or a tile, row
counts that leave remainders.
"""
import math

import torch

from mlrs_amd import neighbors, prims

_DT = {"f32": torch.float32, "f64": torch.float64}
_SIZE = {"f32": 4, "f64": 8}


def listed():
    return [
        # A service that classifies a few dozen rows per request against a
        # table of 20,000: launches and host work are all there is.
        dict(name="classify_online", op="classify", dtype="f32", n=20_000, q=64, d=30, k=5, classes=10),
        # The small benchmark configuration: one batch of queries against a
        # 10,000-row table of 64 features.
        dict(name="knn_small", op="knn", dtype="f32", metric="euclidean", n=10_000, q=1_000, d=64, k=10,
             data="normal"),
        # A table of 50 columns (rows not 16-byte aligned) searched with a
        # held-out part of it: counts and width all ragged.
        dict(name="knn_ragged", op="knn", dtype="f32", metric="euclidean", n=50_021, q=5_003, d=50, k=15,
             data="mixture"),
        # The headline configuration: a large index, a large batch.
        dict(name="knn_large", op="knn", dtype="f32", metric="euclidean", n=1_000_000, q=10_000, d=128, k=32,
             data="mixture"),
        # Cosine search over embeddings in double precision, NumPy's default type.
        dict(name="knn_cosine_f64", op="knn", dtype="f64", metric="cosine", n=200_000, q=5_000, d=256, k=16,
             data="uniform"),
        # Every point of a point cloud against the cloud, exact copies among
        # them: the shape of core distances.
        dict(name="selfknn_points", op="selfknn", dtype="f32", n=500_000, d=3, k=8),
        # Manhattan search in double precision over a table of mixed features.
        dict(name="knn_manhattan_f64", op="metric_knn", dtype="f64", metric="manhattan", n=60_013, q=2_001, d=40,
             k=10),
        # Assignment of five million points to 1,024 centres.
        dict(name="assign_large", op="assign", dtype="f32", n=5_000_000, c=1_024, d=64),
        # A whole fit at an everyday size: k-means++ starts, ten iterations.
        dict(name="fit_mid", op="fit", dtype="f32", n=150_001, c=50, d=20, iters=10),
        # The neighbour graph that UMAP is given, single-precision rows in and
        # the reference's double-precision distances out.
        dict(name="graph_umap", op="graph", dtype="f32", metric="euclidean", n=60_000, d=50, k=15),
        # Every neighbour within a radius, double precision, about fifty each:
        # the query of density clustering.
        dict(name="radius_f64", op="radius", dtype="f64", metric="euclidean", n=40_009, q=10_001, d=10, near=50),
        # A full distance matrix for a kernel or a linkage.
        dict(name="pairwise_f32", op="pairwise", dtype="f32", metric="euclidean", n=8_209, q=8_009, d=100),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more call of the ranges the listed ones stand for."""
    op = rng.choice(["classify", "knn", "knn", "knn", "selfknn", "metric_knn", "assign", "fit", "graph", "radius",
                     "pairwise"])
    dtype = rng.choice(["f32", "f64"])
    if op == "classify":
        return dict(op=op, dtype=dtype, n=_log(rng, 2_000, 100_000), q=_log(rng, 1, 512), d=_log(rng, 4, 128),
                    k=rng.choice([3, 5, 10, 15, 31]), classes=_log(rng, 2, 50))
    if op == "knn":
        d = _log(rng, 17, 256)
        pairs = (1e10 if dtype == "f32" else 2e9) * 128.0 / max(d, 64) / 2.0
        q = _log(rng, 50, 10_000)
        n = _log(rng, 5_000, max(5_001, min(1_000_000, pairs / q)))
        metric = rng.choice(["euclidean", "euclidean", "cosine"])
        return dict(op=op, dtype=dtype, metric=metric, n=n, q=q, d=d, k=rng.choice([1, 5, 10, 15, 30, 50, 100]),
                    data=rng.choice(["normal", "mixture", "uniform"]))
    if op == "selfknn":
        d = rng.choice([2, 3, 4, 6, 8])
        most = 500_000 * math.sqrt((3.0 if dtype == "f32" else 1.5) / (d + 2.0))
        return dict(op=op, dtype=dtype, n=_log(rng, 5_000, most), d=d, k=rng.choice([2, 5, 8]))
    if op == "metric_knn":
        d = _log(rng, 4, 128)
        q = _log(rng, 50, 3_000)
        n = _log(rng, 3_000, max(3_001, min(200_000, 4e9 / (d * q))))
        return dict(op=op, dtype=dtype, metric=rng.choice(["manhattan", "chebyshev"]), n=n, q=q, d=d,
                    k=rng.choice([1, 5, 10, 30]))
    if op == "assign":
        d = _log(rng, 2, 128)
        c = _log(rng, 2, 1_024)
        most = 3e11 / (max(d, 16) * max(c, 32)) / (1 if dtype == "f32" else 4)
        return dict(op=op, dtype=dtype, n=_log(rng, 5_000, max(5_001, min(2_000_000, most))), c=c, d=d)
    if op == "fit":
        return dict(op=op, dtype=dtype, n=_log(rng, 5_000, 150_000), c=_log(rng, 3, 50), d=_log(rng, 2, 64),
                    iters=10)
    if op == "graph":
        d = _log(rng, 4, 128)
        most = math.sqrt(3.6e9 * 50.0 / max(d, 50))
        return dict(op=op, dtype=dtype, metric=rng.choice(["euclidean", "euclidean", "cosine"]),
                    n=_log(rng, 3_000, most), d=d, k=rng.choice([5, 15, 30]))
    if op == "radius":
        d = _log(rng, 2, 32)
        q = _log(rng, 100, 10_000)
        return dict(op=op, dtype=dtype, metric="euclidean", n=_log(rng, 3_000, min(100_000, 4e9 / (d * q))), q=q, d=d,
                    near=_log(rng, 5, 100))
    d = _log(rng, 4, 200)
    return dict(op=op, dtype=dtype, metric=rng.choice(["euclidean", "cosine", "manhattan"]), n=_log(rng, 300, 6_000),
                q=_log(rng, 300, 6_000), d=d)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, shape, dtype):
    return torch.randn(shape, generator=g, device="cuda", dtype=dtype)


def _uniform(g, shape, dtype):
    return torch.rand(shape, generator=g, device="cuda", dtype=dtype)


def _mixture(g, centres, n):
    """n rows about the centres, unit standard deviation, and their component."""
    comp = torch.randint(0, centres.shape[0], (n,), generator=g, device="cuda")
    return _normal(g, (n, centres.shape[1]), centres.dtype) + centres[comp], comp


def _rows(g, kind, sizes, d, dtype):
    """One matrix per size, all of one distribution."""
    if kind == "mixture":
        centres = _uniform(g, (100, d), dtype) * 20.0 - 10.0
        return [_mixture(g, centres, n)[0] for n in sizes]
    make = _normal if kind == "normal" else _uniform
    return [make(g, (n, d), dtype) for n in sizes]


def _inputs(case, seed):
    """The call's matrices, from the seed alone."""
    g, op, dtype, d = _gen(seed), case["op"], _DT[case["dtype"]], case["d"]
    if op == "classify":
        centres = _normal(g, (case["classes"], d), dtype) / math.sqrt(d)  # classes that overlap
        x, y = _mixture(g, centres, case["n"])
        y[:case["classes"]] = torch.arange(case["classes"], device="cuda")  # every class occurs
        return dict(x=x, y=y, q=_mixture(g, centres, case["q"])[0])
    if op == "knn":
        x, q = _rows(g, case["data"], (case["n"], case["q"]), d, dtype)
        return dict(x=x, q=q)
    if op == "selfknn":
        x = _uniform(g, (case["n"], d), dtype)
        perm = torch.randperm(case["n"], generator=g, device="cuda")
        copies = case["n"] // 20
        x[perm[:copies]] = x[perm[copies:2 * copies]]
        return dict(x=x, q=x)
    if op in ("metric_knn", "pairwise"):
        x, q = _rows(g, "normal", (case["n"], case["q"]), d, dtype)
        return dict(x=x, q=q)
    if op == "assign":
        centres = 5.0 * _normal(g, (case["c"], d), dtype)
        x = _mixture(g, centres, case["n"])[0]
        return dict(x=x, c=centres + 0.1 * _normal(g, (case["c"], d), dtype))
    if op == "fit":
        return dict(x=_mixture(g, 3.0 * _normal(g, (case["c"], d), dtype), case["n"])[0], seed=int(seed) & 0xFFFF)
    if op == "graph":
        return dict(x=_mixture(g, 2.0 * _normal(g, (10, d), dtype), case["n"])[0])
    # radius: compact clusters of `near` points on a grid whose spacing is four
    # radii, what is left over alone on sites of its own; every query lies in a
    # cluster and within the radius of all its points, so the match total does
    # not depend on the seed
    near, groups = case["near"], case["n"] // case["near"]
    alone = case["n"] - groups * near
    side = math.ceil((groups + alone) ** (1.0 / d))
    site = torch.arange(groups + alone, device="cuda")
    sites = torch.stack([(site // side ** j) % side for j in range(d)], 1).to(dtype) * 4.0
    member = torch.cat([site[:groups].repeat_interleave(near), site[groups:]])
    member = member[torch.randperm(case["n"], generator=g, device="cuda")]
    wanted = torch.randint(0, groups, (case["q"],), generator=g, device="cuda")
    x, q = (sites[m] + (_uniform(g, (m.shape[0], d), dtype) - 0.5) / math.sqrt(d) for m in (member, wanted))
    return dict(x=x, q=q, r=1.001)


def prepare(case, seed):
    s = _inputs(case, seed)
    if case["op"] == "classify":
        s["model"] = neighbors.KNeighborsClassifier(n_neighbors=case["k"], weights="distance").fit(s["x"], s["y"])
    s["case"] = case
    return s


# ---------------------------------------------------------------------------
# the calls
# ---------------------------------------------------------------------------
def run(s):
    c = s["case"]
    op = c["op"]
    if op == "classify":
        return s["model"].predict_proba(s["q"])
    if op == "knn" or op == "metric_knn":
        return prims.knn_topk(s["q"], s["x"], c["k"], c["metric"])
    if op == "selfknn":
        return prims.knn_topk(s["q"], s["x"], c["k"])
    if op == "assign":
        return prims.kmeans_assign(s["x"], s["c"])
    if op == "fit":
        return prims.kmeans_fit(s["x"], c["c"], "k-means++", seed=s["seed"], max_iter=c["iters"], tol=0.0)
    if op == "graph":
        return prims.knn_graph(s["x"], c["k"], c["metric"])
    if op == "radius":
        return prims.radius_neighbors(s["q"], s["x"], s["r"], c["metric"])
    return prims.pairwise_distance(s["q"], s["x"], c["metric"], sqrt=True)


def work(case):
    """Each matrix read once and each result written once; two operations per
    feature of a pair (a multiply and an add, or a difference and an add)."""
    op, e, n, d = case["op"], _SIZE[case["dtype"]], case["n"], case["d"]
    if op == "assign":
        c = case["c"]
        return {"bytes": float(e * d * (n + c) + n * (e + 8)), "flops": 2.0 * n * c * d}
    if op == "fit":
        c, it = case["c"], case["iters"]
        return {"bytes": float(e * d * n * (c + 2 * it + 1) + 8 * n), "flops": 2.0 * n * c * d * (it + 2)}
    if op in ("graph", "selfknn"):
        out = case["k"] * (16 if op == "graph" else e + 8)
        return {"bytes": float(n * (e * d + out)), "flops": 2.0 * n * n * d}
    q = case["q"]
    if op == "pairwise":
        out = e * q * n
    elif op == "radius":
        out = q * (8 + case["near"] * (e + 4))
    elif op == "classify":
        out = q * case["classes"] * e
    else:
        out = q * case["k"] * (e + 8)
    return {"bytes": float(e * d * (n + q) + out), "flops": 2.0 * n * q * d}


def tolerance(case):
    """Every result is the reference CPU backend's bit for bit: each value is
    evaluated in the reference's operation order whatever kernel finds the
    pair, ties go to the lower index, and the tests hold each kernel family to
    the same bits.  (Measured: repeated calls, and the kernel families against
    each other, differ nowhere.)"""
    return "exact"


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _blocks(rows, cols):
    step = max(1, int(4e8) // max(1, cols))
    return [(a, min(rows, a + step)) for a in range(0, rows, step)]


def _pair_values(q, x, metric):
    """One block of distances (squared for Euclidean) in double precision."""
    if metric in ("manhattan", "chebyshev"):
        v = torch.zeros((q.shape[0], x.shape[0]), dtype=torch.float64, device="cuda")
        for j in range(q.shape[1]):
            diff = (q[:, j, None] - x[None, :, j]).abs_()
            v = v.add_(diff) if metric == "manhattan" else torch.maximum(v, diff)
        return v
    if metric == "cosine":
        return (1.0 - (q / q.norm(dim=1, keepdim=True)) @ (x / x.norm(dim=1, keepdim=True)).T).clamp(0.0, 2.0)
    return (q * q).sum(1)[:, None] + (x * x).sum(1)[None, :] - 2.0 * (q @ x.T)


def _nearest(q, x, k, metric):
    """The k smallest distances of every row, ascending, and their columns.
    Euclidean candidates come from the expansion, with room for its rounding,
    and are evaluated again as sums of squared differences."""
    q, x = q.double(), x.double()
    euclid = metric == "euclidean"
    kk = min(x.shape[0], k + 16) if euclid else k
    dist, idx = [], []
    for a, b in _blocks(q.shape[0], x.shape[0]):
        v, i = _pair_values(q[a:b], x, metric).topk(kk, dim=1, largest=False)
        if euclid:
            v = torch.stack([(q[a:b] - x[i[:, j]]).square().sum(1) for j in range(kk)], 1)
            v, o = v.sort(dim=1, stable=True)
            v, i = v[:, :k].sqrt(), i.gather(1, o)[:, :k]
        dist.append(v)
        idx.append(i)
    return torch.cat(dist), torch.cat(idx)


def exact(case, seed):
    op, n, d = case["op"], case["n"], case["d"]
    if op == "fit" or (op == "selfknn" and float(n) * n > 2.5e10):
        return None  # a whole fit follows its rounding; 500,000 x 500,000 takes too long here
    s = _inputs(case, seed)
    if op == "classify":
        dist, idx = _nearest(s["q"], s["x"], case["k"], "euclidean")
        w = 1.0 / dist
        proba = torch.zeros((case["q"], case["classes"]), dtype=torch.float64, device="cuda")
        proba.scatter_add_(1, s["y"][idx], w)
        return proba / proba.sum(1, keepdim=True)
    if op in ("knn", "metric_knn", "selfknn"):
        # indices of pairs closer than the input type resolves have no 64-bit value
        return _nearest(s["q"], s["x"], case["k"], case.get("metric", "euclidean"))[0], None
    if op == "assign":
        x, c = s["x"], s["c"].double()
        best = []
        for a, b in _blocks(n, case["c"]):
            xb = x[a:b].double()
            best.append((xb - c[_pair_values(xb, c, "euclidean").argmin(1)]).square().sum(1))
        return None, torch.cat(best)
    if op == "graph":
        x = s["x"].double()
        if case["metric"] == "cosine":
            x = x / x.norm(dim=1, keepdim=True)
        dist = []
        for a, b in _blocks(n, n):
            v = _pair_values(x[a:b], x, "euclidean")
            v[torch.arange(b - a, device="cuda"), torch.arange(a, b, device="cuda")] = float("inf")
            i = v.topk(min(n - 1, case["k"] + 16), dim=1, largest=False)[1]
            w = torch.stack([(x[a:b] - x[i[:, j]]).square().sum(1) for j in range(i.shape[1])], 1)
            w = w.sort(dim=1)[0][:, :case["k"]]
            dist.append(0.5 * w if case["metric"] == "cosine" else w.sqrt())
        return None, torch.cat(dist)
    q, x = s["q"].double(), s["x"].double()
    if op == "radius":
        dist, counts = [], []
        for a, b in _blocks(q.shape[0], n):
            at = (_pair_values(q[a:b], x, "euclidean") <= s["r"] ** 2).nonzero()
            dist.append((q[a:b][at[:, 0]] - x[at[:, 1]]).square().sum(1).sqrt())
            counts.append(torch.bincount(at[:, 0], minlength=b - a))
        return torch.cat(dist), None, torch.cat(counts)
    if case["metric"] == "euclidean":
        v = torch.zeros((q.shape[0], n), dtype=torch.float64, device="cuda")
        for j in range(d):
            v += (q[:, j, None] - x[None, :, j]).square_()
        return v.sqrt_()
    return torch.cat([_pair_values(q[a:b], x, case["metric"]) for a, b in _blocks(q.shape[0], n)])
