"""GPU parity of the group-minimum search (knn_groupmin.hip) with the CPU
oracle, bit for bit, where it can go wrong: index sizes around a 16-row group,
a 32-row tile and the 128 rows of one store; row widths around the 8-column
steps; both selection kernels (a workgroup per query below 1,000 queries, a
wave per query from there) and both list lengths; rows the screen is not
trusted with (norms past the f32 range, infinities, NaN) singly and more than
are listed; ties past the candidate lists; clusters and offsets the screen
does not resolve; the parts of an index too large for the allocation-free
entry point's scratch."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from mlrs_amd import _lib, prims

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.fixture(autouse=True)
def _family():
    prims.force_path("fused")
    yield
    prims.force_path("auto")


def _check(xq, xt, k, metric="euclidean"):
    wd, wi = oracle.knn_topk(xq, xt, k, metric)
    gd, gi = prims.knn_topk(torch.from_numpy(xq).to(DEV), torch.from_numpy(xt).to(DEV), k, metric)
    gd, gi = gd.cpu().numpy(), gi.cpu().numpy()
    bits = np.int32 if gd.dtype == np.float32 else np.int64
    assert np.array_equal(gi, wi.astype(np.int64)), np.argwhere(gi != wi)[:3].tolist()
    assert np.array_equal(gd.view(bits), wd.view(bits)), np.argwhere(gd.view(bits) != wd.view(bits))[:3].tolist()


def _rows(seed, n, d, dtype):
    return np.random.default_rng(seed).standard_normal((n, d)).astype(dtype)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("nt,d,k,nq", [
    (2, 1, 2, 1), (16, 3, 5, 3), (31, 8, 31, 4), (32, 9, 32, 31), (33, 7, 33, 33), (127, 16, 64, 5), (128, 17, 65, 127),
    (129, 24, 128, 128), (4097, 50, 16, 129), (1000, 63, 17, 999), (1000, 64, 17, 1000), (5000, 65, 64, 1003),
    (2049, 120, 1, 1001), (700, 127, 10, 64), (700, 128, 10, 64), (700, 129, 10, 64), (300, 192, 100, 20),
    (300, 193, 3, 20), (300, 255, 7, 20), (300, 256, 7, 1000)])
def test_edges(dtype, nt, d, k, nq):
    xt, xq = _rows(nt + d, nt, d, dtype), _rows(nq + k, nq, d, dtype)
    xt[nt // 2] = xt[nt - 1]  # a tie
    for metric in ("euclidean", "cosine"):
        _check(xq, xt, k, metric)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("metric", ["euclidean", "cosine"])
@pytest.mark.parametrize("d,k,nq", [(6, 12, 60), (50, 100, 60), (50, 12, 1040)])
def test_rows_the_screen_is_not_trusted_with(dtype, metric, d, k, nq):
    """A few such rows go to every query from a list; more than it holds, and
    queries of the kind, have every row evaluated."""
    xt, xq = _rows(3, 1500, d, dtype), _rows(4, nq, d, dtype)
    xt[[10, 11]] = 0.0
    xt[20, 0] = np.nan
    xt[30, 0], xt[31, d - 1] = np.inf, -np.inf
    for r, scale in ((40, 1e18), (41, 1e30), (42, 1e-25), (43, 1e-35)):
        xt[r] *= dtype(scale)
    xq[:20] = xt[[10, 11, 12, 20, 21, 30, 31, 32, 40, 41, 42, 43, 44, 5, 6, 7, 8, 9, 1, 2]]
    xq[21] *= dtype(1e30)
    _check(xq, xt, k, metric)
    xt[100:500] *= dtype(1e25)
    _check(xq, xt, k, metric)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("metric", ["euclidean", "cosine"])
@pytest.mark.parametrize("nq", [40, 1000])
def test_ties_past_the_candidate_lists(dtype, metric, nq):
    """Far more groups than a query lists stand at its k-th minimum."""
    rng = np.random.default_rng(9)
    xt = rng.integers(0, 2, (20_000, 4)).astype(dtype)
    _check(xt[:nq].copy(), xt, 25, metric)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("nq", [30, 1000])
def test_distances_the_screen_does_not_resolve(dtype, nq):
    """Clusters a thousandth of their spacing wide, and a common offset."""
    rng = np.random.default_rng(11)
    centres = rng.uniform(-10, 10, (8, 20))
    xt = (centres[rng.integers(0, 8, 6000)] + 1e-3 * rng.standard_normal((6000, 20))).astype(dtype)
    _check(xt[:nq].copy(), xt, 20)
    _check((xt[:nq] + dtype(500)), (xt + dtype(500)), 20)


@pytest.mark.parametrize("n,d,k,metric", [(2500, 5, 15, "euclidean"), (1300, 50, 100, "euclidean"),
                                          (1100, 33, 9, "cosine")])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_graph(dtype, n, d, k, metric):
    x = _rows(n, n, d, dtype)
    x[100:140] = x[3]
    wi, wd = oracle.knn_graph(x, k, metric)
    gi, gd = prims.knn_graph(torch.from_numpy(x).to(DEV), k, metric)
    assert np.array_equal(gi.cpu().numpy(), wi.astype(np.int64))
    assert np.array_equal(gd.cpu().numpy().view(np.int64), wd.view(np.int64))


@pytest.mark.parametrize("nt,d,metric", [(300_000, 50, 0), (300_000, 50, 1), (260_000, 64, 0)])
def test_noalloc_index_parts(nt, d, metric):
    """Rows that are not 16-byte aligned are copied a part at a time there."""
    g = torch.Generator(device="cpu").manual_seed(nt + d)
    xt = torch.randn((nt, d), generator=g).to(DEV)
    xt[nt - 3] = xt[1]
    xt[nt - 5] *= 1e25  # a row for the forced list, in the last part
    xq = torch.randn((300, d), generator=g).to(DEV)
    xq[0] = xt[1]
    out = []
    for name in ("mlrs_knn_topk_f32", "mlrs_knn_topk_f32_noalloc"):
        dist = torch.empty((300, 12), dtype=torch.float32, device=DEV)
        idx = torch.empty((300, 12), dtype=torch.int32, device=DEV)
        _lib.check(getattr(_lib.load(), name)(
            xq.data_ptr(), xq.numel(), 300, d, xt.data_ptr(), xt.numel(), nt, 12, metric, ctypes.c_double(2.0),
            dist.data_ptr(), idx.data_ptr(), dist.numel(), torch.cuda.current_stream(DEV).cuda_stream))
        out.append((dist.view(torch.int32), idx))
    torch.cuda.synchronize()
    assert torch.equal(out[0][1], out[1][1]) and torch.equal(out[0][0], out[1][0])


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("metric", ["manhattan", "chebyshev"])
@pytest.mark.parametrize("nt,d,k,nq", [(5, 1, 5, 1), (33, 7, 33, 65), (129, 16, 100, 63), (4100, 17, 10, 1000),
                                       (2000, 40, 65, 200), (700, 256, 3, 64), (20_000, 3, 12, 30)])
def test_metric_arms(dtype, metric, nt, d, k, nq):
    """The exact tiles' minima: edges of the 64 x 128 tile, values past the f32
    range, infinities, NaN, ties."""
    prims.force_path("auto")
    xt, xq = _rows(nt + d, nt, d, dtype), _rows(nq, nq, d, dtype)
    xt[nt // 2] = xt[nt - 1]
    if nt > 100:
        xt[3, 0], xt[4, d - 1], xt[5, 0] = np.nan, np.inf, -np.inf
        xt[6] *= dtype(1e30)
        if dtype is np.float64:
            xt[7] *= 1e200
        xq[0] = xt[nt - 1]
        xq[nq - 1, 0] = np.inf
        if nq > 60:
            xq[nq - 2, 0] = np.nan
    _check(xq, xt, k, metric)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("metric", ["euclidean", "cosine", "manhattan", "chebyshev"])
@pytest.mark.parametrize("nx,ny,d", [(1, 1, 1), (63, 129, 15), (64, 128, 16), (65, 127, 17), (130, 300, 50)])
def test_pairwise_tile_edges(dtype, metric, nx, ny, d):
    x, y = _rows(nx, nx, d, dtype), _rows(ny + 1, ny, d, dtype)
    want = oracle.pairwise(x, y, metric, sqrt=True)
    got = prims.pairwise_distance(torch.from_numpy(x).to(DEV), torch.from_numpy(y).to(DEV), metric, sqrt=True)
    bits = np.int32 if dtype == np.float32 else np.int64
    assert np.array_equal(got.cpu().numpy().view(bits), want.view(bits))


@pytest.mark.parametrize("d", [5, 16, 17, 100, 128])
def test_two_query_blocks(d):
    """Searches of 2^26 pairs and more, up to 128 columns: two query blocks per
    workgroup, the last of them partly and wholly empty; rows of every scale,
    down to where they share one."""
    xt, xq = _rows(d, 9001, d, np.float32), _rows(d + 1, 7500 if d % 2 else 7700, d, np.float32)
    rng = np.random.default_rng(d)
    for x in (xt, xq):
        rows = rng.choice(len(x), 2000, replace=False)
        x[rows] *= np.exp2(rng.integers(-60, 12, 2000)).astype(np.float32)[:, None]
    xt[17] = xt[9000]
    _check(xq, xt, 7)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("metric", ["euclidean", "cosine", "manhattan"])
@pytest.mark.parametrize("nt,k", [(135, 100), (300, 100), (333, 128), (1300, 70)])
@pytest.mark.parametrize("d", [5, 50, 140])
def test_last_batch_of_rows(dtype, metric, nt, k, d):
    """Lists of two blocks where the last, partly filled batch of 64 rows holds
    the nearest: for queries that evaluate every row (untrusted themselves, or
    more untrusted rows than are listed) and for the others."""
    prims.force_path("auto" if metric == "manhattan" else "fused")
    rng = np.random.default_rng(nt + k + d)
    xt, xq = (rng.standard_normal((n, d)) for n in (nt, 64))
    xt = xt[np.argsort(-((xt - xq[0]) ** 2).sum(1))]
    xt, xq = np.ascontiguousarray(xt.astype(dtype)), xq.astype(dtype)
    xq[10:20] *= dtype(1e25)
    _check(xq, xt, k, metric)
    far = max(nt // 4, min(nt - k, 300))
    xt[:far] *= dtype(1e25)
    _check(xq, xt, k, metric)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("nq", [40, 1000])
@pytest.mark.parametrize("scale", [30.0, 1e3, 1e8])
def test_outliers(dtype, nq, scale):
    """Rows and queries far from the rest, near one another among them."""
    xt, xq = _rows(5, 3000, 20, dtype), _rows(6, nq, 20, dtype)
    xt[100:130] *= dtype(scale)
    xt[200:240] += dtype(scale)
    xq[:30] = xt[100:130] + dtype(0.5) * xq[:30]
    xq[30:38] = xt[200:208]
    _check(xq, xt, 20)
    _check(xq, np.ascontiguousarray(xt[90:260]), 100)


def _clusters(seed, nt, nq, d, width, count, dtype):
    rng = np.random.default_rng(seed)
    centres = rng.uniform(-10, 10, (count, d))
    return tuple((centres[rng.integers(0, count, n)] + width * rng.standard_normal((n, d))).astype(dtype) for n in (nt, nq))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("metric", ["euclidean", "cosine"])
@pytest.mark.parametrize("nt,nq,d,k", [(30_000, 40, 20, 10), (6_000, 1_100, 37, 100), (30_100, 1_003, 5, 24)])
@pytest.mark.parametrize("width", [1e-2, 1e-5])
def test_clusters_past_the_lists(dtype, metric, nt, nq, d, k, width):
    """Clusters of more groups than are listed: the pass over the groups, its
    probe and its gathered rows, in both selections."""
    xt, xq = _clusters(nt + d, nt, nq, d, width, 3, dtype)
    xt[nt - 100:nt - 50] = xt[50:100]
    _check(xq, xt, k, metric)


@pytest.mark.parametrize("dtype,metric", [(np.float64, "euclidean"), (np.float64, "cosine")])
@pytest.mark.parametrize("d", [3, 31, 33, 64, 100, 150, 193, 256])
@pytest.mark.parametrize("nt,nq,k", [(100_001, 3_000, 10), (300_000, 1_001, 70)])
def test_precise_scan(dtype, metric, d, nt, nq, k):
    """Searches large enough for the second scan: its column counts, partly
    filled query blocks and tiles, rows left out, flagged queries among others;
    against the exact tiles."""
    xt, xq = _clusters(nt + d, nt, nq, d, 1e-3, 4, dtype)
    rng = np.random.default_rng(d)
    far = rng.choice(nq, nq // 3, replace=False)
    xq[far] = rng.uniform(-10, 10, (len(far), d)).astype(dtype)  # not flagged
    xt[nt - 90:nt - 60] = xt[60:90]
    xt[17, 0], xt[18, d - 1] = np.nan, np.inf
    xt[19] *= dtype(1e25)
    xq[0], xq[1] = xt[19], 0
    xt, xq = (torch.from_numpy(x).to(DEV) for x in (xt, xq))
    got = prims.knn_topk(xq, xt, k, metric)
    prims.force_path("generic")
    want = prims.knn_topk(xq, xt, k, metric)
    if metric == "euclidean" and nq == 1_001:  # f32 rows, f64 values
        x = xt[:20_000].float()
        wi, wd = prims.knn_graph(x, k, metric)
        prims.force_path("fused")
        gi, gd = prims.knn_graph(x, k, metric)
        assert torch.equal(gi, wi) and torch.equal(gd.view(torch.int64), wd.view(torch.int64))
    assert torch.equal(got[1], want[1]) and torch.equal(got[0].view(torch.int32), want[0].view(torch.int32))


@pytest.mark.parametrize("p", [3.0, 2.0 ** 36, 2.0 ** 40])
def test_root_ties_of_large_exponents(p):
    """Sums that differ by more than the minima's rounding and whose roots are one
    double: the graph ranks them by index."""
    rng = np.random.default_rng(3)
    steps = 0.69 / (p * 2.0 ** -53) if p > 3 else 1e14
    x = np.stack([np.ones(2000), 1.0 - (np.floor(steps) + rng.integers(0, 31, 2000)) * 2.0 ** -53], 1)
    x[0] = 0.0
    x = torch.from_numpy(x).to(DEV)
    out = []
    for family in ("auto", "generic"):
        prims.force_path(family)
        out.append(prims.knn_graph(x, 15, "minkowski", p=p))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1].view(torch.int64), out[1][1].view(torch.int64))
