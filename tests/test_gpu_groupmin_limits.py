"""The group-minimum search where it works under limits: an index searched in
parts, several sets of queries, and what either may cost.  Bits are compared
with the call that has no limit (held to the CPU oracle elsewhere); times with
one another on the same box, with room for noise."""
import ctypes

import pytest
import torch

from mlrs_amd import _lib, prims

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _rows(seed, n, d, dtype=torch.float32):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn((n, d), generator=g, device=DEV, dtype=dtype)


def _search(name, xq, xt, k, metric=0):
    nq, d = xq.shape
    dist = torch.empty((nq, k), dtype=xq.dtype, device=DEV)
    idx = torch.empty((nq, k), dtype=torch.int32, device=DEV)

    def call():
        _lib.check(getattr(_lib.load(), name)(
            xq.data_ptr(), xq.numel(), nq, d, xt.data_ptr(), xt.numel(), xt.shape[0], k, metric, ctypes.c_double(2.0),
            dist.data_ptr(), idx.data_ptr(), dist.numel(), torch.cuda.current_stream(DEV).cuda_stream))
        return dist, idx
    return call


def _ms(call, reps=3):
    """The fastest of a few passes after one to warm up."""
    call()
    best = float("inf")
    for _ in range(reps):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        call()
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b))
    return best


# two parts; four; two sets of queries by sixteen parts
@pytest.mark.parametrize("nt,nq,d,k", [(600_000, 300, 50, 12), (600_000, 2_500, 50, 12), (250_000, 40_000, 50, 5),
                                       (600_000, 60, 50, 100), (400_000, 1_000, 96, 40)])
@pytest.mark.parametrize("metric", [0, 1])
def test_parts_and_sets(nt, nq, d, k, metric):
    xt, xq = _rows(nt + d, nt, d), _rows(nq, nq, d)
    xt[nt - 3] = xt[1]  # ties between the first part and the last
    xt[nt // 2] = xt[1]
    for r in (0, nt // 2 + 1, nt - 5):  # rows for the forced list, in several parts
        xt[r] *= 1e25
    xt[7, 0] = float("nan")
    xq[0] = xq[nq - 1] = xt[1]
    xq[1] = xq[nq - 2] = 0.0
    xq[2] *= 1e25  # every row is evaluated for these
    xq[nq - 3, 0] = float("nan")
    free, bound = (_search(n, xq, xt, k, metric)() for n in ("mlrs_knn_topk_f32", "mlrs_knn_topk_f32_noalloc"))
    torch.cuda.synchronize()
    assert torch.equal(free[1], bound[1])
    assert torch.equal(free[0].view(torch.int32), bound[0].view(torch.int32))


def test_a_limit_on_the_scratch_costs_no_multiple():
    """1M rows against 10,000 queries in 128 MiB: the index is copied once, not
    once per few hundred queries."""
    xt, xq = _rows(1, 1_000_000, 128), _rows(2, 10_000, 128)
    free, bound = (_ms(_search(n, xq, xt, 32)) for n in ("mlrs_knn_topk_f32", "mlrs_knn_topk_f32_noalloc"))
    assert bound < 2.2 * free, (bound, free)


@pytest.mark.parametrize("nt,nq,d,k,metric", [(5_000_000, 1_000, 3, 8, 0), (5_000_000, 4_000, 3, 8, 0),
                                              (8_000_000, 3_000, 2, 5, 0), (4_000_000, 2_000, 11, 16, 1),
                                              (20_000_000, 64, 3, 8, 0)])
def test_few_columns_against_long_indexes_fit(nt, nq, d, k, metric):
    """Searches the allocation-free entry point always took: few columns, few
    thousand queries, millions of rows."""
    xt, xq = _rows(nt + d, nt, d), _rows(nq, nq, d)
    xt[nt - 3] = xt[1]
    xq[0] = xt[1]
    free, bound = (_search(n, xq, xt, k, metric)() for n in ("mlrs_knn_topk_f32", "mlrs_knn_topk_f32_noalloc"))
    torch.cuda.synchronize()
    assert torch.equal(free[1], bound[1])
    assert torch.equal(free[0].view(torch.int32), bound[0].view(torch.int32))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_an_outlier_costs_the_others_nothing(dtype):
    """The error bound of a pair follows its own norms: one far row does not
    make every query evaluate the index."""
    xt, xq = _rows(3, 100_000, 64, dtype), _rows(4, 2_000, 64, dtype)
    name = "mlrs_knn_topk_" + ("f32" if dtype is torch.float32 else "f64")
    plain = _ms(_search(name, xq, xt, 10))
    xt[777] *= 1e4
    assert _ms(_search(name, xq, xt, 10)) < 3.0 * plain


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("metric", [0, 1])
def test_rows_the_screen_is_not_trusted_with_cost_their_share(dtype, metric):
    """300 infinite (Euclidean) or NaN (cosine) rows, more than are listed: they
    are evaluated for every query, and not the whole index."""
    xt, xq = _rows(5, 100_000, 100, dtype), _rows(6, 2_000, 100, dtype)
    name = "mlrs_knn_topk_" + ("f32" if dtype is torch.float32 else "f64")
    plain = _ms(_search(name, xq, xt, 10, metric))
    xt[1_000:1_300, 3] = float("nan") if metric else float("inf")
    assert _ms(_search(name, xq, xt, 10, metric)) < 5.0 * plain


@pytest.mark.parametrize("nt,nq,d,k,metric,dtype,kernel", [
    (100, 20_000, 50, 5, "euclidean", torch.float32, "pairwise_tile_kernel"),
    (300, 20_000, 20, 5, "cosine", torch.float64, "pairwise_tile_kernel"),
    (300, 20_000, 50, 5, "manhattan", torch.float32, "pairwise_tile_kernel"),
    (3_000, 16, 50, 1, "euclidean", torch.float64, "pairwise_tile_kernel"),
    (32, 300_000, 8, 5, "euclidean", torch.float32, "knn_lowd_kernel"),
    (1_000_000, 4_000, 2, 2, "euclidean", torch.float32, "knn_lowd_kernel"),
    (1_000_000, 4_000, 2, 2, "euclidean", torch.float64, "knn_lowd_kernel"),
    (1_000_000, 1_000, 3, 8, "euclidean", torch.float32, "knn_groupmin_kernel"),
    (1_000_000, 4_000, 8, 8, "cosine", torch.float64, "knn_groupmin_kernel"),
    (10_000, 1_000, 64, 10, "euclidean", torch.float32, "knn_groupmin_kernel"),
    (3_000, 20_000, 50, 5, "euclidean", torch.float32, "knn_groupmin_kernel"),
    (300, 300_000, 50, 1, "euclidean", torch.float32, "knn_gram_f32_kernel"),
    (300, 120_000, 130, 1, "euclidean", torch.float32, "knn_gram_f32_kernel"),
    (500_000, 2_000, 50, 1, "euclidean", torch.float32, "knn_groupmin_kernel"),
    (60_000, 2_000, 40, 10, "manhattan", torch.float64, "groupmin_tile_kernel")])
def test_family_chosen(nt, nq, d, k, metric, dtype, kernel):
    """Small indexes and few columns go where they were measured fastest, and
    with the same answer as the group minima."""
    xt, xq = _rows(nt, nt, d, dtype), _rows(nq, nq, d, dtype)
    lib = _lib.load()
    _lib.check(lib.mlrs_timing_enable(1))
    try:
        dist, idx = prims.knn_topk(xq, xt, k, metric)
        ms, launches, name = ctypes.c_double(), ctypes.c_int64(), ctypes.create_string_buffer(64)
        _lib.check(lib.mlrs_timing_read(ctypes.byref(ms), ctypes.byref(launches), name, 64))
    finally:
        _lib.check(lib.mlrs_timing_enable(0))
    assert name.value.decode() == kernel
    if metric != "manhattan":
        prims.force_path("fused")
        try:
            d2, i2 = prims.knn_topk(xq, xt, k, metric)
        finally:
            prims.force_path("auto")
        assert torch.equal(idx, i2) and torch.equal(dist, d2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_few_rows_take_narrow_tiles(dtype):
    """A matrix of 64 columns costs about half of one of 128, not as much."""
    x, y = _rows(1, 200_000, 200, dtype), _rows(2, 128, 200, dtype)
    half = y[:64].contiguous()
    assert _ms(lambda: prims.pairwise_distance(x, half)) < 0.75 * _ms(lambda: prims.pairwise_distance(x, y))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("nt,nq,metric", [(100_000, 2_000, 3), (100_000, 400, 3), (30_000, 3_000, 0)])
def test_ties_cost_no_pass_over_the_index(dtype, nt, nq, metric):
    """Rows of three values in thirty columns at one Chebyshev distance nearly
    all, and rows that are all the same: of equal distances the first rows are
    the answer, and no later one is evaluated."""
    g = torch.Generator(device="cuda").manual_seed(nt)
    name = "mlrs_knn_topk_" + ("f32" if dtype is torch.float32 else "f64")
    xt, xq = _rows(7, nt, 30, dtype), _rows(8, nq, 30, dtype)
    plain = _ms(_search(name, xq, xt, 10, metric))
    if metric:
        xt, xq = (torch.randint(0, 3, x.shape, generator=g, device=DEV).to(dtype) for x in (xt, xq))
    else:
        xt, xq = torch.ones_like(xt), torch.ones_like(xq)
    assert _ms(_search(name, xq, xt, 10, metric)) < 3.0 * plain


@pytest.mark.parametrize("dtype,metric,limit", [(torch.float32, 0, 30.0), (torch.float32, 1, 30.0),
                                                (torch.float64, 0, 10.0), (torch.float64, 1, 10.0)])
def test_clusters_the_screen_does_not_resolve(dtype, metric, limit):
    """Clusters a thousandth of their spacing wide, where every group has a row of
    the query's cluster: f64 searches take a second scan in their precision, f32
    ones evaluate the cluster's rows, neither every row of every group."""
    name = "mlrs_knn_topk_" + ("f32" if dtype is torch.float32 else "f64")
    xt, xq = _rows(9, 100_000, 128, dtype), _rows(10, 5_000, 128, dtype)
    plain = _ms(_search(name, xq, xt, 16, metric))
    g = torch.Generator(device="cuda").manual_seed(11)
    centres = 20.0 * torch.rand((20, 128), generator=g, device=DEV, dtype=dtype) - 10.0
    xt, xq = (centres[torch.randint(0, 20, (x.shape[0],), generator=g, device=DEV)] + 0.01 * x for x in (xt, xq))
    assert _ms(_search(name, xq, xt, 16, metric)) < limit * plain


@pytest.mark.parametrize("metric", [2, 3])
def test_metric_sets(metric):
    """Two sets of queries of the exact tiles' minima."""
    nt, nq = 300_000, 2_500
    xt, xq = _rows(nt, nt, 4), _rows(nq, nq, 4)
    xt[nt - 3] = xt[1]
    xt[7, 0], xt[8, 1] = float("nan"), float("inf")
    xq[0] = xq[nq - 1] = xt[1]
    xq[nq - 2, 0] = float("inf")
    free, bound = (_search(n, xq, xt, 9, metric)() for n in ("mlrs_knn_topk_f32", "mlrs_knn_topk_f32_noalloc"))
    torch.cuda.synchronize()
    assert torch.equal(free[1], bound[1])
    assert torch.equal(free[0].view(torch.int32), bound[0].view(torch.int32))
    at = [0, 1, nq // 2, nq - 3, nq - 2, nq - 1]
    prims.force_path("generic")
    try:
        dist, idx = prims.knn_topk(xq[at].contiguous(), xt, 9, "manhattan" if metric == 2 else "chebyshev")
    finally:
        prims.force_path("auto")
    assert torch.equal(idx, bound[1][at].long()) and torch.equal(dist, bound[0][at])
