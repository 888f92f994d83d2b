"""k-means on the GPU against the oracle's restatement of src/kmeans.cpp:
every assignment, centroid, normed difference and final index must be
bit-identical."""
import numpy as np
import pytest
import torch

from oracle import kmeans_oracle as KO
from thcpp_amd import _lib as L

pytestmark = pytest.mark.gpu


def _lattice(n, L_=5.0):
    i, j, k = np.meshgrid(np.arange(n), np.arange(n), np.arange(n), indexing="ij")
    return np.stack([i, j, k], -1).reshape(-1, 3) * (L_ / n)


@pytest.mark.parametrize("n,k,seed", [(5000, 97, 1), (20000, 1000, 2), (3, 1, 3), (777, 777, 4)])
def test_classify_random(ctx, n, k, seed):
    rng = np.random.default_rng(seed)
    grid = rng.uniform(0, 10, size=(n, 3))
    cen = rng.uniform(0, 10, size=(k, 3))
    got = ctx.classify_grid_points(grid, cen).cpu().numpy()
    np.testing.assert_array_equal(got, KO.classify(grid, cen))


def test_classify_lattice_ties(ctx):
    """Centroids on lattice points and midpoints: many exactly equal distances."""
    grid = _lattice(16)
    rng = np.random.default_rng(5)
    pick = rng.choice(grid.shape[0], 300, replace=False)
    cen = grid[pick].copy()
    cen[::3] += (5.0 / 16) / 2  # midpoints -> ties between neighbours
    got = ctx.classify_grid_points(grid, cen).cpu().numpy()
    np.testing.assert_array_equal(got, KO.classify(grid, cen))


def test_classify_duplicate_centroids(ctx):
    """Identical centroids: the first index must win."""
    rng = np.random.default_rng(6)
    grid = rng.uniform(0, 4, size=(3000, 3))
    cen = rng.uniform(0, 4, size=(50, 3))
    cen[30:40] = cen[5]
    got = ctx.classify_grid_points(grid, cen).cpu().numpy()
    ref = KO.classify(grid, cen)
    np.testing.assert_array_equal(got, ref)
    assert not np.isin(np.arange(30, 40), ref).any()


@pytest.mark.parametrize("n,k", [(10000, 64), (50000, 2000)])
def test_update_centroids(ctx, n, k):
    rng = np.random.default_rng(n)
    grid = rng.uniform(0, 7, size=(n, 3))
    rho = rng.uniform(0.1, 2.0, size=n)
    gmap = rng.integers(0, k, size=n).astype(np.int32)
    gmap[:k] = np.arange(k)  # no empty cluster
    got, st = ctx.update_centroids(rho, grid, gmap, k)
    ref, crit = KO.update_centroids(rho, grid, gmap, k)
    assert st == L.THC_OK and crit == 0
    np.testing.assert_array_equal(got.cpu().numpy(), ref)


def test_update_centroids_empty_cluster(ctx):
    rng = np.random.default_rng(9)
    grid = rng.uniform(0, 7, size=(1000, 3))
    rho = rng.uniform(0.1, 2.0, size=1000)
    gmap = rng.integers(0, 10, size=1000).astype(np.int32)
    gmap[gmap == 4] = 5
    _, st = ctx.update_centroids(rho, grid, gmap, 10)
    _, crit = KO.update_centroids(rho, grid, gmap, 10)
    assert crit == 1 and st == L.THC_ERR_EMPTY_CLUSTER


@pytest.mark.parametrize("n,k", [(4096, 40), (30000, 700)])
def test_map_to_grid(ctx, n, k):
    rng = np.random.default_rng(k)
    grid = rng.uniform(0, 9, size=(n, 3))
    cen = rng.uniform(0, 9, size=(k, 3))
    got, st = ctx.map_to_grid(grid, cen)
    ref, dups = KO.map_to_grid(grid, cen)
    np.testing.assert_array_equal(got.cpu().numpy(), ref)
    assert (st == L.THC_WARN_DUPLICATE_INDICES) == (dups > 0)


def test_map_to_grid_lattice(ctx):
    grid = _lattice(20, 6.0)
    rng = np.random.default_rng(3)
    cen = grid[rng.choice(grid.shape[0], 200, replace=False)] + (6.0 / 20) / 2  # equidistant to 8 points
    got, _ = ctx.map_to_grid(grid, cen)
    ref, _ = KO.map_to_grid(grid, cen)
    np.testing.assert_array_equal(got.cpu().numpy(), ref)


@pytest.mark.parametrize("n,k,seed", [(32768, 128, 0), (1000, 7, 3), (65536, 10, 11), (65535, 33, 5),
                                      (262144, 1024, 0), (884736, 3456, 0)])
def test_initial_indices(n, k, seed):
    from thcpp_amd.api import Context
    np.testing.assert_array_equal(Context.initial_indices(n, k, seed), KO.initial_indices(n, k, seed))


def test_kmeans_cfg0_every_iteration(ctx, cfg0, cfg0_kmeans):
    s, ref = cfg0, cfg0_kmeans
    out = ctx.kmeans(s.grid, s.rho, s.K, s.max_it, -1.0, 0, want_map=True, want_centroids=True)
    assert out["status"] == L.THC_OK
    assert out["iters"] == ref["iters"] == s.max_it
    np.testing.assert_array_equal(out["diffs"], ref["diffs"])
    np.testing.assert_array_equal(out["pcts"], ref["pcts"])
    np.testing.assert_array_equal(out["interp_idx"].cpu().numpy(), ref["interp_idx"])
    np.testing.assert_array_equal(out["grid_map"].cpu().numpy(), ref["maps"][-1])
    np.testing.assert_array_equal(out["centroids"].cpu().numpy(), ref["centroids"])


@pytest.mark.parametrize("iters", [1, 2, 7])
def test_kmeans_maps_per_iteration(ctx, cfg0, cfg0_kmeans, iters):
    s, ref = cfg0, cfg0_kmeans
    out = ctx.kmeans(s.grid, s.rho, s.K, iters, -1.0, 0, want_map=True)
    np.testing.assert_array_equal(out["grid_map"].cpu().numpy(), ref["maps"][iters - 1])
    np.testing.assert_array_equal(out["diffs"], ref["diffs"][:iters])


def test_kmeans_graph_vs_eager_and_replay(ctx, ctx_graph, cfg0, cfg0_kmeans):
    s = cfg0
    a = ctx_graph.kmeans(s.grid, s.rho, s.K, s.max_it, -1.0, 0)
    b = ctx_graph.kmeans(s.grid, s.rho, s.K, s.max_it, -1.0, 0)  # graph replay
    c = ctx.kmeans(s.grid, s.rho, s.K, s.max_it, -1.0, 0)
    for o in (a, b, c):
        np.testing.assert_array_equal(o["interp_idx"].cpu().numpy(), cfg0_kmeans["interp_idx"])
        np.testing.assert_array_equal(o["diffs"], cfg0_kmeans["diffs"])


def test_kmeans_threshold_converges(ctx, cfg0, cfg0_kmeans):
    s = cfg0
    thr = float(cfg0_kmeans["diffs"][8]) * 1.0000001
    ref = KO.kmeans(s.grid, s.rho, s.K, 50, thr, 0)
    out = ctx.kmeans(s.grid, s.rho, s.K, 50, thr, 0)
    assert out["iters"] == ref["iters"] and out["converged"]
    np.testing.assert_array_equal(out["interp_idx"].cpu().numpy(), ref["interp_idx"])
    np.testing.assert_array_equal(out["diffs"], ref["diffs"])


def test_kmeans_threshold_equal_leaves_zeros(ctx, cfg0, cfg0_kmeans):
    """diff == threshold on the last iteration: neither branch maps, indices stay 0
    (kmeans.cpp:239,250)."""
    s = cfg0
    it = 6
    thr = float(cfg0_kmeans["diffs"][it - 1])
    ref = KO.kmeans(s.grid, s.rho, s.K, it, thr, 0)
    out = ctx.kmeans(s.grid, s.rho, s.K, it, thr, 0)
    assert not ref["interp_idx"].any()
    assert out["interp_zeroed"] and not out["interp_idx"].cpu().numpy().any()


def test_kmeans_seeds(ctx, cfg0):
    s = cfg0
    for seed in (1, 12345):
        ref = KO.kmeans(s.grid, s.rho, 64, 8, -1.0, seed)
        out = ctx.kmeans(s.grid, s.rho, 64, 8, -1.0, seed)
        np.testing.assert_array_equal(out["interp_idx"].cpu().numpy(), ref["interp_idx"])
        np.testing.assert_array_equal(out["diffs"], ref["diffs"])


def test_kmeans_empty_cluster(ctx):
    """Zero density where a centroid starts -> weight 0 -> the reference exits."""
    g = _lattice(12, 4.0)
    rho = np.ones(g.shape[0])
    idx = KO.initial_indices(g.shape[0], 20, 0)
    first = KO.classify(g, g[idx])
    rho[first == 3] = 0.0
    ref = KO.kmeans(g, rho, 20, 5, -1.0, 0)
    out = ctx.kmeans(g, rho, 20, 5, -1.0, 0)
    assert ref["status"] == 1
    assert out["status"] == L.THC_ERR_EMPTY_CLUSTER


def test_kmeans_full_size_prefix(ctx):
    """The 64-atom, 64^3-grid system with N_mu = 1024: first 4 iterations and the
    points they give, against the oracle."""
    from thcpp_amd import synthetic
    s = synthetic.make_config("diamond64_n64_k1024")
    ref = KO.kmeans(s.grid, s.rho, s.K, 4, -1.0, 0)
    out = ctx.kmeans(s.grid, s.rho, s.K, 4, -1.0, 0)
    np.testing.assert_array_equal(out["diffs"], ref["diffs"])
    np.testing.assert_array_equal(out["pcts"], ref["pcts"])
    np.testing.assert_array_equal(out["interp_idx"].cpu().numpy(), ref["interp_idx"])


def test_device_sqrt_correctly_rounded(ctx):
    """The device FP64 square root of the distance kernels (thc_device_sqrt)
    against numpy's IEEE sqrt, bit for bit: log-uniform arguments over the
    whole normal range, subnormals, exact squares, the doubles next to exact
    squares and next to the midpoints between adjacent square roots (the
    hardest cases for a correctly rounded sqrt), 0, -0 and inf."""
    import ctypes
    rng = np.random.default_rng(11)
    parts = [np.exp(rng.uniform(np.log(1e-300), np.log(1e300), 1 << 20)),
             rng.uniform(0, 1, 1 << 14) * 2.0 ** -1022,  # subnormals
             np.array([0.0, -0.0, np.inf, 1.0, 4.0, 2.0, 0.5, 2.0 ** -1074, np.finfo(np.float64).max])]
    s = np.exp(rng.uniform(np.log(1e-150), np.log(1e150), 1 << 18))
    sq = s * s  # squares of doubles, rounded
    parts += [sq, np.nextafter(sq, 0), np.nextafter(sq, np.inf)]
    mid = (s + np.nextafter(s, np.inf)) / 2  # midpoints between adjacent roots
    m2 = mid * mid
    parts += [m2, np.nextafter(m2, 0), np.nextafter(m2, np.inf)]
    x = np.concatenate(parts)
    x = x[np.isfinite(x) | np.isinf(x)]
    xd = torch.from_numpy(x).to(ctx.device)
    yd = torch.empty_like(xd)
    print("device sqrt: %d arguments" % x.size, flush=True)
    st = L.lib().thc_device_sqrt(ctx.h, ctypes.c_void_p(xd.data_ptr()), x.size, ctypes.c_void_p(yd.data_ptr()))
    assert st == L.THC_OK
    got = yd.cpu().numpy()
    ref = np.sqrt(x)
    bad = np.flatnonzero(got.view(np.int64) != ref.view(np.int64))
    assert bad.size == 0, (bad.size, x[bad[:5]], got[bad[:5]], ref[bad[:5]])


@pytest.mark.parametrize("n,k,big", [(70000, 301, 42000), (200000, 90, 1500), (3000, 2, 1024), (3000, 2, 1025),
                                     (2000, 3, 512), (2000, 3, 513)])
def test_update_centroids_cluster_sizes(ctx, n, k, big):
    """Clusters either side of what a workgroup sums at a time (512), keeps in registers (1024) and finds in its
    bucket (8 n / k), members spread over several 65536-point windows of the index range."""
    rng = np.random.default_rng(n + k + big)
    grid = rng.uniform(0, 7, size=(n, 3))
    rho = rng.uniform(0.1, 2.0, size=n)
    gmap = np.empty(n, dtype=np.int32)
    order = rng.permutation(n)
    gmap[order[:big]] = k // 2
    rest = np.array([c for c in range(k) if c != k // 2])
    gmap[order[big:]] = rest[np.arange(n - big) % len(rest)]
    got, st = ctx.update_centroids(rho, grid, gmap, k)
    ref, crit = KO.update_centroids(rho, grid, gmap, k)
    assert st == L.THC_OK and crit == 0
    np.testing.assert_array_equal(got.cpu().numpy(), ref)


@pytest.mark.parametrize("k", [1, 256, 257, 1024, 1025, 2048, 2049, 4096])
def test_kmeans_cluster_counts(ctx, k):
    """Either side of the assignment's centroids-per-thread variants; a loop that no threshold can stop and one
    with a threshold that is never reached give the same run."""
    rng = np.random.default_rng(k)
    n = 6000
    grid = rng.uniform(0, 9, size=(n, 3))
    rho = rng.uniform(0.1, 2.0, size=n)
    ref = KO.kmeans(grid, rho, k, 3, -1.0, 5)
    for thr in (-1.0, 0.0 if ref["diffs"][-1] > 0 else -2.0):
        out = ctx.kmeans(grid, rho, k, 3, thr, 5, want_map=True, want_centroids=True)
        np.testing.assert_array_equal(out["interp_idx"].cpu().numpy(), ref["interp_idx"])
        np.testing.assert_array_equal(out["diffs"], ref["diffs"])
        np.testing.assert_array_equal(out["pcts"], ref["pcts"])
        np.testing.assert_array_equal(out["centroids"].cpu().numpy(), ref["centroids"])


def test_kmeans_dense_clump(ctx):
    """All but a few points in a clump that holds one starting centroid: a cluster beyond its bucket, and tiles
    whose bounds keep almost every centroid."""
    rng = np.random.default_rng(8)
    n, k = 20000, 60
    grid = rng.uniform(0, 30, size=(n, 3))
    grid[100:] = 15.0 + 0.4 * rng.standard_normal((n - 100, 3))
    rho = rng.uniform(0.1, 2.0, size=n)
    init = np.concatenate([np.arange(k - 1), [150]]).astype(np.int32)
    ref = KO.kmeans(grid, rho, k, 4, -1.0, 0, init_idx=init, keep_maps=True)
    assert np.bincount(ref["maps"][0], minlength=k).max() > 8 * (n // k + 1)
    for thr in (-1.0, 1e-300):
        out = ctx.kmeans(grid, rho, k, 4, thr, 0, init_idx=init, want_map=True)
        np.testing.assert_array_equal(out["interp_idx"].cpu().numpy(), ref["interp_idx"])
        np.testing.assert_array_equal(out["diffs"], ref["diffs"])
        np.testing.assert_array_equal(out["grid_map"].cpu().numpy(), ref["maps"][-1])


@pytest.mark.parametrize("n,k,seed", [(40, 12, 132), (40, 12, 1857), (60, 25, 1710)])
def test_kmeans_empty_cluster_later(ctx, n, k, seed):
    """A weight that vanishes in the second iteration (densities over 13 decades) stops the run there, whether or
    not the loop waits for the differences."""
    rng = np.random.default_rng(seed)
    grid = rng.integers(0, 5, size=(n, 3)).astype(float)
    rho = 10.0 ** rng.uniform(-12, 1, size=n)
    ref = KO.kmeans(grid, rho, k, 8, -1.0, seed)
    assert ref["status"] == 1 and ref["iters"] == 2
    for thr in (-1.0, 0.0):
        out = ctx.kmeans(grid, rho, k, 8, thr, seed)
        assert out["status"] == L.THC_ERR_EMPTY_CLUSTER
        assert out["iters"] == 2
        assert out["diffs"][0] == ref["diffs"][0]


@pytest.mark.parametrize("n,k", [(4000, 1), (9000, 300), (30000, 1500)])
@pytest.mark.parametrize("stop", [0, 1, 2, 5])
def test_kmeans_stops_beside_next_iteration(ctx, n, k, stop):
    """A threshold that stops the loop while the next iteration is on its way: the points, map, centroids and
    differences are those of the iteration that it stopped at."""
    rng = np.random.default_rng(k + stop)
    grid = rng.uniform(0, 9, size=(n, 3))
    rho = rng.uniform(0.1, 2.0, size=n)
    run = KO.kmeans(grid, rho, k, 6, -1.0, 7)["diffs"]
    thr = float(np.nextafter(run[: stop + 1].min(), np.inf))
    ref = KO.kmeans(grid, rho, k, 20, thr, 7, keep_maps=True)
    assert ref["status"] in (0, 2) and ref["iters"] <= stop + 1  # 2: two centroids on one point
    out = ctx.kmeans(grid, rho, k, 20, thr, 7, want_map=True, want_centroids=True)
    assert out["status"] == (L.THC_WARN_DUPLICATE_INDICES if ref["status"] else L.THC_OK) and out["converged"]
    assert out["iters"] == ref["iters"]
    np.testing.assert_array_equal(out["interp_idx"].cpu().numpy(), ref["interp_idx"])
    np.testing.assert_array_equal(out["diffs"], ref["diffs"])
    np.testing.assert_array_equal(out["pcts"], ref["pcts"])
    np.testing.assert_array_equal(out["grid_map"].cpu().numpy(), ref["maps"][-1])
    np.testing.assert_array_equal(out["centroids"].cpu().numpy(), ref["centroids"])


@pytest.mark.parametrize("n,k,seed", [(40, 12, 132), (40, 12, 1857), (60, 25, 1710)])
def test_kmeans_converged_before_empty_cluster(ctx, n, k, seed):
    """The runs of test_kmeans_empty_cluster_later with a threshold that ends them after the first iteration: the
    weight that vanishes in the second, which has been started by then, is none of their business."""
    rng = np.random.default_rng(seed)
    grid = rng.integers(0, 5, size=(n, 3)).astype(float)
    rho = 10.0 ** rng.uniform(-12, 1, size=n)
    thr = 2 * KO.kmeans(grid, rho, k, 8, -1.0, seed)["diffs"][0]
    _check_converged_first(ctx, grid, rho, k, thr, seed, None)


def test_kmeans_converged_before_empty_cluster_many(ctx):
    """The same with 1200 centroids, whose loop control ends well after the next iteration has started.  On a line
    away from the rest, the middle one of three centroids has two heavy points and a light one; its neighbours move
    towards the heavy ones and take them."""
    rng = np.random.default_rng(12)
    n, k = 6000, 1200
    grid = rng.uniform(0, 9, size=(n, 3))
    rho = rng.uniform(0.1, 2.0, size=n)
    grid[:7, 1:] = 0.0
    grid[:7, 0] = [-26.0, -23.5, -22.0, -20.0, -18.0, -16.5, -14.0]
    rho[:7] = [1e-3, 1.0, 1.0, 1e-12, 1.0, 1.0, 1e-3]
    init = np.concatenate([[0, 3, 6], np.arange(100, 100 + k - 3)]).astype(np.int32)
    run = KO.kmeans(grid, rho, k, 8, -1.0, 0, init_idx=init)
    assert run["status"] == 1 and run["iters"] == 2
    _check_converged_first(ctx, grid, rho, k, 2 * run["diffs"][0], 0, init)


def _check_converged_first(ctx, grid, rho, k, thr, seed, init):
    ref = KO.kmeans(grid, rho, k, 8, thr, seed, init_idx=init)
    assert ref["iters"] == 1 and ref["status"] in (0, 2)
    out = ctx.kmeans(grid, rho, k, 8, thr, seed, init_idx=init, want_centroids=True)
    assert out["status"] == (L.THC_WARN_DUPLICATE_INDICES if ref["status"] else L.THC_OK)
    assert out["converged"] and out["iters"] == 1
    np.testing.assert_array_equal(out["interp_idx"].cpu().numpy(), ref["interp_idx"])
    np.testing.assert_array_equal(out["centroids"].cpu().numpy(), ref["centroids"])


@pytest.mark.parametrize("k", [40, 1500])
def test_kmeans_difference_not_a_number(ctx, k):
    """A density that is not a number leaves no difference to compare: after the last iteration the reference maps
    neither set of centroids and the points stay zero, whether the difference comes in the loop or after it."""
    rng = np.random.default_rng(k)
    n = 5000
    grid = rng.uniform(0, 9, size=(n, 3))
    rho = rng.uniform(0.1, 2.0, size=n)
    rho[77] = np.nan
    for thr in (-1.0, 1e-3):
        ref = KO.kmeans(grid, rho, k, 1, thr, 1)
        assert ref["iters"] == 1 and np.isnan(ref["diffs"]).all() and not ref["interp_idx"].any()
        out = ctx.kmeans(grid, rho, k, 1, thr, 1)
        assert out["iters"] == 1 and not out["converged"] and out["interp_zeroed"]
        assert np.isnan(out["diffs"]).all()
        assert not out["interp_idx"].cpu().numpy().any()


def _windows_map(case):
    """(n, k, map): cluster sizes and index ranges at the edges of the sums' 65536-point windows and 256-member runs."""
    rng = np.random.default_rng(3)
    if case == "dense":  # two windows full of one cluster, then a window of another
        return 140000, 2, (np.arange(140000) >= 131072).astype(np.int32)
    if case == "runs":  # 255, 256, 257, 512, 513 members in five windows, an empty window between, ends of windows
        n = 6 * 65536 + 5
        gmap = (1 + np.arange(n) % 9).astype(np.int32)
        for w, m in ((0, 255), (1, 256), (2, 257), (4, 512), (5, 513)):
            gmap[65536 * w + np.concatenate([[0, 65535], 1 + rng.choice(65534, m - 2, replace=False)])] = 0
        gmap[3 * 65536:4 * 65536][gmap[3 * 65536:4 * 65536] == 0] = 1
        return n, 10, gmap
    if case == "near":  # up to 1024 members in one to nine windows of the register path, some empty, ends on both sides
        n = 10 * 65536
        gmap = np.full(n, 7, dtype=np.int32)
        for c, lo, hi, m in ((0, 64, 64 + 8 * 65536 - 1, 1024), (1, 96, 96 + 8 * 65536, 1024), (2, 65535, 65536, 2),
                             (3, 65537, 3 * 65536, 700), (4, 40, 40 + 65535, 1023), (5, 41, 41 + 65536, 1023)):
            inner = np.setdiff1d(np.concatenate([lo + 1 + np.arange(640), hi - 1 - np.arange(640)]),
                                 np.flatnonzero(gmap != 7)) if hi - lo > 2000 else np.empty(0, dtype=np.int64)
            gmap[np.concatenate([[lo, hi], rng.permutation(inner)[:m - 2]])] = c
        gmap[200000] = 6
        return n, 8, gmap
    if case == "shared":  # six clusters beyond their buckets (8 n / k members) share the list
        n, k = 150000, 900
        gmap = rng.integers(0, 6, n).astype(np.int32) * 150
        gmap[:k] = np.arange(k)
        return n, k, gmap
    n = 513 * 65536 + 100  # "far": more windows than one partition takes
    gmap = np.zeros(n, dtype=np.int32)
    gmap[rng.integers(0, n, 3000)] = 1
    gmap[[0, n - 1]] = 2
    return n, 3, gmap


@pytest.mark.parametrize("case", ["dense", "runs", "near", "shared", "far"])
def test_update_centroids_windows(ctx, case):
    n, k, gmap = _windows_map(case)
    rng = np.random.default_rng(n)
    grid = rng.uniform(0, 7, size=(n, 3))
    rho = rng.uniform(0.1, 2.0, size=n)
    got, st = ctx.update_centroids(rho, grid, gmap, k)
    ref, crit = KO.update_centroids(rho, grid, gmap, k)
    assert st == L.THC_OK and crit == 0
    np.testing.assert_array_equal(got.cpu().numpy(), ref)


def test_kmeans_vacuum(ctx):
    """A density that falls off into vacuum: the centroids follow it and the few left outside own far more points
    than a bucket holds, more of them with every iteration."""
    rng = np.random.default_rng(4)
    n, k = 40000, 600
    grid = rng.uniform(0, 24, size=(n, 3))
    rho = np.exp(-1.0 * np.linalg.norm(grid - 12.0, axis=1))
    ref = KO.kmeans(grid, rho, k, 16, -1.0, 2, keep_maps=True)
    big = [(np.bincount(m, minlength=k) > 8 * -(-n // k)).sum() for m in ref["maps"]]
    assert ref["status"] == 0 and big[0] == 0 and big[-1] > 3
    for thr in (-1.0, 1e-300):
        out = ctx.kmeans(grid, rho, k, 16, thr, 2, want_map=True, want_centroids=True)
        np.testing.assert_array_equal(out["interp_idx"].cpu().numpy(), ref["interp_idx"])
        np.testing.assert_array_equal(out["diffs"], ref["diffs"])
        np.testing.assert_array_equal(out["grid_map"].cpu().numpy(), ref["maps"][-1])
        np.testing.assert_array_equal(out["centroids"].cpu().numpy(), ref["centroids"])


@pytest.mark.parametrize("n,k", [(1, 1), (255, 2), (1023, 4), (1024, 1024), (1025, 7), (5000, 4096)])
def test_update_centroids_tile_edges(ctx, n, k):
    """Point counts either side of the 1024-point tiles that fill the buckets, every key count; a key outside
    [0, k) in the first and last place of a tile is refused."""
    rng = np.random.default_rng(n + k)
    grid = rng.uniform(0, 7, size=(n, 3))
    rho = rng.uniform(0.1, 2.0, size=n)
    gmap = rng.permutation(np.arange(n) % k).astype(np.int32)
    got, st = ctx.update_centroids(rho, grid, gmap, k)
    ref, crit = KO.update_centroids(rho, grid, gmap, k)
    assert st == L.THC_OK and crit == 0
    np.testing.assert_array_equal(got.cpu().numpy(), ref)
    for at in sorted({0, min(n, 1024) - 1, n - 1}):
        for key in (-1, k, 2 ** 31 - 1):
            bad = gmap.copy()
            bad[at] = key
            assert ctx.update_centroids(rho, grid, bad, k)[1] == L.THC_ERR_ARG
