"""Fused levels that run ahead of the host: batches of levels that end in the
middle, queues that outgrow their grid, levels that are slow enough to leave
the fused mode, level limits, and records of every level."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FUSED = "Push-Queue-WM-Fused"


def path(gsw, n):
    return gsw.from_edges(n, np.arange(n - 1), np.arange(1, n))


def tree(gsw, fan, depth):
    """Every vertex of a level has `fan` children: the queue grows fan-fold."""
    src, dst, lo, cnt = [], [], 0, 1
    for _ in range(depth):
        kids = lo + cnt + np.arange(cnt * fan)
        src.append(np.repeat(np.arange(lo, lo + cnt), fan))
        dst.append(kids)
        lo, cnt = lo + cnt, cnt * fan
    return gsw.from_edges(lo + cnt, np.concatenate(src), np.concatenate(dst))


def check_records(g, ref, levels):
    recs = g.records()
    assert len(recs) == levels
    for i, r in enumerate(recs):
        assert r["level"] == i + 1
        if r["fmt"] == "Queue" and r["dir"] == "Push":
            assert r["frontier"] == int((ref == i).sum())
            assert r["verts"] == r["frontier"] or r["lb"] == "STRICT"


@pytest.mark.parametrize("n", [2, 3, 9, 10, 17, 18, 200])
@pytest.mark.parametrize("configs", [None, FUSED])
def test_bfs_batches_end_anywhere(gsw, orc, n, configs):
    h = path(gsw, n)
    g = gsw.Graph(h)
    for root in (0, n // 2):
        for _ in range(2):
            ref = orc.bfs(h.row_ptr, h.col, root)
            assert np.array_equal(g.bfs(root, configs=configs), ref)
            if configs:
                check_records(g, ref, int(ref.max()) + 1)
    g.close()


@pytest.mark.parametrize("fan,depth", [(2, 14), (9, 5), (120, 2), (1000, 2)])
@pytest.mark.parametrize("configs", [None, FUSED])
def test_bfs_queue_outgrows_its_grid(gsw, orc, fan, depth, configs):
    h = tree(gsw, fan, depth)
    g = gsw.Graph(h)
    for root in (0, h.n - 1):
        ref = orc.bfs(h.row_ptr, h.col, root)
        assert np.array_equal(g.bfs(root, configs=configs), ref)
        if configs:
            check_records(g, ref, int(ref.max()) + 1)
    g.close()


@pytest.mark.parametrize("fan,depth", [(20, 3), (24, 3), (64, 2), (64, 3)])
def test_steep_growth_level_by_level(gsw, orc, fan, depth):
    """Growth above the limit of a batch: one level per batch, with or without
    leaving the fused mode after it."""
    h = tree(gsw, fan, depth)
    src = np.repeat(np.arange(h.n), np.diff(h.row_ptr))
    up = src < h.col
    w = np.random.default_rng(fan).integers(1, 65, int(up.sum())).astype(np.uint32)
    hw = gsw.from_edges(h.n, src[up], h.col[up], w)
    g = gsw.Graph(hw)
    for root in (0, 1, h.n - 1):
        for _ in range(2):
            assert np.array_equal(g.bfs(root), orc.bfs(h.row_ptr, h.col, root))
            assert np.array_equal(g.sssp(root), orc.spfa(hw.row_ptr, hw.col, hw.w, root))
    roots = [0, h.n // 2, h.n - 1]
    far = np.iinfo(np.int32).max
    each = [orc.bfs(h.row_ptr, h.col, r) for r in roots]
    want = np.min([np.where(x < 0, far, x) for x in each], axis=0)
    assert np.array_equal(g.bfs_multi(roots), want)
    g.close()


@pytest.mark.parametrize("limit", [1, 2, 5, 9, 10, 30])
def test_bfs_level_limit(gsw, orc, limit):
    h = path(gsw, 60)
    g = gsw.Graph(h)
    lv = g.bfs(0, configs=FUSED, max_levels=limit)
    ref = orc.bfs(h.row_ptr, h.col, 0)
    assert np.array_equal(lv, np.where(ref <= limit, ref, -1))
    assert g.last_stats.levels == limit
    assert np.array_equal(g.bfs(0, configs=FUSED), ref)
    g.close()


def test_bfs_leaves_the_fused_mode(gsw, orc):
    """A random graph whose levels grow sixfold: fused while they are small."""
    h = gsw.erdos_renyi(400000, 6.0, 5)
    g = gsw.Graph(h)
    for root in (0, 77, 399999):
        ref = orc.bfs(h.row_ptr, h.col, root)
        assert np.array_equal(g.bfs(root), ref)
        assert sum(r["verts"] for r in g.records() if r["fused"]) <= h.n
    g.close()


@pytest.mark.parametrize("configs", [None, FUSED])
@pytest.mark.parametrize("spec", ["path", "tree", "grid", "rmat"])
def test_sssp_and_bc_deduplicate_per_level(gsw, orc, spec, configs):
    """Vertices pushed again by later levels: both marking bitmaps are clean
    where a level needs them."""
    rng = np.random.default_rng(8)
    h = {"path": lambda: path(gsw, 300), "tree": lambda: tree(gsw, 7, 4),
         "grid": lambda: gsw.grid2d(70, 60, 0.1, 0.01, 3),
         "rmat": lambda: gsw.rmat(11, 8, seed=3)}[spec]()
    src = np.repeat(np.arange(h.n), np.diff(h.row_ptr))
    up = src < h.col
    hw = gsw.from_edges(h.n, src[up], h.col[up],
                        rng.integers(1, 65, int(up.sum())).astype(np.uint32))
    g = gsw.Graph(hw)
    for root in (0, h.n - 1):
        for _ in range(2):
            d = g.sssp(root, configs=configs)
            assert np.array_equal(d, orc.spfa(hw.row_ptr, hw.col, hw.w, root))
    g.close()
    g = gsw.Graph(h)
    for root in (0, h.n // 3):
        lv, nsp, dep = g.bc(root)
        elv, ensp, edep = orc.bc(h.row_ptr, h.col, root)
        assert np.array_equal(lv, elv)
        assert np.allclose(nsp, ensp, rtol=1e-12, atol=0)
        # 64-bit sums of the same terms in another order
        dep[root] = edep[root] = 0  # (the root is not between any pair)
        assert np.allclose(dep, edep, rtol=1e-10, atol=1e-12)
    g.close()


@pytest.mark.parametrize("iters", [0, 1, 2, 3, 9, 20])
def test_pagerank_iterations_bound_fused_levels(gsw, iters):
    """Fused PageRank levels keep every vertex queued, so only the iteration
    count ends them."""
    h = gsw.rmat(10, 8, seed=4)
    g = gsw.Graph(h)
    g.pagerank(0.85, iters, configs=FUSED)
    assert g.last_stats.levels == iters
    recs = g.records()
    assert [r["level"] for r in recs] == list(range(1, iters + 1))
    assert all(r["edges"] == h.m for r in recs)
    g.close()
