"""The initial partitioner where it changes its method, against the oracle's
restatement of its rules: growing by a scan of the gains or from the heap,
coarse rows built by one thread or several, the last pass's vertices picked by
one thread or several, parts that start above the cap.  Whole numbers, so
exactly; on one thread and on the pool."""
import numpy as np
import pytest


def bipartite(gk, a, n, seed):
    """a vertices adjacent to all the others: matching stalls at a pairs, so
    the whole graph is grown."""
    rng = np.random.default_rng(seed)
    left, right = np.repeat(np.arange(a), n - a), np.tile(np.arange(a, n), a)
    w = rng.integers(1, 30, len(left))
    src, dst, ww = np.concatenate([left, right]), np.concatenate([right, left]), np.concatenate([w, w])
    at = np.lexsort((dst, src))
    xadj = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))])
    return gk.Graph(xadj, dst[at], ww[at], rng.integers(1, 6, n))


def check(gk, oracle, g, k, cap, seed=3):
    exp = oracle.initpart(g, k, cap, seed)
    for threads in (1, 8):
        part, cut = gk.initpart(g, k, cap, seed=seed, threads=threads)
        assert np.array_equal(part, exp[0]), threads
        assert cut == exp[1]


# around the scan's 256 vertices and four entries a row (a = 1: two a row)
@pytest.mark.parametrize("n", [8, 121, 249, 256, 257, 400])
@pytest.mark.parametrize("a", [1, 2, 5])
def test_growing(gk, oracle, n, a):
    g = bipartite(gk, a, n, n + a)
    for k in (2, 5):
        check(gk, oracle, g, k, gk.lib().gk_part_cap(int(g.vwgt.sum()), k, 30))


# rows around the sizes from which ranges are built and picked in parallel
@pytest.mark.parametrize("n", [1300, 2800, 11000, 25000])
def test_parallel_ranges(gk, oracle, n):
    g = gk.delaunay(n, n)
    check(gk, oracle, g, 8, gk.lib().gk_part_cap(g.n, 8, 30))


# no room above the average: parts start above the cap and are repaired
@pytest.mark.parametrize("k", [3, 16, 64])
@pytest.mark.parametrize("slack", [-2, 0, 1])
def test_tight_cap(gk, oracle, k, slack):
    for g in (gk.dag(4000, 60, k), gk.delaunay(3000, k)):
        check(gk, oracle, g, k, int(g.vwgt.sum()) // k + slack)
