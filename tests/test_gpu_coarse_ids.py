"""Grouping by walking and coarse ids by counting (gk_k_group, gk_k_cluster
and the coarsening levels) where they change their method: trees as deep as
the walk goes and deeper, groups as large as the ranking takes and larger,
tiles that end inside, and more tiles than a block sums by itself.  Whole
numbers: every comparison with the oracle is exact."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def gpu_cluster(gk, ctx, label, stamp, vw, G):
    from _dev import dev, host, ptr
    n = len(label)
    order, cmap, cvw = (torch.full((n,), -1, dtype=torch.int32, device="cuda") for _ in range(3))
    nc = ctypes.c_int32(0)
    assert gk.lib().gk_k_cluster(ctx.handle, n, ptr(dev(label)), ptr(dev(stamp)), ptr(dev(vw)), G, ptr(order), ptr(cmap),
                                 ptr(cvw), ctypes.cast(ctypes.pointer(nc), gk.I32P), None) == 0
    return host(order), host(cmap), host(cvw)[: nc.value], nc.value


# sizes of the groups, repeated to the vertex count; the ranking takes groups
# of up to 512, the counting kernels tiles of 2048 labels and blocks of 256
@pytest.mark.parametrize("n,sizes", [(1, [1]), (255, [1, 2, 3]), (2049, [6, 7, 5]), (5000, [512, 1]), (5000, [513, 1]),
                                     (4096, [511, 64, 2]), (20001, [20001]), (70000, [4000, 3, 1]), (33333, [1])])
@pytest.mark.parametrize("G", [1, 6, 2**31 - 1])
def test_cluster_sizes(gk, oracle, ctx, n, sizes, G):
    rng = np.random.default_rng(n + len(sizes))
    of = np.repeat(np.arange(n), np.resize(sizes, n))[:n]
    label = rng.permutation(n)[of][rng.permutation(n)].astype(np.int32)
    # few stamps (many ties, decided by the vertex id), and stamps of any size
    stamp = np.where(rng.random(n) < 0.5, rng.integers(0, 3, n), rng.integers(0, 2**31 - 1, n)).astype(np.int32)
    vw = rng.integers(1, 9, n).astype(np.int32)
    got = gpu_cluster(gk, ctx, label, stamp, vw, G)
    exp = oracle.cluster(label, stamp, vw, G)
    assert got[3] == exp[3]
    for a, b in zip(got[:3], exp[:3]):
        assert np.array_equal(a, b[: len(a)])


def test_cluster_many_tiles(gk, oracle, ctx):
    n = 8192 * 2048 + 777
    rng = np.random.default_rng(1)
    label = (rng.integers(0, n // 4, n) * 4 + 3).astype(np.int32)
    stamp = rng.integers(0, 4, n).astype(np.int32)
    vw = np.ones(n, np.int32)
    got = gpu_cluster(gk, ctx, label, stamp, vw, 6)
    exp = oracle.cluster(label, stamp, vw, 6)
    assert got[3] == exp[3]
    for a, b in zip(got[:3], exp[:3]):
        assert np.array_equal(a, b[: len(a)])


# chains of the given number of hops to a mutual pair, and one vertex alone;
# the walk goes 64 hops
@pytest.mark.parametrize("hops", [0, 1, 2, 3, 16, 17, 63, 64, 65, 66, 300])
def test_group_depth(gk, oracle, ctx, hops):
    from _dev import dev, host, ptr
    chains = 37
    per = hops + 2  # the pair and the vertices before it
    n = chains * per + 1
    name = np.random.default_rng(hops).permutation(n)
    cand = np.empty(n, np.int64)
    for c in range(chains):
        ids = name[c * per:(c + 1) * per]
        cand[ids[:-1]] = ids[1:]
        cand[ids[-1]] = ids[-2]
    cand[name[-1]] = name[-1]
    cand = cand.astype(np.int32)
    label, stamp = (torch.zeros(n, dtype=torch.int32, device="cuda") for _ in range(2))
    sweeps = ctypes.c_int32(-1)
    assert gk.lib().gk_k_group(ctx.handle, n, ptr(dev(cand)), ptr(label), ptr(stamp),
                               ctypes.cast(ctypes.pointer(sweeps), gk.I32P), None) == 0
    olabel, ostamp, osweeps = oracle.group(cand)
    assert np.array_equal(host(label), olabel)
    assert np.array_equal(host(stamp), ostamp)
    assert sweeps.value == osweeps


def chain_graph(gk, n):
    """A path whose weights rise along it: every vertex's candidate is the
    next one, so the whole path is one group, n - 2 hops deep."""
    ends = np.arange(n - 1)
    src = np.concatenate([ends, ends + 1])
    dst = np.concatenate([ends + 1, ends])
    w = np.concatenate([ends + 1, ends + 1])
    at = np.lexsort((dst, src))
    xadj = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))])
    return gk.Graph(xadj, dst[at], w[at])


def star_graph(gk, n):
    """One hub adjacent to every other vertex, and a ring among those."""
    v = np.arange(1, n)
    a = np.concatenate([np.zeros(n - 1, np.int64), v])
    b = np.concatenate([v, np.where(v == n - 1, 1, v + 1)])
    w = np.concatenate([np.full(n - 1, 5), np.ones(n - 1, np.int64)])
    src, dst, ww = np.concatenate([a, b]), np.concatenate([b, a]), np.concatenate([w, w])
    at = np.lexsort((dst, src))
    xadj = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))])
    return gk.Graph(xadj, dst[at], ww[at])


@pytest.mark.parametrize("make,n", [(chain_graph, 3001), (star_graph, 3001)])
def test_vcycle_deep_and_large_groups(gk, oracle, ctx, make, n):
    from test_gpu_parity import compare
    compare(gk, oracle, ctx, make(gk, n), 4)


def test_batch_deep_and_large_groups(gk, ctx):
    """The same inside a batch, beside a graph that needs neither."""
    graphs = [chain_graph(gk, 3001), gk.delaunay(3000, 2), star_graph(gk, 2777), chain_graph(gk, 700)]
    ks = [4, 8, 2, 2]
    parts, _ = ctx.partition_batch(graphs, ks)
    for g, k, p in zip(graphs, ks, parts):
        assert np.array_equal(p, ctx.partition(g, k)[0])
