"""The apply of a round that moves many vertices, where its table of first
occurrences changes: movers and neighbours (items) of one less, as many and
one more than the round kernel's table takes (8192), the round loop's (4096)
and a few movers' (512), with neighbours shared by movers and without."""
import numpy as np
import pytest

from test_gpu_round import compare_rounds, gpu_rounds, oracle_rounds

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def stars(gk, movers, items, ring, shared):
    """`movers` centres (the smallest ids) in part 0 and leaves in part 1, so
    that centres and neighbours are `items`; with ring the leaves hold each
    other (only the centres gain by moving); with shared the centres' rows
    overlap by half."""
    deg = np.full(movers, items // movers - 1)
    deg[: items - movers - deg.sum()] += 1
    start = np.concatenate([[0], np.cumsum(deg)])[:-1]
    if shared:
        start = start // 2
    leaves = int((start + deg).max())
    a = np.repeat(np.arange(movers), deg)
    b = movers + np.concatenate([np.arange(s, s + d) for s, d in zip(start, deg)])
    w = np.full(len(a), 3)
    if ring:
        v = movers + np.arange(leaves)
        a, b, w = np.concatenate([a, v]), np.concatenate([b, movers + (np.arange(leaves) + 1) % leaves]), \
            np.concatenate([w, np.full(leaves, 50)])
    s, d, w = np.concatenate([a, b]), np.concatenate([b, a]), np.concatenate([w, w])
    at = np.lexsort((d, s))
    n = movers + leaves
    g = gk.Graph(np.concatenate([[0], np.cumsum(np.bincount(s, minlength=n))]), d[at], w[at], np.ones(n, np.int64))
    return g, np.r_[np.zeros(movers, np.int32), np.ones(leaves, np.int32)]


@pytest.mark.parametrize("movers,items,ring", [(m, i + x, r) for m, i, r in [(1024, 8192, False), (512, 4096, True),
                                                                            (1024, 8192, True), (40, 512, True),
                                                                            (20, 4096, True), (20, 4096, False)]
                                               for x in (-1, 0, 1)])
@pytest.mark.parametrize("shared", [False, True])
def test_items(gk, oracle, ctx, movers, items, ring, shared):
    g, part = stars(gk, movers, items, ring, shared)
    bnd, gain, dest = oracle.gain(g, 2, part, np.ones(g.n, np.int32))
    pw = np.bincount(part, minlength=2).astype(np.int32)
    cap = 2 * g.n
    exp = oracle_rounds(oracle, g, 2, cap, 1024, 3, part, bnd, gain, dest, pw)
    got = gpu_rounds(gk, ctx, g, 2, cap, 1024, 3, part, bnd, gain, dest, pw)
    print(f"n={g.n} candidates={int((gain > 0).sum())} nmoves={got['nmoves']} pos={got['pos']}", flush=True)
    compare_rounds(got, exp, 1024)
