"""Matching with the neighbours' degrees as bytes (graphs of 2^20 vertices and
more): vertex counts around the line and off the table's multiples of four, and
hubs whose degrees decide between equal weights where a byte ends."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

DEGREES = [253, 254, 255, 256, 257, 255, 300, 254, 600, 256]


@pytest.mark.parametrize("n", [2**20 - 1, 2**20, 2**20 + 1, 2**20 + 2, 2**20 + 3])
def test_hub_degrees(gk, oracle, ctx, n):
    from _dev import DevGraph, host, ptr
    rng = np.random.default_rng(n)
    hubs = rng.choice(n, len(DEGREES), replace=False)
    rest = np.setdiff1d(np.arange(n), hubs)
    # hub edges of one weight, to vertices that mostly have two of them; a
    # lighter ring through the other vertices
    ends = np.repeat(np.arange(len(DEGREES)), np.array(DEGREES))
    leaves = rest[: len(ends) // 2 + 1]
    a, b = [], []
    for i, d in enumerate(DEGREES):
        a.append(np.full(d, hubs[i]))
        b.append(rng.choice(leaves, d, replace=False))
    a, b = np.concatenate(a + [rest]), np.concatenate(b + [np.roll(rest, 1)])
    w = np.where(np.arange(len(a)) < len(ends), 5, 1)
    s, d, w = np.concatenate([a, b]), np.concatenate([b, a]), np.concatenate([w, w])
    at = np.lexsort((d, s))
    g = gk.Graph(np.concatenate([[0], np.cumsum(np.bincount(s, minlength=n))]), d[at], w[at], np.ones(n, np.int64))
    dg = DevGraph(g)
    cand = torch.full((n,), -1, dtype=torch.int32, device="cuda")
    print(f"match n={n} nnz={g.nnz}", flush=True)
    assert gk.lib().gk_k_match(ctx.handle, dg.ref(), ptr(cand), None) == 0
    assert np.array_equal(host(cand), oracle.match(g))
