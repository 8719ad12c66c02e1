"""Grouping and clustering with results in the place of their inputs, in trees
the walk resolves and deeper ones, and groups that are ranked and sorted."""
import ctypes

import numpy as np
import pytest

from test_gpu_coarse_ids import chain_graph, star_graph

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("make", [lambda gk: gk.delaunay(5000, 2), lambda gk: chain_graph(gk, 900),
                                  lambda gk: star_graph(gk, 900)], ids=["mesh", "chain", "star"])
def test_in_place(gk, oracle, ctx, make):
    from _dev import dev, host, ptr
    g = make(gk)
    cand = oracle.match(g)
    label, stamp, sweeps = oracle.group(cand)
    L = gk.lib()
    for where in ("label", "stamp"):
        d = dev(cand)
        other = torch.full_like(d, -1)
        r = ctypes.c_int32()
        a, b = (d, other) if where == "label" else (other, d)
        assert L.gk_k_group(ctx.handle, g.n, ptr(d), ptr(a), ptr(b), ctypes.cast(ctypes.pointer(r), gk.I32P), None) == 0
        assert np.array_equal(host(a), label) and np.array_equal(host(b), stamp) and r.value == sweeps
    order, cmap, cvw, nc = oracle.cluster(label, stamp, g.vwgt, 6)
    dl, ds, dw = dev(label), dev(stamp), dev(g.vwgt)
    r = ctypes.c_int32()
    assert L.gk_k_cluster(ctx.handle, g.n, ptr(dl), ptr(ds), ptr(dw), 6, ptr(ds), ptr(dl), ptr(dw),
                          ctypes.cast(ctypes.pointer(r), gk.I32P), None) == 0
    assert r.value == nc
    assert np.array_equal(host(ds), order) and np.array_equal(host(dl), cmap) and np.array_equal(host(dw)[:nc], cvw[:nc])
