"""Labels and coarse ids that a caller gets wrong: outside [0, n), just beyond
it, far beyond it and negative, in one place, in many and in all.  Such calls
are refused, and a right call after them gives its result."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def wrong(values, n, how, where):
    v = values.copy()
    at = {"first": slice(0, 1), "last": slice(n - 1, n), "many": slice(0, n, 3), "all": slice(None)}[where]
    v[at] = {"n": n, "far": 2**31 - 1, "negative": -1, "lowest": -2**31}[how]
    return v


@pytest.mark.parametrize("n", [63, 1000, 1024, 70001])
@pytest.mark.parametrize("how", ["n", "far", "negative", "lowest"])
@pytest.mark.parametrize("where", ["first", "last", "many", "all"])
def test_refused(gk, oracle, ctx, n, how, where):
    from _dev import DevGraph, dev, host, ptr
    g = gk.delaunay(n, 5)
    label, stamp, _ = oracle.group(oracle.match(g))
    order, cmap, cvw, nc = oracle.cluster(label, stamp, g.vwgt, 6)
    ex, ea, ew = oracle.contract(g, cmap, nc)
    L, dg, ds, dw = gk.lib(), DevGraph(g), dev(stamp), dev(g.vwgt)
    o, c, w, cx = (torch.full((n + 1,), -1, dtype=torch.int32, device="cuda") for _ in range(4))
    ca, cw = (torch.full((g.nnz,), -1, dtype=torch.int32, device="cuda") for _ in range(2))
    r = ctypes.c_int32(-7)
    ri = ctypes.cast(ctypes.pointer(r), gk.I32P)

    def cluster(lab):
        d = dev(lab)
        torch.cuda.synchronize()
        return L.gk_k_cluster(ctx.handle, n, ptr(d), ptr(ds), ptr(dw), 6, ptr(o), ptr(c), ptr(w), ri, None)

    def contract(cm, ncoarse):
        d = dev(cm)
        torch.cuda.synchronize()
        return L.gk_k_contract(ctx.handle, dg.ref(), ptr(d), ncoarse, ptr(cx), ptr(ca), ptr(cw), ri, None)

    assert cluster(wrong(label, n, how, where)) == -1
    bad = wrong(cmap, n, how, where)
    # every number of coarse vertices that such a map could be taken for
    inside = bad[(bad >= 0) & (bad < n)]
    for ncoarse in {nc, len(np.unique(inside)), len(np.unique(bad))}:
        assert contract(bad, ncoarse) == -1, ncoarse
    assert r.value == -7
    assert cluster(label) == 0 and r.value == nc
    assert np.array_equal(host(o)[:n], order) and np.array_equal(host(c)[:n], cmap) and np.array_equal(host(w)[:nc], cvw)
    assert contract(cmap, nc) == 0 and r.value == len(ea)
    assert np.array_equal(host(cx)[:nc + 1], ex)
    assert np.array_equal(host(ca)[:len(ea)], ea) and np.array_equal(host(cw)[:len(ea)], ew)
