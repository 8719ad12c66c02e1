"""Cuts with as many parts as a compute unit's LDS holds weights of, and more."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def cut(gk, ctx, dg, k, part):
    c, pw = ctypes.c_int64(-1), np.full(k, -1, np.int64)
    from _dev import ptr
    rc = gk.lib().gk_k_cut(ctx.handle, dg.ref(), k, ptr(part), ctypes.byref(c),
                           pw.ctypes.data_as(ctypes.POINTER(ctypes.c_int64)), None)
    return rc, c.value, pw


@pytest.mark.parametrize("n", [3000, 150_000])
@pytest.mark.parametrize("k", [16376, 40929, 40952])
def test_accepted(gk, oracle, ctx, n, k):
    from _dev import DevGraph, dev
    g = gk.dag(n, 50, 2)
    part = np.random.default_rng(k).integers(0, k, n).astype(np.int32)
    exp, epw = oracle.cut(g, k, part)
    rc, got, pw = cut(gk, ctx, DevGraph(g), k, dev(part))
    assert rc == 0 and got == exp and np.array_equal(pw, epw)


@pytest.mark.parametrize("k", [40953, 50000, 2**20])
def test_refused(gk, ctx, k):
    from _dev import DevGraph, dev
    g = gk.dag(3000, 50, 2)
    rc, got, _ = cut(gk, ctx, DevGraph(g), k, dev(np.zeros(g.n, np.int32)))
    assert rc == -7 and got == -1
    assert b"40952" in gk.lib().gk_last_error()
