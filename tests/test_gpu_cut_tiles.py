"""The cut kernel around its tiles: one block of 256 vertices, the largest grid
with one vertex a group (131072) and beyond it, rows shorter and longer than
eight entries, few and many parts, with and without room for all blocks' slots."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n", [1, 255, 256, 257, 131071, 131072, 131073, 300001])
@pytest.mark.parametrize("k", [1, 17, 1025, 8192])
@pytest.mark.parametrize("long_rows", [False, True])
def test_cut(gk, oracle, ctx, n, k, long_rows):
    from _dev import DevGraph, dev, ptr
    rng = np.random.default_rng(n + k)
    # a ring, or a ring and spokes to three hubs
    a, b = np.arange(n), (np.arange(n) + 1) % n
    if long_rows:
        v = rng.integers(0, n, n // 2)
        a, b = np.concatenate([a, v]), np.concatenate([b, v % 3 * (n // 3)])
    keep = a != b
    key = np.unique(np.minimum(a, b)[keep] * n + np.maximum(a, b)[keep])
    a, b = key // n, key % n
    w = rng.integers(1, 1 << 20, len(a))
    s, d, w = np.concatenate([a, b]), np.concatenate([b, a]), np.concatenate([w, w])
    at = np.lexsort((d, s))
    g = gk.Graph(np.concatenate([[0], np.cumsum(np.bincount(s, minlength=n))]), d[at], w[at], rng.integers(1, 99, n))
    part = rng.integers(0, k, n).astype(np.int32)
    exp, epw = oracle.cut(g, k, part)
    dg, dp = DevGraph(g), dev(part)
    cut = ctypes.c_int64()
    pw = np.zeros(k, np.int64)
    L, vp = gk.lib(), ctypes.c_void_p
    assert L.gk_k_cut(ctx.handle, dg.ref(), k, ptr(dp), ctypes.byref(cut), pw.ctypes.data_as(ctypes.POINTER(ctypes.c_int64)), None) == 0
    assert cut.value == exp and np.array_equal(pw, epw)
    dcut = torch.full((1,), -1, dtype=torch.int64, device="cuda")
    dpw = torch.full((k,), -1, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    assert L.gk_k_cut_noalloc(ctx.handle, dg.ref(), k, ptr(dp), vp(dcut.data_ptr()), vp(dpw.data_ptr()), None) == 0
    torch.cuda.synchronize()
    assert int(dcut.item()) == exp and np.array_equal(dpw.cpu().numpy(), epw)
