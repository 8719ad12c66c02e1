"""Pool limits that leave no room for the members' records or for coarse rows
of the fine level's size: clustering goes by the sort, rows are copied once
their number is known, and results are those without a limit.  A call either
gives them or reports that there is no room."""
import ctypes

import numpy as np
import pytest

from test_gpu_coarse_ids import star_graph

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n", [4097, 50000, 300000])
def test_cluster(gk, oracle, n):
    from _dev import dev, host, ptr
    g = gk.delaunay(n, 3)
    label, stamp, _ = oracle.group(oracle.match(g))
    order, cmap, cvw, nc = oracle.cluster(label, stamp, g.vwgt, 6)
    done = []
    with gk.Context(0) as ctx:
        # By the sort 8 (results) + 32 bytes a vertex and its counters; with
        # the records 8 + 16 + 32 and theirs.
        for per in (42, 48, 54, 64):
            gk.lib().gk_ctx_set_pool_limit(ctx.handle, per * n + (1 << 17))
            o, c, w = (torch.full((n,), -1, dtype=torch.int32, device="cuda") for _ in range(3))
            r = ctypes.c_int32(-1)
            dl, ds, dw = dev(label), dev(stamp), dev(g.vwgt)
            rc = gk.lib().gk_k_cluster(ctx.handle, n, ptr(dl), ptr(ds), ptr(dw), 6, ptr(o), ptr(c), ptr(w),
                                       ctypes.cast(ctypes.pointer(r), gk.I32P), None)
            print(f"n={n} bytes/vertex={per} rc={rc}", flush=True)
            done.append(rc == 0)
            if rc == 0:
                assert r.value == nc
                assert np.array_equal(host(o), order) and np.array_equal(host(c), cmap)
                assert np.array_equal(host(w)[:nc], cvw[:nc])
    assert all(done)


@pytest.mark.parametrize("make", [lambda gk: gk.delaunay(6000, 2), lambda gk: gk.delaunay(120000, 4),
                                  lambda gk: star_graph(gk, 9000)], ids=["small", "mesh", "star"])
def test_partition(gk, oracle, make):
    g = make(gk)
    expect, _ = oracle.partition(g, 8)
    done = []
    for step in range(24):
        limit = int((16 << 20) * 0.8 ** step) + 4 * (g.n + g.nnz)
        with gk.Context(0) as ctx:
            gk.lib().gk_ctx_set_pool_limit(ctx.handle, limit)
            try:
                part, _ = ctx.partition(g, 8)
            except RuntimeError as e:
                assert "pool limit" in str(e)
                done.append(False)
                continue
            done.append(True)
            assert np.array_equal(part, expect), limit
    print(f"n={g.n} succeeded={sum(done)}", flush=True)
    assert done[0] and not done[-1]
    assert done == sorted(done, reverse=True)
