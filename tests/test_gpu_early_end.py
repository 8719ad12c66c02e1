"""Stage calls that end early leave nothing queued: when the call returns its
stream has run out, so the next call, on another stream, may use the memory
again and the caller may free the arguments."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def stage_buffers(n, nnz):
    return {name: torch.full((size,), -1, dtype=torch.int32, device="cuda")
            for name, size in (("cxadj", n + 1), ("cadj", nnz), ("cw", nnz))}


def contract(gk, ctx, dg, cmap, nc, out, stream):
    from _dev import ptr
    r = ctypes.c_int32(-1)
    rc = gk.lib().gk_k_contract(ctx.handle, dg.ref(), ptr(cmap), nc, ptr(out["cxadj"]), ptr(out["cadj"]), ptr(out["cw"]),
                                ctypes.cast(ctypes.pointer(r), gk.I32P), ctypes.c_void_p(stream.cuda_stream))
    return rc, r.value


@pytest.mark.parametrize("n", [5000, 1_000_000])
def test_refused_contraction(gk, oracle, n):
    """A coarse map that leaves an id out, and at once a right one on another stream."""
    from _dev import DevGraph, dev, host
    g = gk.delaunay_hilbert(n, 7)
    label, stamp, _ = oracle.group(oracle.match(g))
    _, cmap, _, nc = oracle.cluster(label, stamp, g.vwgt, 6)
    ex, ea, ew = oracle.contract(g, cmap, nc)
    dg = DevGraph(g)
    good, gap = dev(cmap), dev(cmap + (cmap >= nc // 2))
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with gk.Context(0) as ctx:
        for rep in range(3):
            bad, out = stage_buffers(n, g.nnz), stage_buffers(n, g.nnz)
            torch.cuda.synchronize()
            rc, _ = contract(gk, ctx, dg, gap, nc + 1, bad, first)
            idle = first.query()
            rc2, cnnz = contract(gk, ctx, dg, good, nc, out, second)
            assert rc == -1 and idle
            assert rc2 == 0 and cnnz == len(ea)
            assert np.array_equal(host(out["cxadj"])[:nc + 1], ex)
            assert np.array_equal(host(out["cadj"])[:cnnz], ea) and np.array_equal(host(out["cw"])[:cnnz], ew)


@pytest.mark.parametrize("n", [5000, 300_000])
def test_no_room(gk, oracle, n):
    """Pool limits from ample down to none: every failure finds the stream idle."""
    from _dev import DevGraph, dev, ptr
    g = gk.delaunay_hilbert(n, 8)
    cand = oracle.match(g)
    label, stamp, _ = oracle.group(cand)
    _, cmap, _, nc = oracle.cluster(label, stamp, g.vwgt, 6)
    L, dg, out = gk.lib(), DevGraph(g), stage_buffers(n, g.nnz)
    dc, dl, ds, dw, dm = dev(cand), dev(label), dev(stamp), dev(g.vwgt), dev(cmap)
    a, b, c = (torch.full((n,), -1, dtype=torch.int32, device="cuda") for _ in range(3))
    part = torch.zeros(n, dtype=torch.int32, device="cuda")
    stream = torch.cuda.Stream()
    st = ctypes.c_void_p(stream.cuda_stream)
    r, cut = ctypes.c_int32(), ctypes.c_int64()
    ri = ctypes.cast(ctypes.pointer(r), gk.I32P)
    calls = {
        "group": lambda h: L.gk_k_group(h, n, ptr(dc), ptr(a), ptr(b), ri, st),
        "cluster": lambda h: L.gk_k_cluster(h, n, ptr(dl), ptr(ds), ptr(dw), 6, ptr(a), ptr(b), ptr(c), ri, st),
        "contract": lambda h: L.gk_k_contract(h, dg.ref(), ptr(dm), nc, ptr(out["cxadj"]), ptr(out["cadj"]), ptr(out["cw"]), ri, st),
        "cut": lambda h: L.gk_k_cut(h, dg.ref(), 64, ptr(part), ctypes.byref(cut), None, st),
    }
    torch.cuda.synchronize()
    for name, call in calls.items():
        failed = 0
        with gk.Context(0) as ctx:
            for per in (160, 96, 64, 56, 48, 40, 32, 24, 16, 12, 8, 4, 1):
                L.gk_ctx_set_pool_limit(ctx.handle, per * n)
                rc = call(ctx.handle)
                assert stream.query(), (name, per)
                assert rc in (0, -6), (name, per, L.gk_last_error())
                failed += rc != 0
        print(f"{name} n={n} failed={failed}", flush=True)
        assert failed > 0 or name == "cut"
