"""Transfers on both sides of what the pinned staging memory takes (16 MiB): a
coarsest graph, its initial partition, a round history.  Same results, and no
context is left with a staging area as large as its largest graph."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

STAGE = 16 << 20


def device_mappings():
    """Sizes of the mappings through which this process sees pinned and device memory."""
    out = {}
    with open("/proc/self/maps") as f:
        for line in f:
            if "/dev/dri/" in line or "/dev/kfd" in line:
                a, b = (int(x, 16) for x in line.split()[0].split("-"))
                out[a] = b - a
    return out


def partition(gk, ctx, dg, k, **kw):
    from _dev import host, ptr
    part = torch.full((dg.g.n,), -1, dtype=torch.int32, device="cuda")
    p, st = gk.params(k, **kw), gk.Stats()
    torch.cuda.synchronize()
    rc = gk.lib().gk_partition_device(ctx.handle, dg.ref(), ctypes.byref(p), ptr(part), ctypes.byref(st), None)
    assert rc == 0, gk.lib().gk_last_error().decode()
    return host(part), st


# n around which 4 bytes a word of the coarsest graph (here the graph itself)
# and, in the last case, of the initial partition, pass the limit
@pytest.mark.parametrize("n,edges", [(280_000, "mesh"), (320_000, "mesh"), (450_000, "mesh"), (5_000_000, "ring")])
def test_no_coarsening(gk, oracle, n, edges):
    from _dev import DevGraph
    if edges == "mesh":
        g = gk.delaunay_hilbert(n, 3)
    else:
        v = np.arange(n)
        a = np.sort(np.stack([(v - 1) % n, (v + 1) % n], 1), 1)
        g = gk.Graph(np.arange(0, 2 * n + 1, 2), a.reshape(-1), np.ones(2 * n), np.ones(n))
    dg = DevGraph(g)
    words = 2 * g.n + 2 * g.nnz
    with gk.Context(0) as ctx:
        before = device_mappings()
        part, st = partition(gk, ctx, dg, 2, max_levels=1)
        new = [size for at, size in device_mappings().items() if before.get(at) != size]
        print(f"n={n} coarsest graph {4 * words >> 20} MiB, largest new mapping {max(new, default=0) >> 20} MiB", flush=True)
        # the context's largest device array is its copy of the partition
        assert max(new, default=0) < max(STAGE + (1 << 20), 4 * n + (4 << 20))
        again, _ = partition(gk, ctx, dg, 2, max_levels=1)
    assert np.array_equal(part, again) and st.cut == st.cut_tracked
    if n <= 320_000:
        expect, _ = oracle.partition(g, 2, max_levels=1)
        assert np.array_equal(part, expect)


def test_large_coarse_graph(gk):
    """One level of coarsening that leaves more than the limit: as the batched form."""
    from _dev import DevGraph
    g = gk.delaunay_hilbert(1_600_000, 4)
    with gk.Context(0) as ctx:
        part, st = partition(gk, ctx, DevGraph(g), 2, max_levels=2)
        print(f"coarse n={st.levels[1].n} nnz={st.levels[1].nnz}", flush=True)
        assert st.nlevels == 2 and 8 * (st.levels[1].n + st.levels[1].nnz) > STAGE
        parts, _ = ctx.partition_batch([g], [2], max_levels=2)
    assert np.array_equal(part, parts[0])


@pytest.mark.parametrize("R", [(1 << 21) - 5, (1 << 21) + 5])
def test_long_history(gk, ctx, R):
    from test_gpu_round import compare_rounds, gpu_rounds, state
    g = gk.delaunay_hilbert(2000, 2)
    start = state(gk, g, 4, seed=2, gain_bits=6, flip=0.01)
    cap = int(gk.lib().gk_part_cap(int(g.vwgt.sum()), 4, 30))
    few = gpu_rounds(gk, ctx, g, 4, cap, 64, 200, *start)
    many = gpu_rounds(gk, ctx, g, 4, cap, 64, R, *start)
    assert few["nmoves"][-1] == 0
    assert not any(many["nmoves"][200:]) and all(p == -1 for p in many["pos"][200:])
    many["nmoves"], many["pos"] = many["nmoves"][:200], many["pos"][:200]
    compare_rounds(many, few, 64)
