"""The launches that begin a level and carry the V-cycle's small copies: vertex
counts around their tiles, coarsest graphs that are the whole graph, numbers of
parts up to the largest, and a result buffer that is aligned to its type only.
Whole numbers: every comparison with the oracle is exact."""
import ctypes

import numpy as np
import pytest

from test_gpu_parity import compare

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1023, 1024, 1025, 4096, 4097, 20481])
@pytest.mark.parametrize("k", [1, 2, 257])
def test_vertex_counts(gk, oracle, ctx, n, k):
    g = gk.delaunay(n, n) if n > 3 else gk.Graph([0] * (n + 1), [])
    compare(gk, oracle, ctx, g, k)


def test_most_parts(gk, oracle, ctx):
    compare(gk, oracle, ctx, gk.delaunay(30000, 5), 8192)


def test_result_alignment(gk, oracle, ctx):
    from _dev import DevGraph, host, ptr
    g = gk.delaunay(10001, 3)
    dg = DevGraph(g)
    room = torch.full((g.n + 8,), -7, dtype=torch.int32, device="cuda")
    prm = gk.Params()
    gk.lib().gk_params_default(ctypes.byref(prm), 16)
    assert gk.lib().gk_partition_device(ctx.handle, dg.ref(), ctypes.byref(prm), ptr(room[1:]), None, None) == 0
    got = host(room)
    part, _ = oracle.partition(g, 16)
    assert np.array_equal(got[1 : g.n + 1], part)
    assert (got[0], set(got[g.n + 1 :])) == (-7, {-7})
