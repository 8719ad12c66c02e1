"""Contraction where it changes its method: coarse rows with as many entries
as a class takes and one more (lanes, a workgroup, the global sort), distinct
neighbours and repeated ones, coarse graphs up to the size whose lane classes
go in one launch and larger.  Whole numbers: every comparison with the oracle
is exact."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

EDGES = [0, 1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 1023, 1024, 1025, 2047, 2048, 2049, 5000]


def rows_graph(gk, entries, others, targets, seed):
    """A bipartite graph: one hub group per number of entries, made of up to
    seven members, whose entries go to vertices of `targets` coarse ids drawn
    with repetition (an entry per edge); `others` vertices on their own."""
    rng = np.random.default_rng(seed)
    src, dst, cmap = [], [], []
    nv = 0
    pool0 = nv
    npool = max(max(entries), 1)
    cmap += list(rng.integers(0, targets, npool))
    nv += npool
    c = targets
    for e in entries:
        members = int(rng.integers(1, 8))
        own = rng.integers(0, members, e)
        src.append(nv + own)
        dst.append(pool0 + rng.permutation(npool)[:e])
        cmap += [c] * members
        nv += members
        c += 1
    cmap += list(range(c, c + others))
    nv += others
    cmap = np.array(cmap, np.int64)
    # onto: ids without members are closed up
    _, cmap = np.unique(cmap, return_inverse=True)
    s, d = np.concatenate(src), np.concatenate(dst)
    w = rng.integers(1, 50, len(s))
    s, d, w = np.concatenate([s, d]), np.concatenate([d, s]), np.concatenate([w, w])
    at = np.lexsort((d, s))
    xadj = np.concatenate([[0], np.cumsum(np.bincount(s, minlength=nv))])
    return gk.Graph(xadj, d[at], w[at], np.ones(nv, np.int64)), cmap.astype(np.int32)


@pytest.mark.parametrize("others", [0, 1, 2**16 - 2869 + 1, 2**16 - 2869 + 2, 70001])
@pytest.mark.parametrize("targets", [1, 3, 4000])
def test_contract_class_edges(gk, oracle, ctx, others, targets):
    from _dev import DevGraph, dev, host, ptr
    g, cmap = rows_graph(gk, EDGES, others, targets, others + targets)
    nc = int(cmap.max()) + 1
    dg = DevGraph(g)
    cx, ca, cw = (torch.zeros(x, dtype=torch.int32, device="cuda") for x in (nc + 1, g.nnz, g.nnz))
    cnnz = ctypes.c_int32(0)
    print(f"contract n={g.n} nnz={g.nnz} nc={nc}", flush=True)
    assert gk.lib().gk_k_contract(ctx.handle, dg.ref(), ptr(dev(cmap)), nc, ptr(cx), ptr(ca), ptr(cw),
                                  ctypes.cast(ctypes.pointer(cnnz), gk.I32P), None) == 0
    ox, oa, ow = oracle.contract(g, cmap, nc)
    assert cnnz.value == len(oa)
    assert np.array_equal(host(cx), ox)
    assert np.array_equal(host(ca)[: len(oa)], oa)
    assert np.array_equal(host(cw)[: len(ow)], ow)
