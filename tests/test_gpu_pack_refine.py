"""The launches of a batched refinement step where they can go wrong: graphs
whose sizes lie around the kernels' tiles (2048 vertices of a pack, 512 of a
finished graph), many graphs inside one tile, and a single graph.  Whole
numbers: every partition and cut equals the oracle's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

pytest.importorskip("torch")


@pytest.mark.parametrize("sizes", [[2048], [2047, 1, 2049, 2], [511, 512, 513, 1537, 4096, 4097], [300] * 37 + [6000],
                                   [1023, 9001, 1025, 2, 3, 20481]])
@pytest.mark.parametrize("ks", [[2, 3, 7], [64, 256, 5], [300, 2]])
def test_sizes(gk, oracle, ctx, sizes, ks):
    graphs = [gk.delaunay(n, n + i) if n > 3 else gk.Graph([0] * (n + 1), []) for i, n in enumerate(sizes)]
    kk = [ks[i % len(ks)] for i in range(len(sizes))]
    print(f"batch n={sizes} k={kk}", flush=True)
    parts, stats = ctx.partition_batch(graphs, kk)
    for g, k, part, st in zip(graphs, kk, parts, stats):
        exp, est = oracle.partition(g, k)
        assert np.array_equal(part, exp)
        assert st.cut == est.cut == st.cut_tracked
        for l in range(est.nlevels):
            a, b = st.levels[l], est.levels[l]
            assert (a.n, a.nnz, a.rounds, a.moves, a.cut_after) == (b.n, b.nnz, b.rounds, b.moves, b.cut_after)
