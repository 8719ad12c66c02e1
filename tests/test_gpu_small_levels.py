"""Grouping of small graphs in one workgroup: vertex counts around its limit
(4096) and its threads (1024), trees too deep for it and groups too large,
chunk sizes from one vertex to all; alone and in a batch (which wants the
members' order as well).  Whole numbers: every comparison with the oracle is
exact, level by level."""
import numpy as np
import pytest

from test_gpu_coarse_ids import chain_graph, star_graph
from test_gpu_parity import compare

pytestmark = pytest.mark.gpu

pytest.importorskip("torch")


@pytest.mark.parametrize("n", [4, 5, 1023, 1024, 1025, 2049, 4095, 4096, 4097])
@pytest.mark.parametrize("family", ["delaunay", "dag", "road", "chain", "star"])
def test_sizes(gk, oracle, ctx, n, family):
    g = {"delaunay": lambda: gk.delaunay(n, 3), "dag": lambda: gk.dag(n, max(2, n // 40), 5),
         "road": lambda: gk.road(n, 2), "chain": lambda: chain_graph(gk, n), "star": lambda: star_graph(gk, n)}[family]()
    compare(gk, oracle, ctx, g, 2, coarsen_to=3)


@pytest.mark.parametrize("group", [1, 2, 6, 64])
def test_chunks(gk, oracle, ctx, group):
    compare(gk, oracle, ctx, gk.dag(4000, 60, 8), 4, coarsen_to=9, max_group=group)


def test_batch_of_one_tile(gk, oracle, ctx):
    sizes = [1300, 700, 1, 2000, 95]  # 4096 together
    graphs = [gk.delaunay(n, n) if n > 3 else gk.Graph([0, 0], []) for n in sizes]
    parts, stats = ctx.partition_batch(graphs, [4] * len(sizes), coarsen_to=20)
    for g, part in zip(graphs, parts):
        assert np.array_equal(part, oracle.partition(g, 4, coarsen_to=20)[0])
