"""The round loop (many refinement rounds in one launch, one workgroup per
job) where it changes its method: jobs around the size of the movable bitmap,
candidate lists around their capacity and beyond it, rounds that move or
update more than one workgroup takes, rows longer than the lanes that share
them, the smallest and largest part counts.  Round by round against the
oracle's select / balance / apply / gain; whole numbers, so exactly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from test_gpu_round import compare_rounds, gpu_rounds, oracle_rounds, state  # noqa: E402
from test_gpu_stages import hub_graph  # noqa: E402


def check(gk, oracle, ctx, g, k, M, R, gbits, slack, flip, seed=5):
    part, bnd, gain, dest, pw = state(gk, g, k, seed=seed, gain_bits=gbits, flip=flip)
    cap = int(gk.lib().gk_part_cap(int(g.vwgt.sum()), k, 30)) if slack is None else int(pw.max()) + slack
    exp = oracle_rounds(oracle, g, k, cap, M, R, part, bnd, gain, dest, pw)
    got = gpu_rounds(gk, ctx, g, k, cap, M, R, part, bnd, gain, dest, pw)
    print(f"n={g.n} k={k} candidates={int((gain > 0).sum())} nmoves={got['nmoves']} pos={got['pos']}", flush=True)
    compare_rounds(got, exp, M)


# vertices around one bitmap (65536 ids) and candidates from a few to far more
# than the list holds (4096): flips of the given share of the vertices make
# about ten candidates each
@pytest.mark.parametrize("n", [700, 65535, 65536, 65537, 200000])
@pytest.mark.parametrize("flip", [0.0005, 0.005, 0.05])
def test_sizes(gk, oracle, ctx, n, flip):
    check(gk, oracle, ctx, gk.delaunay(n, 4), 16, 1024, 12, 8, None, flip)


@pytest.mark.parametrize("k", [1, 2, 3, 255, 256, 257])
def test_part_counts(gk, oracle, ctx, k):
    check(gk, oracle, ctx, gk.dag(20000, 40, 6), k, 1024, 15, 10, 12, 0.01)


# caps that cut the prefix short (few moves a round, the list corrected many
# times over) and small move caps (thresholds, deferred tests)
@pytest.mark.parametrize("M,slack", [(1024, 2), (1024, 30), (7, 5), (64, 1000), (65, 1000), (16, None)])
def test_many_rounds(gk, oracle, ctx, M, slack):
    check(gk, oracle, ctx, gk.dag(50000, 100, 8), 64, M, 120, 12, slack, 0.004)


# rows longer than the lanes of a vertex and than a lane tests by itself, and
# hubs whose moves update more than the workgroup does
@pytest.mark.parametrize("fan,k", [(40, 8), (300, 16), (1500, 200)])
def test_long_rows(gk, oracle, ctx, fan, k):
    g = hub_graph(gk, n=6000, hubs=30, fan=fan, seed=fan)
    check(gk, oracle, ctx, g, k, 1024, 20, 9, 20, 0.02)


def test_batch_more_jobs_than_compute_units(gk, ctx):
    """More than 256 jobs take the short candidate list; some of them exceed
    it (flat random weights make many candidates)."""
    rng = np.random.default_rng(3)
    graphs, ks = [], []
    for i in range(300):
        n = int(rng.integers(300, 900)) if i % 30 else 20000
        graphs.append(gk.dag(n, max(2, int(np.sqrt(n))), 100 + i) if i % 2 == 0 else gk.delaunay(n, 100 + i))
        ks.append(int(rng.choice([2, 4, 8])) if n < 1000 else 64)
    for flags in (0, gk.GK_FLAG_GRAPH_ROUNDS | gk.GK_FLAG_PERSISTENT):
        parts, stats = ctx.partition_batch(graphs, ks, flags=flags)
        for i in list(range(0, 300, 37)) + [0, 30, 60]:
            assert np.array_equal(parts[i], ctx.partition(graphs[i], ks[i])[0]), i


# The short way of the V-cycle's rounds (the best movable vertices, applied one
# after another by one wave, with the proof that no later prefix is balanced)
# against the oracle, level by level: unit weights (hundreds of equal gains in
# one class), weights over several orders of magnitude, hubs, a tight and a
# loose cap, move caps below and above a round's movable vertices.
def weighted(gk, g, top, seed):
    """g with symmetric edge weights 1..top, spread over their logarithm."""
    rng = np.random.default_rng(seed)
    src = np.repeat(np.arange(g.n), g.degrees())
    key = np.minimum(src, g.adjncy) * np.int64(g.n) + np.maximum(src, g.adjncy)
    _, inv = np.unique(key, return_inverse=True)
    w = np.exp(rng.uniform(0, np.log(top), inv.max() + 1)).astype(np.int64)[inv]
    return gk.Graph(g.xadj, g.adjncy, np.maximum(w, 1), rng.integers(1, 9, g.n))


@pytest.mark.parametrize("k,ub,moves", [(2, 30, 1024), (8, 0, 1024), (64, 5, 1024), (256, 30, 1024), (32, 30, 300), (16, 100, 40)])
@pytest.mark.parametrize("name", ["mesh", "weighted", "dag", "hubs"])
def test_vcycle_rounds(gk, oracle, ctx, name, k, ub, moves):
    from test_gpu_parity import compare
    g = {"mesh": lambda: gk.delaunay(70000, 21), "weighted": lambda: weighted(gk, gk.delaunay(30000, 22), 20000, 1),
         "dag": lambda: gk.dag(40000, 120, 23), "hubs": lambda: hub_graph(gk, n=12000, hubs=40, fan=200, seed=24)}[name]()
    compare(gk, oracle, ctx, g, k, ubfactor=ub, max_moves=moves)
