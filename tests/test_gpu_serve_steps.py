"""Steps with a job that has more candidates than the round loop holds (the
largest graph, on its levels of 171 and 43 thousand vertices) and ones that
end by the separate kernels' share of the rounds: each job goes on in a later
step, and its result is that of the graph alone.  Alone and with small jobs."""
import pytest

from test_gpu_serve import check_alone

pytestmark = pytest.mark.gpu


def run(gk, graphs, ks):
    with gk.Server() as srv:
        ids = srv.submit_many(graphs, ks)
        res = [srv.wait(r) for r in ids]
        return res, srv.stats()


@pytest.mark.parametrize("n", [40_000, 200_000, 600_000])
@pytest.mark.parametrize("small", [0, 1, 9])
def test_left_out(gk, ctx, n, small):
    graphs = [gk.dag(n, 200, 5)] + [gk.delaunay(3000 + 500 * i, i) for i in range(small)]
    ks = [256] + [16] * small
    res, stats = run(gk, graphs, ks)
    rounds = [max(1, st.levels[l].rounds) for _, st in res[:1] for l in range(st.nlevels)]
    print(f"n={n} small={small} steps={stats.steps} rounds={rounds}", flush=True)
    for (part, st), g, k in zip(res, graphs, ks):
        check_alone(ctx, g, k, part, st)
