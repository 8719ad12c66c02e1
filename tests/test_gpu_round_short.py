"""Rounds that are decided by their best moves alone (the round loop's short
way), which gk_k_round takes when nobody asks for the moves: the state after
every round against the oracle's select / balance / apply / gain.  Whole
numbers, so exactly.

The cases lie where the short way ends or hands over: a tight cap (a few moves
decide) and loose ones (64 moves prove nothing, all are ordered), fewer and more
movable vertices than the 256 it looks at, gains that all fall in one class or
in many, move caps below, at and above the 64 moves it applies, more vertices
than the movable bitmap has bits, hubs."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from test_gpu_round import gpu_rounds, oracle_rounds, state  # noqa: E402
from test_gpu_stages import hub_graph  # noqa: E402

STATE = ("part", "bnd", "gain", "dest", "pw")


def unseen_rounds(gk, ctx, g, k, cap, M, calls, R, start):
    """calls times R rounds without nmoves, pos and order; the state after each call."""
    from _dev import DevGraph, dev, host, ptr
    dg = DevGraph(g)
    d = {name: dev(a) for name, a in zip(STATE, start)}
    gs, paths, out = ctypes.c_int64(0), (ctypes.c_int64 * 3)(), []
    for _ in range(calls):
        rc = gk.lib().gk_k_round(ctx.handle, dg.ref(), k, cap, M, R, *(ptr(d[x]) for x in STATE), None, None,
                                 ctypes.byref(gs), None, paths, None)
        assert rc == 0, gk.lib().gk_last_error().decode()
        out.append({**{name: host(t).copy() for name, t in d.items()}, "gain_sum": gs.value, "paths": list(paths)})
    return out


def check(gk, oracle, ctx, g, k, M, R, gbits, slack, flip, seed=5):
    start = state(gk, g, k, seed=seed, gain_bits=gbits, flip=flip)
    part, bnd, gain, dest, pw = start
    cap = int(gk.lib().gk_part_cap(int(g.vwgt.sum()), k, 30)) if slack is None else int(pw.max()) + slack
    print(f"n={g.n} k={k} M={M} candidates={int((gain > 0).sum())} cap={cap}", flush=True)
    # all rounds in one call, then one round a call
    exp = oracle_rounds(oracle, g, k, cap, M, R, *start)
    got = unseen_rounds(gk, ctx, g, k, cap, M, 1, R, start)[0]
    assert got["gain_sum"] == exp["gain_sum"]
    for name in STATE:
        assert np.array_equal(got[name], exp[name]), name
    print(f"  nmoves={exp['nmoves']} pos={exp['pos']}", flush=True)
    now = start
    for r, got in enumerate(unseen_rounds(gk, ctx, g, k, cap, M, min(R, 12), 1, start)):
        exp = oracle_rounds(oracle, g, k, cap, M, 1, *now)
        assert got["gain_sum"] == exp["gain_sum"], r
        for name in STATE:
            assert np.array_equal(got[name], exp[name]), (r, name)
        now = tuple(exp[name] for name in STATE)


# The list of the round loop holds 3584 candidates: graphs of fewer vertices, or
# compact blocks of a mesh numbered along a curve, whose borders are short.
@pytest.mark.parametrize("slack", [1, 4, 30, 1000, None])
@pytest.mark.parametrize("gbits", [1, 4, 14])
@pytest.mark.parametrize("name", ["dag", "mesh"])
def test_caps_and_gains(gk, oracle, ctx, name, slack, gbits):
    g = gk.dag(3500, 30, 3) if name == "dag" else gk.delaunay_hilbert(30000, 3)
    check(gk, oracle, ctx, g, 16, 1024, 40, gbits, slack, 0.002)


@pytest.mark.parametrize("M", [1, 4, 63, 64, 65, 128, 256])
@pytest.mark.parametrize("slack", [3, 500])
def test_move_caps(gk, oracle, ctx, M, slack):
    check(gk, oracle, ctx, gk.delaunay_hilbert(12000, 6), 8, M, 40, 10, slack, 0.003)


@pytest.mark.parametrize("n,k,flip", [(65535, 2, 0.004), (65536, 8, 0.0005), (65537, 8, 0.0005), (200000, 4, 0.0002)])
def test_sizes(gk, oracle, ctx, n, k, flip):
    check(gk, oracle, ctx, gk.delaunay_hilbert(n, 9), k, 1024, 20, 12, 6, flip)


# from a handful of movable vertices to beyond the 256 that it looks at
@pytest.mark.parametrize("n,k", [(300, 2), (700, 4), (1500, 4), (2500, 256), (3400, 100)])
def test_few(gk, oracle, ctx, n, k):
    check(gk, oracle, ctx, gk.dag(n, 20, 9), k, 1024, 30, 8, 4, 0.01)


@pytest.mark.parametrize("fan,k", [(40, 8), (300, 16)])
def test_hubs(gk, oracle, ctx, fan, k):
    check(gk, oracle, ctx, hub_graph(gk, n=3000, hubs=20, fan=fan, seed=fan), k, 1024, 20, 9, 5, 0.01)


def test_same_as_seen(gk, ctx):
    """Asked for or not, the rounds leave the same state."""
    g, k, M, R = gk.delaunay_hilbert(30000, 4), 12, 200, 25
    start = state(gk, g, k, seed=8, gain_bits=11, flip=0.004)
    cap = int(start[4].max()) + 10
    seen = gpu_rounds(gk, ctx, g, k, cap, M, R, *start)
    got = unseen_rounds(gk, ctx, g, k, cap, M, 1, R, start)[0]
    assert got["gain_sum"] == seen["gain_sum"]
    for name in STATE:
        assert np.array_equal(got[name], seen[name]), name


@pytest.mark.parametrize("M,slack", [(64, 30), (60, 1000), (45, 30)])
def test_paths_count_what_ran(gk, ctx, M, slack):
    """More than M vertices are selected in most rounds: asked for, their moves
    are ordered by the radix select every time; decided by the best ones alone,
    the rounds are not among those that the select ordered."""
    g, k, R = gk.delaunay_hilbert(30000, 3), 16, 60
    start = state(gk, g, k, seed=5, gain_bits=4, flip=0.002)
    cap = int(start[4].max()) + slack
    seen = gpu_rounds(gk, ctx, g, k, cap, M, R, *start)
    got = unseen_rounds(gk, ctx, g, k, cap, M, 1, R, start)[0]
    print(f"M={M} nmoves={seen['nmoves']} pos={seen['pos']} paths: seen {seen['paths']} unseen {got['paths']}", flush=True)
    for name in STATE:
        assert np.array_equal(got[name], seen[name]), name
    assert sum(m == M for m in seen["nmoves"]) >= seen["paths"][0] > 0
    assert got["paths"][0] < seen["paths"][0]
    assert got["paths"][1] <= got["paths"][0]
