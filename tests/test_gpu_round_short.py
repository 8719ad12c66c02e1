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


@pytest.mark.parametrize("slack", [1, 4, 30, 1000, None])
@pytest.mark.parametrize("flip", [0.0005, 0.004, 0.02])
@pytest.mark.parametrize("gbits", [1, 4, 14])
def test_caps_and_gains(gk, oracle, ctx, slack, flip, gbits):
    check(gk, oracle, ctx, gk.dag(20000, 60, 3), 32, 1024, 40, gbits, slack, flip)


@pytest.mark.parametrize("M", [1, 4, 63, 64, 65, 128, 256])
@pytest.mark.parametrize("slack", [3, 500])
def test_move_caps(gk, oracle, ctx, M, slack):
    check(gk, oracle, ctx, gk.delaunay(12000, 6), 16, M, 40, 10, slack, 0.003)


@pytest.mark.parametrize("n,k", [(65535, 2), (65537, 256), (200000, 64)])
def test_sizes(gk, oracle, ctx, n, k):
    check(gk, oracle, ctx, gk.delaunay(n, 9), k, 1024, 20, 12, 6, 0.001)


@pytest.mark.parametrize("fan,k", [(40, 8), (300, 16)])
def test_hubs(gk, oracle, ctx, fan, k):
    check(gk, oracle, ctx, hub_graph(gk, n=6000, hubs=30, fan=fan, seed=fan), k, 1024, 20, 9, 5, 0.01)


def test_same_as_seen(gk, ctx):
    """Asked for or not, the rounds leave the same state."""
    g, k, M, R = gk.dag(30000, 80, 4), 48, 200, 25
    start = state(gk, g, k, seed=8, gain_bits=11, flip=0.004)
    cap = int(start[4].max()) + 10
    seen = gpu_rounds(gk, ctx, g, k, cap, M, R, *start)
    got = unseen_rounds(gk, ctx, g, k, cap, M, 1, R, start)[0]
    assert got["gain_sum"] == seen["gain_sum"]
    for name in STATE:
        assert np.array_equal(got[name], seen[name]), name
