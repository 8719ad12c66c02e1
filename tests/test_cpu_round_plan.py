"""The bookkeeping of a level's refinement rounds (csrc/round_plan.hpp), compiled
for the host and driven through made-up answers of the device: which launches
follow, how many rounds are accounted for, and what bounds them."""
import ctypes
import os
import random
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dac_g-kway_amd", "csrc")
SHIM = r"""
#include "round_plan.hpp"
using P = gkrt::RoundPlan;
extern "C" {
P* make(int can_loop, long long n, int nj, int max_rounds, int exact, int graph) {
  return new P(can_loop, n, nj, max_rounds, exact, graph);
}
void drop(P* p) { delete p; }
int ended(P* p) { return p->ended(); }
int loop(P* p) { return p->loop(); }
int rounds(P* p) { return p->rounds(); }
int captured(P* p) { return p->captured(); }
int pair_of(P* p) { return p->pair(); }
int done(P* p) { return p->done(); }
void loop_ran(P* p, int live, int left_out, int ordered) { p->loop_ran(live, left_out, ordered); }
int wide_ran(P* p, int live) { return p->wide_ran(live); }
}
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    d = tmp_path_factory.mktemp("round_plan")
    (d / "shim.cpp").write_text(SHIM)
    so = d / "shim.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-shared", "-fPIC", "-I", CSRC, str(d / "shim.cpp"), "-o", str(so)],
                   check=True, timeout=120)
    L = ctypes.CDLL(str(so))
    L.make.restype = ctypes.c_void_p
    L.make.argtypes = [ctypes.c_int, ctypes.c_longlong] + [ctypes.c_int] * 4
    for f in ("ended", "loop", "rounds", "captured", "pair_of", "done", "drop"):
        getattr(L, f).argtypes = [ctypes.c_void_p]
    L.loop_ran.argtypes = [ctypes.c_void_p] + [ctypes.c_int] * 3
    L.wide_ran.argtypes = [ctypes.c_void_p, ctypes.c_int]
    return L


class Plan:
    def __init__(self, shim, can_loop=True, n=100000, nj=1, max_rounds=0, exact=False, graph=False):
        self.L, self.p = shim, shim.make(can_loop, n, nj, max_rounds, exact, graph)

    def __del__(self):
        self.L.drop(self.p)

    def __getattr__(self, name):
        return getattr(self.L, {"pair": "pair_of"}.get(name, name))(self.p)

    def loop_ran(self, live, left_out, ordered=0):
        self.L.loop_ran(self.p, live, left_out, ordered)

    def wide_ran(self, live):
        return self.L.wide_ran(self.p, live)


def test_rounds_given_back_are_those_of_the_launch(shim):
    """A launch that leaves a job out gives back its own rounds, not those that
    the separate kernels have run before it."""
    p = Plan(shim, nj=3, max_rounds=64)
    assert p.loop and p.rounds == 64
    p.loop_ran(3, 3)
    assert not p.loop and p.done == 0 and p.rounds == 4
    assert p.wide_ran(900) == 1
    assert p.loop and p.done == 4 and p.rounds == 60
    p.loop_ran(2, 1)
    assert not p.loop and p.done == 4
    assert p.wide_ran(100000) == 0
    assert p.done == 8


@pytest.mark.parametrize("seed", range(60))
def test_every_round_is_accounted_for_once(shim, seed):
    rng = random.Random(seed)
    nj = rng.choice([1, 2, 9, 300])
    p = Plan(shim, can_loop=rng.random() < 0.9, n=rng.choice([1000, 3_000_000]), nj=nj,
             max_rounds=rng.choice([1, 3, 64, 100, 128, 256]), graph=rng.random() < 0.5)
    told = 0
    for _ in range(10000):
        if p.ended:
            break
        n = p.rounds
        assert n > 0
        if p.loop:
            left_out = rng.choice([0, 0, 1, nj])
            live = max(left_out, rng.choice([0, 1, nj]))
            told += n if live == 0 or left_out == 0 else 0
            p.loop_ran(live, left_out)
        else:
            told += n
            p.wide_ran(rng.choice([0, 500, 5000, 5000, 10**6]))
        assert p.done == told
    assert p.ended


# A step of a batch ends soon whatever its jobs do: at most a quarter of its
# rounds by the separate kernels (to the next look), and so many launches of the
# loop that leave jobs out as that number can be halved.  The answers are those
# that once kept a step going for 3000 rounds: selections small enough to go
# back to the loop, which leaves out the same jobs again.
@pytest.mark.parametrize("max_rounds", [4, 16, 64, 128, 256])
@pytest.mark.parametrize("nj", [1, 5, 64, 500])
@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("left", ["same", "one", "halves", "random"])
def test_a_step_is_bounded(shim, max_rounds, nj, graph, left):
    rng = random.Random(nj)
    p = Plan(shim, nj=nj, max_rounds=max_rounds, graph=graph)
    wide = attempts = 0
    out = nj
    while not p.ended and wide + attempts < 10000:
        if p.loop:
            attempts += 1
            p.loop_ran(nj, out)
            out = {"same": out, "one": 1, "halves": max(1, out // 2), "random": rng.randint(1, nj)}[left]
        else:
            wide += p.rounds
            p.wide_ran(rng.randint(1, 1024 * nj))
    assert p.ended
    assert wide < max(4, max_rounds // 4) + 32
    assert attempts <= 2 + nj.bit_length()


@pytest.mark.parametrize("seed", range(60))
def test_launches_find_their_words_cleared(shim, seed):
    """Pairs of counts and status words: a launch of the loop raises its own
    pair, which must be zero, and clears the other; a replay is two launches
    that begin with the pair they were captured with; the separate kernels raise
    pair 0, and both pairs are cleared on the way back to the loop."""
    rng = random.Random(seed)
    nj = rng.choice([1, 4, 100])
    exact = nj == 1 and rng.random() < 0.3
    p = Plan(shim, n=rng.choice([1000, 3_000_000]), nj=nj, max_rounds=0 if rng.random() < 0.3 else rng.randint(1, 256),
             exact=exact, graph=not exact and rng.random() < 0.7)
    zero, held, ordered = [False, True], None, 0

    def launch(pair):
        assert zero[pair]
        zero[pair], zero[1 - pair] = False, True

    for _ in range(300):
        if p.ended:
            break
        if p.loop:
            if p.captured:
                held = p.pair if held is None else held
                launch(held)
                launch(1 - held)
            else:
                launch(p.pair)
            ordered += rng.randint(1, p.rounds)
            live = rng.choice([0, nj, nj, nj])
            p.loop_ran(live, rng.choice([0, 0, 1]) if live else 0, ordered)
        else:
            zero[0] = False
            ordered += p.rounds
            if p.wide_ran(rng.choice([1, 900, 10**6])):
                zero = [True, True]
