"""Words that decide a branch of the round loop (csrc/rounds.hip).

A workgroup's waves pass a barrier one after another.  A branch that holds
barriers must be taken by all of them or by none, so the LDS word that decides
it may not be raised inside the branch before its first barrier: a wave that
comes late would read another value.  Shown twice: the choice of the gain
classes restated and run over many orders of its waves, and the source itself
searched for a word that is both tested and raised.
"""
import os
import random
import re

import pytest

SOURCE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dac_g-kway_amd", "csrc", "rounds.hip")
WAVES = 16
NO_CLASS = -1


def class_cut(appends, enough, rng, decide):
    """Between the barrier after wave 0's choice and the next one: every wave
    reads the deciding word, and in the branch appends its vertices (appends:
    so many per wave).  Returns the branch each wave took and the count."""
    words = {"ntop": 0, "code": 7 if enough else NO_CLASS}
    if decide == "counter" and not enough:
        words["ntop"] = -1

    def wave(n):
        taken = words["ntop"] == 0 if decide == "counter" else words["code"] != NO_CLASS
        yield
        for _ in range(n if taken else 0):
            words["ntop"] += 1
            yield
        return taken

    live = {w: wave(n) for w, n in enumerate(appends)}
    took = [None] * len(appends)
    while live:
        w = rng.choice(list(live))
        try:
            next(live[w])
        except StopIteration as end:
            took[w] = end.value
            del live[w]
    return took, words["ntop"]


@pytest.mark.parametrize("seed", range(20))
@pytest.mark.parametrize("enough", [True, False])
def test_every_wave_takes_the_same_branch(seed, enough):
    rng = random.Random(seed)
    appends = [rng.randint(0, 4) for _ in range(WAVES)]
    took, count = class_cut(appends, enough, rng, "code")
    assert took == [enough] * WAVES
    assert count == (sum(appends) if enough else 0)


def test_a_counter_may_not_decide():
    """The rule that the model rejects: the counter itself as deciding word."""
    split = 0
    for seed in range(100):
        took, _ = class_cut([1] * WAVES, True, random.Random(seed), "counter")
        split += len(set(took)) > 1
    assert split > 0


def body_of(text, brace):
    depth = 0
    for i in range(brace, len(text)):
        depth += {"{": 1, "}": -1}.get(text[i], 0)
        if depth == 0:
            return text[brace:i]
    raise ValueError("unbalanced braces")


def raised_deciders(text):
    """(condition, word) of every `if` on a member of L whose body raises that
    member (takes its address, for an atomic or an append) before a barrier."""
    text = re.sub(r"//[^\n]*", "", text)
    found = []
    for m in re.finditer(r"\bif \(((?:[^(){};]|\([^(){};]*\))*)\) \{", text):
        body = body_of(text, m.end() - 1).split("__syncthreads()")[0]
        if "__syncthreads()" not in body_of(text, m.end() - 1):
            continue  # no barrier inside: the waves need not agree
        for word in set(re.findall(r"\bL\.(\w+)\b(?!\s*[\[(.])", m.group(1))):
            if re.search(r"&L\." + word + r"\b", body) or re.search(r"\bL\." + word + r"\s*[-+|]?=[^=]", body):
                found.append((m.group(1), word))
    return found


def test_no_word_is_tested_and_raised():
    with open(SOURCE) as f:
        assert raised_deciders(f.read()) == []


def test_the_search_finds_one():
    bad = "if (L.ntop == 0) { wave_append(x, i, L.tj, &L.ntop); __syncthreads(); }"
    good = "if (code != kNoClass) { wave_append(x, i, L.tj, &L.ntop); __syncthreads(); }"
    late = "if (L.n > kFull) { n = L.n; __syncthreads(); if (t == 0) L.n = 0; }"
    assert raised_deciders(bad) == [("L.ntop == 0", "ntop")]
    assert raised_deciders(good) == [] and raised_deciders(late) == []
