"""The exchange of the resident CG engine as a model on the CPU: a team's members, each with its words of
two parities, run the kernel's sequence of publications, all-gathers and reads in random interleavings.

Rules of the model are those of the kernel: a word holds the tag it was written under; a reader polls until
every word it needs shows exactly that tag, all of them in one pass; stores of one member to different
words become visible in any order. Lost: a word that a reader still needs has gone on to a later tag (the
reader would poll until it gives up). The sequence with a residual replacement that exchanges x without an
all-gather under its tag is the planted mistake the model has to find."""
from __future__ import annotations

import random

import pytest

MEMBERS = 6


class Lost(Exception):
    pass


class Words:
    """[parity][member] tags; stores travel, in order for each word."""

    def __init__(self, members):
        self.tag = [[0] * members for _ in range(2)]
        self.flying = []

    def store(self, member, tag):
        self.flying.append((tag & 1, member, tag))

    def land(self, rng):
        """One store in flight becomes visible (the oldest of its word)."""
        if not self.flying:
            return
        parity, member, tag = rng.choice(self.flying)
        tag = next(t for p, m, t in self.flying if (p, m) == (parity, member))
        self.flying.remove((parity, member, tag))
        self.tag[parity][member] = tag

    def shows(self, member, tag):
        seen = self.tag[tag & 1][member]
        if seen > tag:
            raise Lost(f"word of member {member}: tag {tag} wanted, {seen} seen")
        return seen == tag


def member(me, sums, vecs, needs, iterations, reset_every, early, sound):
    """The kernel's exchanges as a member runs them; yields between any two accesses to the words."""
    tag = 0

    def all_gather(read=()):
        nonlocal tag
        tag += 1
        sums.store(me, tag)
        yield
        for other in read:  # the vector words, while the sums travel
            while not vecs.shows(other, tag):
                yield
            yield
        done = False
        while not done:
            done = True
            for other in range(MEMBERS):
                done = sums.shows(other, tag) and done
                yield

    def publish():
        vecs.store(me, tag + 1)
        yield

    def fetch(at):
        for other in needs:
            while not vecs.shows(other, at):
                yield
            yield

    yield from all_gather()                      # mean of b
    yield from publish()                         # z
    yield from all_gather(needs if early else ())
    ztag = tag
    for it in range(1, iterations + 1):
        if reset_every and it > 1 and (it - 1) % reset_every == 0:
            yield from publish()                 # x
            if sound:
                yield from all_gather()
            else:
                tag += 1
            yield from fetch(tag)
            yield from publish()                 # z
            yield from all_gather(needs if early else ())
            ztag = tag
        if not early:
            yield from fetch(ztag)
        yield from all_gather()                  # (p, q)
        yield from publish()                     # z
        yield from all_gather(needs if early else ())
        ztag = tag


def run(seed, neighbours, reset_every, early, sound=True, iterations=8):
    rng = random.Random(seed)
    sums, vecs = Words(MEMBERS), Words(MEMBERS)
    team = {m: member(m, sums, vecs, neighbours(m), iterations, reset_every, early, sound) for m in range(MEMBERS)}
    # members of very different speeds, one of them changing now and then
    pace = [10 ** rng.uniform(-1.5, 0) for _ in range(MEMBERS)]
    for _ in range(2_000_000):
        if not team:
            return
        if rng.random() < 0.002:
            pace[rng.randrange(MEMBERS)] = 10 ** rng.uniform(-1.5, 0)
        if rng.random() < 0.5:
            sums.land(rng)
            vecs.land(rng)
        live = list(team)
        m = rng.choices(live, [pace[k] for k in live])[0]
        if next(team[m], "end") == "end":
            del team[m]
    raise AssertionError("the model did not come to an end")


CHAIN = lambda m: [k for k in (m - 1, m + 1) if 0 <= k < MEMBERS]  # noqa: E731
ONE_WAY = lambda m: [k for k in (m - 1,) if k >= 0]  # noqa: E731  (a structurally one-sided pattern)


@pytest.mark.parametrize("early", [True, False], ids=["fetch with the sums", "fetch after them"])
@pytest.mark.parametrize("neighbours", [CHAIN, ONE_WAY], ids=["chain", "one way"])
@pytest.mark.parametrize("reset_every", [0, 1, 3])
def test_no_word_is_lost(neighbours, reset_every, early):
    for seed in range(40):
        run(seed, neighbours, reset_every, early)


@pytest.mark.parametrize("early", [True, False], ids=["fetch with the sums", "fetch after them"])
def test_model_finds_a_replacement_without_an_all_gather(early):
    lost = 0
    for seed in range(40):
        try:
            run(seed, CHAIN, 3, early, sound=False)
        except Lost:
            lost += 1
    assert lost > 20, lost
