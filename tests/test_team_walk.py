"""CPU model of the team decode's indexing (pa_fp8_team_kernel): runs of the
cost order per workgroup, sub-runs per wave, and the two merges.

Restates the kernel's integer steps on random batches and checks what its
results depend on: every chunk of every (sequence, kv head) pair is computed
once; the LDS slots a fold reads are exactly those the pair's pieces in that
run were written to, folded by one wave; a pair cut between workgroups
writes one workspace slot per run, the count that triggers its merge is the
number of slots written, and the merge reads exactly those; a pair short
enough not to be cut is held by one workgroup.  The GPU tests check the
numbers.
"""

from __future__ import annotations

import random

import pytest

from tests.test_balanced_walk import run_begin, run_of_chunk, seq_chunks

W = 8
A = 1
MIN_CHUNKS = 32
SNAP = 32


class Team:
    def __init__(self, nbs, H, grid):
        self.nbs, self.H, self.grid = nbs, H, grid
        self.T = sum(n + A for n in nbs if n) * H
        pairs = sum(1 for n in nbs if n) * H
        self.nw = min(max(self.T // MIN_CHUNKS, pairs), grid) if self.T else 0
        if self.nw:
            self.snap = SNAP if self.nw < grid else min(SNAP, self.T // self.nw // 8)

    def locate(self, g):
        base = 0
        for b, n in enumerate(self.nbs):
            q = n + A if n else 0
            if (base + q) * self.H > g:
                return b, n, base * self.H
            base += q
        raise AssertionError("position past the end")

    def boundary(self, r):
        if r <= 0:
            return 0
        if r >= self.nw:
            return self.T
        g = run_begin(r, self.T, self.nw)
        _, n, base = self.locate(g)
        if n > self.snap:
            return g
        o = (g - base) % (n + A)
        return g - o + (n + A if 2 * o >= n + A else 0)

    def pieces(self, x0, x1):
        """(b, h, c0, n, nb, P) of the wave whose sub-run is [x0, x1)."""
        out = []
        if x1 <= x0:
            return out
        b, nb, base = self.locate(x0)
        h, o = divmod(x0 - base, nb + A)
        c, P = max(o - A, 0), base + h * (nb + A)
        pos = P + A + c
        while pos < x1:
            n = min(nb - c, x1 - pos)
            out.append((b, h, c, n, nb, P))
            c += n
            pos += n
            if pos < x1 and c == nb:
                c, P = 0, P + nb + A
                pos, h = P + A, h + 1
                if h >= self.H:
                    h, b = 0, b + 1
                    while b < len(self.nbs) and self.nbs[b] == 0:
                        b += 1
                    if b == len(self.nbs):
                        break
                    nb = self.nbs[b]
        return out


def check(nbs, H, grid):
    t = Team(nbs, H, grid)
    chunks, whole, slots, counts = {}, set(), {}, {}
    bounds = [t.boundary(r) for r in range(t.nw + 1)]
    assert bounds == sorted(bounds)
    for run in range(t.nw):
        g0, g1 = bounds[run], bounds[run + 1]
        if g1 <= g0:
            continue
        sub = [g0 + (g1 - g0) * w // W for w in range(W + 1)]
        held = {}  # (pair) -> {(wave, lds slot)} written by its cut pieces
        ends = {}
        for w in range(W):
            got = t.pieces(sub[w], sub[w + 1])
            for i, (b, h, c0, n, nb, P) in enumerate(got):
                chunks.setdefault((b, h), []).extend(range(c0, c0 + n))
                if c0 == 0 and n == nb:
                    whole.add((b, h))
                    continue
                assert i in (0, len(got) - 1)
                which = 0 if i == 0 else 1
                held.setdefault((b, h), set()).add((w, which))
                q0 = P + A
                ce = min(nb, g1 - q0)
                if c0 + n == ce:
                    assert (b, h) not in ends
                    ends[b, h] = (w, P, nb, max(g0 - q0, 0), ce)
        assert set(ends) == set(held)
        sides = set()
        for (b, h), (wave, P, nb, cs, ce) in ends.items():
            q0 = P + A
            read = {(r, 0 if sub[r] >= P else 1) for r in range(wave + 1)
                    if max(sub[r], q0) < min(sub[r + 1], q0 + nb)}
            assert read == held[b, h], (b, h, read, held[b, h])
            if cs == 0 and ce == nb:
                whole.add((b, h))
                continue
            side = 0 if cs > 0 else 1
            assert side not in sides  # one pair per side of a run
            sides.add(side)
            rf = run_of_chunk(q0, t.T, t.nw)
            n = run_of_chunk(q0 + nb - 1, t.T, t.nw) - rf + 1
            slots.setdefault((b, h), set()).add(2 * run + side)
            counts.setdefault((b, h), set()).add((rf, n))
    for b, nb in enumerate(nbs):
        for h in range(H):
            assert sorted(chunks.get((b, h), [])) == list(range(nb)), (b, h)
            if nb == 0:
                continue
            assert ((b, h) in whole) != ((b, h) in slots)
            if (b, h) in slots:
                ((rf, n),) = counts[b, h]  # every run derives the same
                assert n > 1 and {2 * (rf + i) + (1 if i == 0 else 0) for i in range(n)} == slots[b, h]
                assert max(slots[b, h]) < 2 * grid
                assert nb > t.snap
    return t, slots


@pytest.mark.parametrize("seed", range(60))
def test_every_chunk_once_and_every_merge_reads_what_was_written(seed):
    rng = random.Random(seed)
    B = rng.randint(1, 60)
    top = rng.choice([40, 600, 6000, 40000])
    ctxs = [rng.choice([0, 1, 2, 17, 31, 32, 33]) if rng.random() < 0.2 else rng.randint(1, top) for _ in range(B)]
    ql, window = rng.choice([1, 1, 2, 4]), rng.choice([0, 0, 100, 1000])
    check([seq_chunks(c, ql, window) for c in ctxs], rng.choice([1, 2, 3, 8]), rng.choice([1, 2, 7, 64, 256]))


def test_short_batches_keep_one_pair_per_workgroup():
    t, slots = check([16, 3, 9, 1], 2, 256)
    assert t.nw == 8 and not slots
    # one long pair is cut once every 32 chunks of cost
    t, slots = check([1024], 1, 256)
    assert t.nw == 32 and len(slots[0, 0]) == 32
    # more pairs than workgroups, none of them longer than an eighth of a run
    t, slots = check([4] * 512, 8, 256)
    assert t.nw == 256 and not slots
