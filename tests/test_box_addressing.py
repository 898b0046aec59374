"""Host replay of the box sweeps' addressing (csrc/dilu_box.hip): the steps of
a tile's three waves, for many tile grids (every tile width, both sweep
directions, whole tiles and the segments of lone ones).  It checks that

- the stream wave's step i reads the slice that the compute wave's step i
  writes, and a step past the end reads the last;
- in a FULL group every in-tile row is valid, and its rows and deliveries are
  reached with the group's scalar offsets and non-negative constants;
- every value delivered across an edge lands in the consumer's inbox, at the
  step of the consumer that needs it;
- the feed wave takes exactly the delivered values, each by one lane, in the
  order of its steps, and the clearing covers them.

The tile grid follows layout.cpp boxWaves (steps = nA + actB - 1 + actC - 1).
"""
import itertools
import random

import pytest

kG, kAhead, kIn = 8, 8, 16


def tangential(a):
    return {0: (1, 2), 1: (0, 2), 2: (0, 1)}[a]


def tile_grid(n, TB):
    a = 0
    for q in (1, 2):
        if n[q] > n[a]:
            a = q
    b, c = tangential(a)
    TC = 64 // TB
    nTB, nTC = -(-n[b] // TB), -(-n[c] // TC)
    tiles = {}
    for tc in range(nTC):
        for tb in range(nTB):
            actB, actC = min(TB, n[b] - tb * TB), min(TC, n[c] - tc * TC)
            tiles[(tb, tc)] = dict(nA=n[a], actB=actB, actC=actC, steps=n[a] + actB - 1 + actC - 1)
    return tiles, TC


def segment(nA, s, segs):
    """dilu.hpp boxSegment: rows [lo, hi) of segment s of segs."""
    return s * nA // segs, (s + 1) * nA // segs


def time_of(m, lo, hi, fwd, i):
    """boxStream timeOf: the slice of step i, clamped to the last."""
    tLo = m["actB"] - 1 + m["actC"] - 1
    i = min(i, hi - lo + tLo - 1)
    return lo + i if fwd else hi - 1 + tLo - i


def groups(m, lo, hi, fwd):
    """boxCompute's groups: (first step, T of its steps, FULL)."""
    tLo = m["actB"] - 1 + m["actC"] - 1
    for g in range(0, hi - lo + tLo, kG):
        T0 = lo + g if fwd else hi - 1 + tLo - g
        tMin = lo + g if fwd else hi - 1 + tLo - (g + kG - 1)
        yield g, [T0 + u if fwd else T0 - u for u in range(kG)], tMin >= lo + tLo and tMin + kG - 1 <= hi - 1


def replay(n, TB, fwd):
    """All tiles of a box; returns the number of FULL groups."""
    tiles, TC = tile_grid(n, TB)
    full_groups = 0
    delivered = {}   # (tile, edge) -> {(inbox row, value): ia}
    for (tb, tc), m in tiles.items():
        nA, actB, actC, nSteps = m["nA"], m["actB"], m["actC"], m["steps"]
        toB = tiles.get((tb + 1, tc) if fwd else (tb - 1, tc))
        toC = tiles.get((tb, tc + 1) if fwd else (tb, tc - 1))
        dB, dC = (1 - TB, 1 - TC) if fwd else (TB - 1, TC - 1)
        mOff = min(dB if toB else 0, dC if toC else 0, 0)
        for g, times, full in groups(m, 0, nA, fwd):
            full_groups += full
            Tlow = min(times)
            for u, T in enumerate(times):
                if g + u < nSteps:
                    assert time_of(m, 0, nA, fwd, g + u) == T
                if full:
                    # the output row: a scalar offset and a constant
                    assert 0 <= Tlow <= T < nSteps and 0 <= T - Tlow < kG
                for bl, cl in itertools.product(range(actB), range(actC)):
                    ia = T - bl - cl
                    valid = 0 <= ia < nA
                    assert valid or not full
                    if not valid:
                        continue
                    assert 0 <= T < nSteps
                    for to, d, edge, val, send in (
                            (toB, dB, "b", cl, bl == (TB - 1 if fwd else 0)), (toC, dC, "c", bl, cl == (TC - 1 if fwd else 0))):
                        if to is None or not send:
                            continue
                        if full:
                            assert T + mOff >= 0 and d - mOff >= 0
                        row = T + d
                        assert 0 <= row < to["steps"]
                        key = ((tb + (edge == "b") * (1 if fwd else -1), tc + (edge == "c") * (1 if fwd else -1)), edge)
                        put = delivered.setdefault(key, {})
                        assert (row, val) not in put
                        put[(row, val)] = ia
    # the consumers
    for (tb, tc), m in tiles.items():
        nA, actB, actC, nL = m["nA"], m["actB"], m["actC"], m["steps"]
        prevB = tiles.get((tb - 1, tc) if fwd else (tb + 1, tc)) is not None
        prevC = tiles.get((tb, tc - 1) if fwd else (tb, tc + 1)) is not None
        for edge, fed, width, every, act in (("b", prevB, TC, TB, actC), ("c", prevC, TB, TC, actB)):
            put = delivered.get(((tb, tc), edge), {})
            assert fed == bool(put)
            taken = {}
            for lane in range(64):
                val = lane % width
                off = (0 if fwd else every - 1) + val
                first = off if fwd else nL - off - nA
                if not fed or val >= act:
                    continue
                for i in range(first + lane // width, first + nA, every):
                    row = i if fwd else nL - 1 - i
                    assert 0 <= i < nL and (row, val) not in taken
                    taken[(row, val)] = i
            assert taken.keys() == put.keys()
            # step i of the consumer computes the delivered cell's neighbour
            for (row, val), i in taken.items():
                T = time_of(m, 0, nA, fwd, i)
                near = 0 if fwd else every - 1
                assert T == row and T - val - near == put[(row, val)]
            # cleared: every row of the tile's steps, `width` values each
            assert all(0 <= row < nL and 0 <= val < width for row, val in put)
    return full_groups


def replay_segments(n, TB, fwd, segs):
    """The lone (tile-local) sweep of each segment of each tile."""
    tiles, _ = tile_grid(n, TB)
    full_groups = 0
    for m in tiles.values():
        covered = set()
        for sg in range(segs):
            lo, hi = segment(m["nA"], sg, segs)
            if hi <= lo:
                continue
            rows = set()
            for g, times, full in groups(m, lo, hi, fwd):
                full_groups += full
                for u, T in enumerate(times):
                    assert 0 <= time_of(m, lo, hi, fwd, g + u + kAhead) < m["steps"]
                    for bl, cl in itertools.product(range(m["actB"]), range(m["actC"])):
                        ia = T - bl - cl
                        valid = lo <= ia < hi
                        assert valid or not full
                        if valid:
                            assert 0 <= T < m["steps"] and time_of(m, lo, hi, fwd, g + u) == T
                            rows.add((bl, cl, ia))
            assert len(rows) == (hi - lo) * m["actB"] * m["actC"] and not rows & covered
            covered |= rows
        assert len(covered) == m["nA"] * m["actB"] * m["actC"]
    return full_groups


def shapes():
    rng = random.Random(7)
    out = [(160, 80, 80), (200, 100, 19), (37, 23, 29), (41, 27, 7), (12, 14, 40), (5, 5, 5), (64, 1, 1),
           (3, 7, 200), (100, 2, 3), (70, 130, 1), (1, 66, 90)]
    out += [tuple(rng.randint(1, 60) for _ in range(3)) for _ in range(8)]
    return out


def small(n):
    return n[0] * n[1] * n[2] <= 60000


@pytest.mark.parametrize("TB", [1, 2, 4, 8, 16, 32, 64])
def test_steps_and_deliveries(TB):
    full = 0
    for n in shapes():
        if small(n):
            for fwd in (True, False):
                full += replay(n, TB, fwd)
    assert full > 0


def test_duct_fluid_tiles_run_mostly_full_groups():
    for fwd in (True, False):
        tiles, _ = tile_grid((160, 80, 80), 8)
        full = sum(f for m in tiles.values() for _, _, f in groups(m, 0, m["nA"], fwd))
        assert full == 18 * len(tiles)   # of 22 groups (174 steps)


@pytest.mark.parametrize("segs", [2, 3])
def test_segments_of_lone_tiles(segs):
    full = 0
    for n in shapes():
        if small(n):
            for TB in (1, 4, 8, 16, 64):
                for fwd in (True, False):
                    full += replay_segments(n, TB, fwd, segs)
    assert full > 0
