"""A model of the tile kernel's slot hand-out (tile_loop.hpp): a wave's first
64 slots are its own, the others come 64 at a draw from 16 cursors over
interleaved groups; the first wave that finds a cursor drained marks it in a
global word, and every one takes that word's marks, for its block too.  The second pass fills its
lanes with the unsure slots of as many batches as it takes.  Checked on the
CPU, with waves interleaved at random: every slot is handed out exactly once,
the second pass takes exactly the unsure pixels, with full waves but for each
wave's last, and every wave ends -- for empty, tiny and ragged launches,
launches of no more slots than lanes and grids that leave cursors without a
block; and, interrupted, no slot is handed out twice."""
import random

import pytest

CURSOR_DRAIN = 1 << 44
NC = 16
ALL = (1 << NC) - 1


def group_shift(left):
    return min(14, max(6, (left // NC | 1).bit_length() - 1))


def run(npts, nblocks, waves_per_block, seed, unsure=None, drain_at=None):
    rnd = random.Random(seed)
    cursors, drained = [0] * NC, 0
    held = 64 * nblocks * waves_per_block
    left = npts - held
    gsh = group_shift(left)
    low = (1 << gsh) - 1

    def slot_of(loc, cx):
        return held + ((((loc >> gsh) * NC + cx) << gsh) | (loc & low))

    def end_of(cx):
        g = left >> gsh
        return (((g + NC - 1 - cx) // NC) << gsh) + (left & low if g % NC == cx else 0)

    if left > 0:
        assert sum(end_of(c) for c in range(NC)) == left
    block_seen = [0] * nblocks
    counts = dict(draws=0, rounds=[])
    taken, skipped = [], []
    waves = [dict(block=b, cur=b % NC, seen=0, first=64 * (b * waves_per_block + v), begun=False, rest=[], sizes=[])
             for b in range(nblocks) for v in range(waves_per_block)]

    def draw(w):
        """The next batch's slots, or None; one cursor tried per call of step."""
        nonlocal drained
        if not w["begun"]:
            w["begun"] = True
            if left <= 0:
                w["seen"] = ALL
            return w["first"]
        while w["seen"] != ALL:
            w["seen"] |= block_seen[w["block"]]
            if w["seen"] == ALL:
                break
            cx = w["cur"] = next(c for c in ((w["cur"] + i) % NC for i in range(NC)) if not w["seen"] >> c & 1)
            loc = cursors[cx]
            cursors[cx] += 64
            counts["draws"] += 1
            if loc < end_of(cx):
                assert loc % 64 == 0
                return slot_of(loc, cx)
            w["seen"] |= drained | 1 << cx
            if loc - end_of(cx) < 64:
                drained |= 1 << cx
            block_seen[w["block"]] |= w["seen"]
        return None

    live = list(range(len(waves)))
    trips = 0
    while live:
        k = rnd.randrange(len(live))
        w = waves[live[k]]
        trips += 1
        if drain_at is not None and trips == drain_at:
            cursors, drained = [c + CURSOR_DRAIN for c in cursors], ALL
        lanes = []
        while len(lanes) < 64:
            if not w["rest"]:
                base = draw(w)
                if base is None:
                    break
                batch = [s for s in range(base, base + 64) if s < npts]
                if unsure is None:
                    lanes = batch
                    break
                w["rest"] = [s for s in batch if s in unsure]
                skipped.extend(s for s in batch if s not in unsure)
            else:
                room = 64 - len(lanes)
                lanes += w["rest"][:room]
                w["rest"] = w["rest"][room:]
        if not lanes:
            live.pop(k)
            continue
        taken.extend(lanes)
        w["sizes"].append(len(lanes))
    counts["sizes"] = [w["sizes"] for w in waves]
    return taken, skipped, counts


@pytest.mark.parametrize("npts,nblocks,waves", [
    (0, 8, 4), (1, 3, 2), (63, 8, 2), (64, 1, 1), (65, 1, 1), (2048, 8, 4), (2049, 8, 4), (64 * 8 * 5 + 17, 16, 4),
    (5000, 5, 3), (777, 1, 1), (100000, 32, 4), (300000, 8, 8), (150001, 2, 2), (1100000, 4, 4),
])
def test_every_slot_once_and_every_wave_ends(npts, nblocks, waves):
    for seed in range(3):
        taken, skipped, counts = run(npts, nblocks, waves, seed)
        assert sorted(taken) == list(range(npts)) and not skipped
        if npts <= 64 * nblocks * waves:
            assert counts["draws"] == 0


def test_second_pass_takes_the_unsure_pixels_in_full_waves():
    rnd = random.Random(3)
    unsure = set(rnd.sample(range(20000), 6000))
    taken, skipped, counts = run(20000, 12, 4, 7, unsure=unsure)
    assert sorted(taken) == sorted(unsure)
    assert sorted(taken + skipped) == list(range(20000))
    assert all(n == 64 for sizes in counts["sizes"] for n in sizes[:-1])


@pytest.mark.parametrize("drain_at", [1, 300, 700])
def test_interrupted_launch_takes_no_slot_twice(drain_at):
    taken, _, _ = run(100000, 16, 4, 5, drain_at=drain_at)
    assert len(set(taken)) == len(taken) < 100000
