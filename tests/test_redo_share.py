"""How the binary64 pass fills its waves (csrc/slot_rule.hpp, run on the host):
every unsure pixel once, no pixel of a drawn batch left behind while a lane is
free, and clustered pixels on many waves at once."""
import random

import pytest

import host_rules


def waves_of(unsure, nbatches, nwaves, seed):
    """The rounds (pixels iterated together) of each wave; batches are drawn in
    order by whichever wave is next."""
    rules, rnd = host_rules.load(), random.Random(seed)
    want = rules.redo_share(len(unsure), nwaves)
    order = iter(range(nbatches))
    rest, rounds = [[] for _ in range(nwaves)], [[] for _ in range(nwaves)]
    live = list(range(nwaves))
    while live:
        w = rnd.choice(live)
        lanes = []
        while len(lanes) < want:
            if not rest[w]:
                b = next(order, None)
                if b is None:
                    break
                rest[w] = [s for s in range(64 * b, 64 * b + 64) if s in unsure]
            else:
                goes = [bool(rules.slot_goes(len(lanes), k)) for k in range(len(rest[w]))]
                sent = [s for s, g in zip(rest[w], goes) if g]
                rest[w] = [s for s, g in zip(rest[w], goes) if not g]
                lanes += sent
                assert len(lanes) <= 64 and (not rest[w] or len(lanes) == 64)    # none left behind by a free lane
        if not lanes:
            live.remove(w)
            continue
        rounds[w].append(lanes)
    return rounds


@pytest.mark.parametrize("nbatches,nwaves,full,sparse", [
    (4096, 256, 4, 0), (4096, 256, 1, 0), (4096, 256, 200, 0), (1000, 64, 20, 30), (1000, 64, 0, 50), (1000, 64, 0, 5000),
    (300, 64, 300, 0), (64, 64, 64, 0), (200, 16, 3, 1000), (7, 64, 2, 3),
])
def test_every_unsure_pixel_once(nbatches, nwaves, full, sparse):
    rnd = random.Random(nbatches + full)
    unsure = {64 * b + k for b in rnd.sample(range(nbatches), full) for k in range(64)}
    unsure |= set(rnd.sample(range(64 * nbatches), sparse))
    rounds = waves_of(unsure, nbatches, nwaves, 5)
    assert sorted(s for w in rounds for r in w for s in r) == sorted(unsure)


@pytest.mark.parametrize("blocks", [1, 7, 63, 256])
def test_full_blocks_take_one_round_each(blocks):
    """As many full blocks as waves, or fewer: one round for each block, where a
    wave that stops at its share took up to 64."""
    unsure = {64 * (8 * b) + k for b in range(blocks) for k in range(64)}
    rounds = waves_of(unsure, 4096, 256, 1)
    assert sum(len(w) for w in rounds) == blocks


def test_share():
    share = host_rules.load().redo_share
    for unsure, waves, want in ((0, 4096, 1), (1, 4096, 1), (4096, 4096, 1), (4097, 4096, 2), (262144, 4096, 64),
                                (262145, 4096, 64), (1 << 40, 4096, 64), (1 << 63, 1, 64), (10, 1, 10)):
        assert share(unsure, waves) == want
