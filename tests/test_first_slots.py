"""The slots that the waves of a launch start with (csrc/slot_rule.hpp, run on
the host): each batch of 64 once, neighbouring batches on different blocks."""
import pytest

import host_rules


@pytest.mark.parametrize("blocks,waves", [(1, 1), (1, 16), (3, 4), (40, 4), (256, 4), (256, 12), (209, 12), (256, 16)])
def test_each_batch_once_and_spread(blocks, waves):
    first = host_rules.load().first_slot
    owner = {first(b, v, blocks): b for b in range(blocks) for v in range(waves)}
    assert sorted(owner) == [64 * k for k in range(blocks * waves)]
    if blocks > 1:
        assert all(owner[64 * k] != owner[64 * k + 64] for k in range(blocks * waves - 1))
        # a square of long pixels, 8 batches wide and high in rows of 64 batches
        if blocks * waves >= 4096:
            held = [owner[64 * (64 * y + x)] for y in range(8) for x in range(8)]
            assert max(held.count(b) for b in set(held)) <= 2


def test_slots_past_32_bits():
    assert host_rules.load().first_slot(5, 3, 1 << 26) == 64 * (3 * (1 << 26) + 5)
