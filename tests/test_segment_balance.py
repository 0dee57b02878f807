"""The segment counts and piece lengths that tops.utils.SegPlan chooses among its candidates
(host plan, CPU): only calls that are split anyway are touched and stay split, every sequence
keeps at least one segment and no segment is empty, and neither the sweep nor the state pass
ends later than with the first candidate by more than what the other one gains."""
import numpy as np
import pytest

from tops.utils import MIN_PIECE_CHUNKS, MIN_SEG_CHUNKS, SegPlan

LAYOUTS = [([39, 15, 14, 37, 25], 8), ([0, 40, 0, 40, 40], 8), ([128], 8), ([128, 128, 128], 8),
           ([512], 1), ([9, 1], 64), ([32] * 5, 16), ([1] * 255 + [400], 4), ([300] * 300, 512),
           ([8, 24, 1, 2, 2, 8, 37], 4)]


def _sizes(ch, m):
    return [[int(n) // int(k) + (i < int(n) % int(k)) for i in range(int(k))] for n, k in zip(ch, m)]


@pytest.mark.parametrize("ch,slots", LAYOUTS, ids=[f"{len(c)}x{max(c)}-{s}" for c, s in LAYOUTS])
def test_balance(ch, slots):
    ch = np.array(ch)
    m = SegPlan.split_counts(ch, slots, None)
    if m.max() <= 1:
        return                                # not split: build() returns before balancing
    b = SegPlan.balance(ch, m, slots)
    assert b.shape == m.shape and b.min() >= 1 and b.max() > 1
    assert np.all(b <= np.maximum(ch, 1))
    s0, s1 = _sizes(ch, m), _sizes(ch, b)
    r = [SegPlan.rounds([x for q in s for x in q], slots) for s in (s0, s1)]
    hand = [[x for q in s for x in q[:-1]] for s in (s0, s1)]
    sub = [max(-(-sum(h) // slots), MIN_PIECE_CHUNKS) if h else 0 for h in hand]
    n = [sum(map(len, s)) + (-(-sum(h) // max(u, 1))) for s, h, u in zip((s0, s1), hand, sub)]
    cost = [r[i] + 2 / 3 * sub[i] + 4 / 3 * n[i] / slots for i in (0, 1)]
    assert cost[1] <= cost[0]
    assert r[1] >= max(-(-int(ch.sum()) // slots), 1)
    if hand[1]:
        x = SegPlan.balance_pieces(hand[1], sub[1], slots)
        assert sub[1] <= x <= 2 * sub[1]
        span = [SegPlan.rounds([hi - lo for n in hand[1] for lo, hi in SegPlan._cut(0, n, y)], slots)
                for y in (sub[1], x)]
        assert span[1] <= span[0]


def test_rounds():
    assert SegPlan.rounds([5], 8) == 5 and SegPlan.rounds([3, 3, 3], 2) == 6
    assert SegPlan.rounds([7, 5, 4, 4, 2], 2) == 11 and SegPlan.rounds([0, 0], 1) == 0
    assert MIN_SEG_CHUNKS >= MIN_PIECE_CHUNKS
