"""The native search over segment counts and piece lengths (tops_segment_balance,
tops_piece_balance, tops_balance_rounds; host, CPU): the same choice as the search stated here
in Python, and a small share of the plan that a call with new boundaries builds before its
first launch."""
import heapq
import time

import numpy as np
import pytest

from tops import utils as U
from tops.utils import MIN_PIECE_CHUNKS, MIN_SEG_CHUNKS, SegPlan


def _rounds(sizes, slots):
    if len(sizes) <= slots:
        return max(sizes)
    sizes = sorted(sizes, reverse=True)
    load = sizes[slots - 1::-1]
    for x in sizes[slots:]:
        heapq.heapreplace(load, load[0] + x)
    return max(load)


def _parts(n, k):
    base, rem = divmod(n, k)
    return [base + 1] * rem + [base] * (k - rem)


def _pieces(handing, sub, slots):
    best = None
    for x in range(sub, 2 * sub + 1, max(sub // 4, 1)):
        parts = [y for n in handing for y in _parts(n, -(-n // x))]
        span = _rounds(parts, slots)
        if best is None or span < best[0]:
            best = span, x
        if len(parts) <= slots:
            break
    return best[1]


def _counts(ch, c0, slots):
    def cost(c):
        seg = [_parts(n, k) for n, k in zip(ch, c)]
        flat = [x for s in seg for x in s]
        hand = sum(sum(s[:-1]) for s in seg)
        sub = max(-(-hand // slots), MIN_PIECE_CHUNKS) if hand else 0
        states = len(flat) + (-(-hand // sub) if hand else 0)
        span = _rounds(flat, slots)
        return span + 2 / 3 * sub + 4 / 3 * states / slots, span

    t0 = max(-(-sum(ch) // slots), MIN_SEG_CHUNKS)
    best, (low, span) = c0, cost(c0)
    if span > 1.1 * t0:
        seen = [c0]
        for t in range(t0, 2 * t0 + 1, max(t0 // 8, 1)):
            c = [max(-(-n // t), 1) for n in ch]
            if c in seen or max(c) <= 1:
                continue
            seen.append(c)
            e = cost(c)[0]
            if e < low:
                best, low = c, e
    return best


@pytest.mark.parametrize("seed", range(8))
def test_native_search_makes_the_stated_choice(seed):
    rng = np.random.default_rng(seed)
    for _ in range(40):
        n = int(rng.integers(1, 40))
        slots = int(rng.choice([1, 2, 3, 4, 8, 16, 32, 64, 128, 256]))
        ch = rng.integers(0, int(rng.choice([4, 40, 400])), n)
        ch[rng.integers(n)] += 9                     # (one sequence has chunks)
        m = SegPlan.split_counts(ch, slots, None)
        assert SegPlan.balance(ch, m, slots).tolist() == _counts(ch.tolist(), m.tolist(), slots)
        hand = [int(x) for x in ch if x > 0]
        assert SegPlan.rounds(hand, slots) == _rounds(hand, slots)
        sub = max(-(-sum(hand) // slots), MIN_PIECE_CHUNKS)
        assert SegPlan.balance_pieces(hand, sub, slots) == _pieces(hand, sub, slots)


def test_native_search_rejects_bad_arguments():
    for args in (([], 4), ([3], 0)):
        with pytest.raises(ValueError):
            SegPlan.rounds(*args)
    for args in (([0, 4], 4, 4), ([4], 0, 4), ([], 4, 4)):
        with pytest.raises(ValueError):
            SegPlan.balance_pieces(*args)
    for ch, m in (([-1, 4], [1, 1]), ([4], [0])):
        with pytest.raises(ValueError):
            SegPlan.balance(np.array(ch), np.array(m), 4)


@pytest.mark.parametrize("n,T,H,V", [(16, 16384, 4, 128), (200, 65536, 2, 64), (100, 131072, 2, 128)])
def test_search_is_a_small_share_of_the_plan(n, T, H, V, monkeypatch):
    """Boundaries are new on most calls of a loader or a server: the search may take a fifth of
    the plan's time (measured 1 to 5 %; 14 to 42 % when it ran in Python)."""
    monkeypatch.setattr(U, "_device_cus", lambda device: 256)
    rng = np.random.default_rng(n)
    cu = np.array([0] + sorted(rng.choice(np.arange(1, T), n - 1, replace=False).tolist()) + [T])
    plan = U.ChunkPlan(1, T, cu, "cpu")
    spent = [0.0]

    def timed(f):
        def g(*a):
            t = time.perf_counter()
            r = f(*a)
            spent[0] += time.perf_counter() - t
            return r
        return staticmethod(g)
    monkeypatch.setattr(SegPlan, "balance", timed(SegPlan.balance))
    monkeypatch.setattr(SegPlan, "balance_pieces", timed(SegPlan.balance_pieces))
    build, search = [], []
    for _ in range(15):
        spent[0] = 0.0
        t = time.perf_counter()
        assert SegPlan.build(plan, H, V) is not None
        build.append(time.perf_counter() - t)
        search.append(spent[0])
    assert 0 < min(search) < 0.2 * min(build)
