"""CPU restatement of the tile schedule's partition (csrc/tiles.hpp): the axis
of rows and segment ends, the 64-probe search, the rows of a tile, and the
chain of partials of a segment that crosses tiles. Over random lengths, tile
sizes and end weights every row is folded exactly once into its segment, every
segment is written exactly once, and a chain is exactly the tiles that hold the
segment's rows, in order. Offsets that break the contract (not ascending, out
of range) stay inside the rows, segments and partials."""
import numpy as np
import pytest

WAVE = 64


def search(offsets, weight, v):
    """First segment whose end position is at least v (64 probes per step)."""
    b = len(offsets) - 1
    lo, hi, steps = 0, b, 0
    while lo < hi:
        step = -(-(hi - lo) // WAVE)
        found = WAVE
        for lane in range(WAVE):
            i = lo + lane * step
            assert i >= hi or 0 <= i < b
            if i >= hi or offsets[i + 1] + weight * i >= v:
                found = lane
                break
        top = lo + found * step
        below = lo + (found - 1) * step + 1 if found else lo
        hi, lo = min(hi, top), min(below, min(hi, top))
        steps += 1
        assert steps < 64
    return lo


def row_at(offsets, n, weight, v, s):
    b = len(offsets) - 1
    a, e = offsets[s], offsets[s + 1] if s < b else n
    r = max(min(v - weight * s, e), a)
    return min(max(r, 0), n)


def tile(offsets, n, weight, items, w):
    """(s0, s1, r0, r1, head open, first tile of the head's chain)."""
    b = len(offsets) - 1
    v0 = w * items
    v1 = min(v0 + items, n + weight * b)
    s0, s1 = search(offsets, weight, v0), search(offsets, weight, v1)
    r0, r1 = row_at(offsets, n, weight, v0, s0), row_at(offsets, n, weight, v1, s1)
    r1 = min(max(r1, r0), r0 + items)
    begin = max(int(offsets[s0]), 0) if s0 < b else r0
    first = (begin + weight * s0) // items
    return s0, s1, r0, r1, w > 0 and begin < r0, min(first, w)


def lengths_of(rng, kind, b):
    if kind == "mixed":
        return rng.integers(0, 40, b) * (rng.random(b) < 0.7)
    if kind == "long":
        return np.where(rng.random(b) < 0.2, rng.integers(200, 900, b), rng.integers(0, 3, b))
    if kind == "one":
        lengths = np.zeros(b, dtype=np.int64)
        lengths[rng.integers(b)] = 1500
        return lengths
    return np.zeros(b, dtype=np.int64)


@pytest.mark.parametrize("kind", ["mixed", "long", "one", "empty"])
def test_every_row_and_segment_once(kind):
    rng = np.random.default_rng(["mixed", "long", "one", "empty"].index(kind))
    for b, weight, items in ((1, 1, 7), (3, 4, 5), (70, 1, 64), (70, 3, 17), (200, 16, 33), (4200, 2, 400)):
        lengths = lengths_of(rng, kind, b).astype(np.int64)
        offsets = np.concatenate([[0], np.cumsum(lengths)])
        n = int(offsets[-1])
        tiles = -(-(n + weight * b) // items)
        parts = {}                 # (tile, which) -> rows folded into that partial
        written = {}               # segment -> rows of its result
        last_row = 0
        for w in range(tiles):
            s0, s1, r0, r1, head, first = tile(offsets, n, weight, items, w)
            assert r0 == last_row and 0 <= s0 <= s1 <= b and r1 - r0 <= items
            last_row = r1
            pos = r0
            for s in range(s0, s1):
                rows = list(range(pos, int(offsets[s + 1])))
                assert offsets[s + 1] <= r1
                pos = int(offsets[s + 1])
                if s == s0 and head:
                    chain = []
                    for t in range(first, w):
                        chain += parts.pop((t, s))
                    rows = chain + rows
                assert s not in written
                written[s] = rows
            if s1 < b and (pos < r1 or (s0 == s1 and head)):
                parts[(w, s1)] = list(range(pos, r1))
                assert parts[(w, s1)]
        assert last_row == n and not parts
        assert sorted(written) == list(range(b))
        for s, rows in written.items():
            assert rows == list(range(offsets[s], offsets[s + 1]))


def test_offsets_that_break_the_contract_stay_in_bounds():
    rng = np.random.default_rng(5)
    for _ in range(300):
        b, n = int(rng.integers(1, 150)), int(rng.integers(0, 400))
        offsets = rng.integers(-50, n + 50, b + 1)
        weight, items = int(rng.integers(1, 9)), int(rng.integers(1, 70))
        for w in range(-(-(n + weight * b) // items)):
            s0, s1, r0, r1, head, first = tile(offsets, n, weight, items, w)
            assert 0 <= s0 <= b and 0 <= s1 <= b and 0 <= r0 <= r1 <= n and r1 - r0 <= items
            assert 0 <= first <= w
