"""CPU model of the partition's present rules (partition.hip), against numpy's
stable argsort: a merged call counts, in its cell's list of movers (in any
order), those with a smaller slot, or bisects the list where it is in slot
order; a cold call sorts by the keys' high digit, tile by tile, and then cell by
cell within a bucket."""
import numpy as np
import pytest

TILE, CELLS = 4096, 1024


def merged(k, h, ncells, rng, heavy):
    n = len(k)
    stay = k == h
    S = np.concatenate([[0], np.cumsum(stay)])[:n]
    stayers, movers = (np.bincount(k[m], minlength=ncells + 1) for m in (stay, ~stay))
    start = np.concatenate([[0], np.cumsum(stayers + movers)])[:-1]
    before = np.concatenate([[0], np.cumsum(stayers)])[:-1]
    part = {c: np.nonzero(~stay & (k == c))[0] for c in np.nonzero(movers)[0]}
    order = np.full(n, -1)
    for i in range(n):
        c = k[i]
        mine = part.get(c, np.zeros(0, np.int64))
        if len(mine) > heavy:
            rank = int(np.searchsorted(mine, i))
        else:
            rank = int((rng.permutation(mine) < i).sum())  # the list comes in any order
        own = S[i] - before[c]
        order[start[c] + rank + (own if stay[i] else min(max(own, 0), stayers[c]))] = i
    return order


def cold(k, ncells, buckets, prefix=True):
    n, shift = len(k), 0
    while (ncells >> shift) >= buckets:
        shift += 1
    b = k >> shift
    hist = np.stack([np.bincount(b[t:t + TILE], minlength=buckets) for t in range(0, n, TILE)])
    first = np.concatenate([[0], np.cumsum(hist.sum(0))])
    slots = np.full(n, -1)
    for t in range(hist.shape[0]):  # every tile adds up the tiles before it
        at = first[:-1] + (hist[:t].sum(0) if prefix else 0)
        for i in range(t * TILE, min(n, (t + 1) * TILE)):
            slots[at[b[i]]] = i
            at[b[i]] += 1
    order, placed = np.full(n, -1), None
    for q in range((ncells >> shift) + 1):
        mine, placed = slots[first[q]:first[q + 1]], first[q]
        end = min((q + 1) << shift, ncells + 1)
        for r0 in range(q << shift, end, CELLS):
            m = min(end - r0, CELLS)
            here = mine[(k[mine] >= r0) & (k[mine] < r0 + m)]
            nxt = placed + np.concatenate([[0], np.cumsum(np.bincount(k[here] - r0, minlength=m))])
            placed = nxt[-1]
            for i in here:
                order[nxt[k[i] - r0]] = i
                nxt[k[i] - r0] += 1
    return order


@pytest.mark.parametrize("ncells", [1, 7, 300, 5000, 300000])
def test_cold_rule_is_the_stable_sort(ncells):
    rng = np.random.default_rng(ncells)
    for n, buckets in ((1, 64), (4096, 64), (4097, 1024), (9001, 73)):
        for k in (rng.integers(0, ncells + 1, n), np.full(n, ncells), rng.integers(0, 2, n)):
            np.testing.assert_array_equal(cold(k, ncells, buckets), np.argsort(k, kind="stable"))


@pytest.mark.parametrize("heavy", [0, 3, 1000])
def test_merge_rule_is_the_stable_sort(heavy):
    rng = np.random.default_rng(heavy)
    for ncells in (1, 9, 400):
        for n in (1, 60, 700):
            h = np.sort(rng.integers(0, ncells + 1, n))
            k = np.where(rng.random(n) < 0.3, rng.integers(0, ncells + 1, n), h)
            np.testing.assert_array_equal(merged(k, h, ncells, rng, heavy), np.argsort(k, kind="stable"))


def test_a_planted_mistake_fails():
    """A tile that does not add up the tiles before it breaks the order."""
    k = np.random.default_rng(5).integers(0, 40, 2 * TILE)
    want = np.argsort(k, kind="stable")
    assert np.array_equal(cold(k, 40, 64), want) and not np.array_equal(cold(k, 40, 64, prefix=False), want)
