"""Host check of the slab-split work items (no GPU): a mirror of ItemIndex and
slab_split (rocket_amd/csrc/gram_items.hpp) must give every (item, slab) of
the triangle exactly once, the split item's slabs in groups of ks, and deal
both kinds of items evenly over the 8 XCDs (id mod 8)."""
import pytest


def items_per_slab(count):
    Q, m = (count + 127) >> 7, (count + 127) >> 8
    return m * (m - 1) // 2 + (m + (m + 4) // 4 if Q % 2 else (6 * m + 7) // 8)


def slab_split(count):
    Q = (count + 127) >> 7
    if Q % 2 == 0:
        return 1
    return {1: 4, 2: 2}.get(((Q >> 1) + 1) & 3, 1)


def ids(T, ks, S, remap):
    Tn, groups = T - (ks > 1), -(-S // ks) if ks > 1 else 0
    up = lambda v: -(-v // 8) * 8 if remap else v   # noqa: E731
    return Tn * up(S) + up(groups)


def at(i, T, ks, S, remap):
    Tn = T - (ks > 1)
    S8 = -(-S // 8) * 8 if remap else S
    if i >= Tn * S8:
        return Tn, (i - Tn * S8) * ks
    return ((i >> 3) % Tn, (i >> 3) // Tn * 8 + (i & 7)) if remap else (i % Tn, i // Tn)


@pytest.mark.parametrize("remap", [True, False])
@pytest.mark.parametrize("S", [1, 3, 8, 37, 64])
@pytest.mark.parametrize("count", [1, 120, 128, 129, 300, 384, 600, 800, 1100, 1400])
def test_every_item_and_slab_once(count, S, remap):
    T, ks = items_per_slab(count), slab_split(count)
    seen, xcds = {}, [0] * 8
    for i in range(ids(T, ks, S, remap)):
        u, s = at(i, T, ks, S, remap)
        if s >= S:
            continue
        split = ks > 1 and u == T - 1
        xcds[i & 7] += 1
        for k in range(ks if split else 1):
            if s + k < S:
                seen[u, s + k] = seen.get((u, s + k), 0) + 1
    assert seen == {(u, s): 1 for u in range(T) for s in range(S)}
    if remap:
        assert max(xcds) - min(xcds) <= T


@pytest.mark.parametrize("count,ks", [(1, 4), (128, 4), (129, 1), (300, 2), (600, 1), (800, 1), (1100, 4), (1300, 2)])
def test_split_fills_the_last_item(count, ks):
    assert slab_split(count) == ks
    m = (count + 127) >> 8
    if ks > 1:  # the one-quarter units of the last item, times ks, are the item's four
        assert ((m + 1) % 4) * ks == 4
