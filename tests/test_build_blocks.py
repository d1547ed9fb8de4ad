"""Grouped launches of the list build: a table of prefix sums, in which a list
without workgroups in a launch repeats its neighbour's entry, and a grid rounded
up to the 8 XCDs.  Every workgroup below the total belongs to exactly one list,
as one of that list's own workgroups; those above it belong to none."""
import numpy as np


def find_replica(block0, lb):
    """tm_internal.h, find_replica"""
    lo, hi = 0, len(block0) - 2
    while lo < hi:
        mid = (lo + hi + 1) >> 1
        if block0[mid] <= lb:
            lo = mid
        else:
            hi = mid - 1
    return lo


def test_every_workgroup_is_one_of_its_list():
    rng = np.random.default_rng(1)
    for _ in range(2000):
        count = rng.integers(0, 9, rng.integers(1, 9)) * rng.integers(0, 2)
        count[rng.random(len(count)) < 0.4] = 0
        block0 = np.concatenate([[0], np.cumsum(count)])
        grid = -(-block0[-1] // 8) * 8
        seen = np.zeros(len(count), dtype=int)
        for b in range(grid):
            lb = (b % 8) * (grid // 8) + b // 8    # logical_block
            if lb >= block0[-1]:
                continue
            r = find_replica(block0, lb)
            assert 0 <= lb - block0[r] < count[r]
            seen[r] += 1
        assert np.array_equal(seen, count)
