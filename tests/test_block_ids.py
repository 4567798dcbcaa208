"""
The id lists of copy_blocks: any iterable of integers, one set of refusals
whatever the length of the list and the size of the pool (short and long
lists, small and large pools are checked in different ways), and a cost that
does not grow with the pool.
"""

from __future__ import annotations

import random
import tracemalloc

import numpy as np
import pytest
import torch

from llm_serving_layer_amd.backend import SHORT_COPY, MI355XBackend, block_ids, copy_ids


@pytest.mark.parametrize("ids, want", [
    ([3, 1, 2], [3, 1, 2]), ((), []), (range(4), [0, 1, 2, 3]), (iter([5, 6]), [5, 6]),
    (np.array([7, 8], np.int32), [7, 8]), (torch.tensor([1, 2]), [1, 2]),
    ([np.int64(4), 5], [4, 5]), ([True, 2], [1, 2]), ([2.0, 3.7], [2, 3]), (["9"], [9]),
    ([-1, 2**63, -2**70], [-1, 2**63 - 1, -1])])
def test_any_iterable_of_integers(ids, want):
    got = block_ids(ids)
    assert got.dtype == np.int64 and got.tolist() == want


@pytest.mark.parametrize("src, dst, error, text", [
    ([1], [2, 3], ValueError, "1 sources but 2 destinations"),
    ([0, 8], [1, 2], IndexError, r"copy_block\(8 -> 2\) outside \[0, 8\)"),
    ([0, 1], [3, -1], IndexError, r"copy_block\(1 -> -1\) outside \[0, 8\)"),
    ([0, 1], [3, 3], ValueError, "distinct destinations"),
    ([0, 3], [3, 4], ValueError, "distinct destinations"),
    (["x"], [1], ValueError, "invalid literal"), ([None], [1], TypeError, "int()")])
def test_refused_before_anything_is_launched(src, dst, error, text):
    bk = object.__new__(MI355XBackend)   # no pool, no device: the checks come first
    bk.num_blocks = 8
    with pytest.raises(error, match=text):
        bk.copy_blocks(src, dst)
    bk.copy_blocks([], [])
    bk.copy_blocks([4, 4], [4, 4])       # copies onto themselves: nothing to do


def _by_pairs(src, dst, num_blocks):
    """The contract, pair by pair."""
    if len(src) != len(dst):
        return ValueError
    if any(not 0 <= i < num_blocks for i in src + dst):
        return IndexError
    pairs = [(s, d) for s, d in zip(src, dst) if s != d]
    to = [d for _, d in pairs]
    if len(set(to)) != len(to) or set(to) & {s for s, _ in pairs}:
        return ValueError
    return [s for s, _ in pairs] + to


@pytest.mark.parametrize("n", [0, 1, 2, SHORT_COPY, SHORT_COPY + 1, 64, 700])
@pytest.mark.parametrize("num_blocks", [1, 3, 100, 1400, 256 * 64, 256 * 64 + 1, 1 << 20])
def test_every_way_of_checking_gives_the_same_answer(n, num_blocks):
    rng = random.Random(n * 7 + num_blocks)
    ids = (rng.sample(range(num_blocks), 2 * n) if 2 * n <= num_blocks
           else [rng.randrange(num_blocks) for _ in range(2 * n)])
    src, dst = ids[:n], ids[n:]
    lists = [(src, dst), (src, dst + [0]), (src, src)]
    for at in {0, n // 2, n - 1} if n else ():
        other = (at + 1) % n
        for bad in (-1, num_blocks, 2**62, -2**70):
            lists += [(src[:at] + [bad] + src[at + 1:], dst), (src, dst[:at] + [bad] + dst[at + 1:])]
        lists += [(src, dst[:at] + [dst[other]] + dst[at + 1:]),    # twice a destination
                  (src, dst[:at] + [src[other]] + dst[at + 1:]),    # also a source
                  (src, dst[:at] + [src[at]] + dst[at + 1:]),       # onto itself
                  (src[:at] + [src[other]] + src[at + 1:], dst)]    # a source twice
    for s, d in lists:
        want = _by_pairs(s, d, num_blocks)
        if isinstance(want, list):
            got = copy_ids(s, d, num_blocks)
            assert got.dtype == torch.int32 and got.tolist() == want
        else:
            with pytest.raises(want):
                copy_ids(s, d, num_blocks)


@pytest.mark.parametrize("n", [1, SHORT_COPY, SHORT_COPY + 1, 500])
def test_nothing_of_the_pools_size_is_made_for_a_few_blocks(n):
    num_blocks = 1 << 24
    src, dst = list(range(n)), list(range(n, 2 * n))
    bk = object.__new__(MI355XBackend)
    bk.num_blocks = num_blocks

    class Reached(Exception):
        pass

    def stop():
        raise Reached
    bk._flush = stop                      # the checks are done
    tracemalloc.start()
    try:
        with pytest.raises(Reached):
            bk.copy_blocks(src, dst)
        assert tracemalloc.get_traced_memory()[1] < num_blocks // 16
    finally:
        tracemalloc.stop()
