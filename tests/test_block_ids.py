"""
The id lists of copy_blocks: any iterable of integers, as before they became
arrays, and the same refusals.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from llm_serving_layer_amd.backend import MI355XBackend, block_ids


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
