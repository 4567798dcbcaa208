"""
pkv_batch, filled by the backend once per plan: its size is the header's
(checked there at compile time), and the calls that read it refuse a missing
one and an append that cannot be fused.
"""

from __future__ import annotations

import ctypes as C

import pytest

from llm_serving_layer_amd import _native


def test_layout_and_refusals():
    assert C.sizeof(_native.Batch) == 152
    lib = _native.load()
    with pytest.raises(ValueError, match="null batch"):
        _native.check(lib.pkv_append_batch(None, None, None, None, None, None), "append")
    with pytest.raises(ValueError, match="null batch"):
        _native.check(lib.pkv_attend_batch(None, None, None, None, None, 1.0, None, None, None),
                      "attend")
    b = _native.Batch(is_prefill=1, n_heads=4, n_kv_heads=4, head_dim=64, page_size=16)
    with pytest.raises(ValueError, match="decodes only"):
        _native.check(lib.pkv_attend_batch(C.addressof(b), None, None, None, None, 1.0, 16, 16,
                                           None), "attend")
