"""
pkv_batch, filled by the backend once per plan: its size is the header's
(checked there at compile time), and the calls that read it refuse a missing
one, an append that cannot be fused, and a mixed batch whose geometry has no
decode kernel that reads a plan.
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


@pytest.mark.parametrize("n_heads, n_kv, d, page, dtype", [
    (4, 4, 64, 16, _native.DTYPE_F32), (4, 4, 80, 16, _native.DTYPE_F16),
    (12, 4, 64, 16, _native.DTYPE_BF16), (4, 4, 64, 8, _native.DTYPE_F16)])
def test_a_mixed_batch_needs_the_decode_kernel_that_reads_its_plan(n_heads, n_kv, d, page, dtype):
    """The other kernels take sequence i's output for row i, which a mixed
    batch's decodes are not: refused before anything is launched."""
    lib = _native.load()
    assert not lib.pkv_decode_fast_path(n_heads, n_kv, d, page, dtype, 17)
    with pytest.raises(ValueError, match="fast decode path"):
        _native.check(lib.pkv_attend_mixed(
            16, 16, 16, 16, 8, None, None, None, None, None, 2, 3, n_heads, n_kv, d, page, 0.125,
            dtype, None, 1, 32, None, 1, 1, 0, 68, None, 0, None, None), "attend")
    b = _native.Batch(num_blocks=8, n_seqs=2, n_tokens=3, is_prefill=1, n_heads=n_heads,
                      n_kv_heads=n_kv, head_dim=d, page_size=page, dtype=dtype, n_tiles=1,
                      q_tile=32, n_decodes=1, n_work=1, plan_stride=68)
    with pytest.raises(ValueError, match="fast decode path"):
        _native.check(lib.pkv_attend_batch(C.addressof(b), 16, 16, 16, 16, 0.125, None, None,
                                           None), "attend")
