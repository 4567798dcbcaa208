"""
The matrix-core prefill's LDS ring starts with whatever the last kernel left
there, and pages past a sequence's end load nothing: neither may reach a
result. A prefill over pools of NaN runs first on every compute unit, then
chunks at the sizes where tiles are partly or wholly empty, against the oracle.
"""

from __future__ import annotations

import pytest
import torch

from llm_serving_layer_amd import BlockAllocator, SequenceBlocks
from llm_serving_layer_amd.backend import MI355XBackend

from ._util import grow_and_assemble
from .test_gpu_attention import Pair, check

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("d, dtype", [(64, torch.float16), (128, torch.bfloat16)])
def test_stale_lds_and_pages_past_the_end_do_not_reach_a_result(d, dtype):
    print(f"prefill ring d={d} {dtype}", flush=True)
    nan = MI355XBackend(1, 64, 16, 8, 32, d, device=DEV, dtype=dtype)
    nan.k_pool[0].fill_(float("nan"))
    nan.v_pool[0].fill_(float("nan"))
    s = SequenceBlocks(BlockAllocator(64, 16), seq_id=0)
    nan_meta = grow_and_assemble([s], [1000], 16, device=DEV)
    nan_q = torch.zeros(1000, 32, d, device=DEV, dtype=dtype)
    p = Pair(1, 64, 16, 8, 32, d, dtype=dtype)
    p.poison(1)
    alloc = BlockAllocator(64, 16)
    seqs = [SequenceBlocks(alloc, seq_id=i) for i in range(6)]
    tol, rtol = (2e-3, 1e-2) if dtype == torch.float16 else (1.6e-2, 8e-2)
    for seed, counts in enumerate([[2, 15, 16, 17, 33, 100], [3, 1, 2, 31, 63, 28]]):
        meta = grow_and_assemble(seqs, counts, 16)
        for _ in range(2):
            nan.attend(nan_q, 0, 0.125, nan_meta)
        res = p.step(meta, seed)
        assert torch.isfinite(res[0][1]).all()
        check(res, f"{counts}", tol, rtol)
