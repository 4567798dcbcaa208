"""
KV append at the row lengths where its thread mapping changes: one vector a
row, a length that is no power of two, whole waves, more vectors than a
workgroup's threads, and rows that only 4- and 2-byte accesses divide; with
token counts around a workgroup's share and a slot outside the pool.
"""

from __future__ import annotations

import pytest
import torch

from llm_serving_layer_amd import BlockAllocator, SequenceBlocks
from llm_serving_layer_amd.backend import MI355XBackend

from ._util import grow_and_assemble

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n_kv, d, dtype", [
    (1, 8, torch.float16), (1, 24, torch.float16), (8, 64, torch.bfloat16),
    (16, 256, torch.float32), (1, 2, torch.float16), (1, 3, torch.float16)])
@pytest.mark.parametrize("tokens", [2, 129, 300])
def test_rows_land_in_their_slots_and_nowhere_else(n_kv, d, dtype, tokens):
    print(f"append rows n_kv={n_kv} d={d} {dtype} tokens={tokens}", flush=True)
    bk = MI355XBackend(1, 32, 16, n_kv, n_kv, d, device=DEV, dtype=dtype)
    alloc = BlockAllocator(32, 16)
    alloc.allocate(32)
    alloc.free([(7 * i) % 32 for i in range(32)])
    seq = SequenceBlocks(alloc, seq_id=0)
    meta = grow_and_assemble([seq], [tokens], 16, device=DEV)
    g = torch.Generator(device=DEV).manual_seed(tokens)
    k, v, kp, vp = [torch.randn(n, n_kv, d, generator=g, device=DEV).to(dtype)
                    for n in (tokens, tokens, 512, 512)]
    bk.k_pool[0].copy_(kp.view_as(bk.k_pool[0]))
    bk.v_pool[0].copy_(vp.view_as(bk.v_pool[0]))
    bk.append_kv(0, k, v, meta)
    slots = meta.slot_mapping.long()
    kp[slots], vp[slots] = k, v
    assert torch.equal(bk.k_pool[0].view_as(kp), kp) and torch.equal(bk.v_pool[0].view_as(vp), vp)
    bk.check_device_errors()
    bad = meta.slot_mapping.clone()     # the last row's slot: outside the pool
    bad[-1] = 512
    bk._launch_append(0, -k, -v, bad, torch.cuda.current_stream().cuda_stream)
    kp[slots[:-1]], vp[slots[:-1]] = -k[:-1], -v[:-1]
    assert torch.equal(bk.k_pool[0].view_as(kp), kp) and torch.equal(bk.v_pool[0].view_as(vp), vp)
    with pytest.raises(IndexError, match="slot_mapping"):
        bk.check_device_errors()
