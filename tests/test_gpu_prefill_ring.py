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

from ._util import grow_and_assemble, make_meta
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


@pytest.mark.parametrize("d, dtype", [(64, torch.float16), (128, torch.bfloat16)])
@pytest.mark.parametrize("n_kv, n_heads", [(8, 32), (1, 4)])
def test_rows_past_the_end_of_a_sequence_never_reach_a_result(d, dtype, n_kv, n_heads):
    """Every length of a last page, beside a decode and without one: a pool
    whose rows past each sequence's end hold NaN (K) and infinity (V), as do
    all blocks that no sequence has, gives the bits of one that holds zeros
    there."""
    print(f"prefill rows past the end d={d} {dtype} n_kv={n_kv}", flush=True)
    lens = [32 * (i % 3) + i for i in range(1, 17)] + [5]
    alloc = BlockAllocator(128, 16)
    alloc.allocate(128)
    alloc.free([(37 * i) % 128 for i in range(127, -1, -1)])
    seqs = [SequenceBlocks(alloc, seq_id=i) for i in range(len(lens))]
    for s, n in zip(seqs, lens):
        s.append(n)
    g = torch.Generator(device=DEV).manual_seed(d + n_kv)
    k, v = [torch.zeros(128, 16, n_kv, d, device=DEV, dtype=dtype) for _ in range(2)]
    live = torch.zeros(128, 16, dtype=torch.bool, device=DEV)
    for s, n in zip(seqs, lens):
        for j, b in enumerate(s.block_ids):
            live[b, :n - 16 * j] = True
    for x in (k, v):
        x[live] = torch.randn(int(live.sum()), n_kv, d, generator=g, device=DEV).to(dtype)
    bk = MI355XBackend(1, 128, 16, n_kv, n_heads, d, device=DEV, dtype=dtype)
    chunks = [max(1, n // 2) for n in lens[:-1]]
    for label, part, counts in (("prefill", seqs[1:-1], chunks[1:]),
                                ("whole prompts", seqs[1:-1], lens[1:-1]),
                                ("mixed", seqs, chunks + [1])):
        meta = make_meta(part, counts, 16, device=DEV)
        q = torch.randn(sum(counts), n_heads, d, generator=g, device=DEV).to(dtype)
        outs = []
        for kx, vx in ((0.0, 0.0), (float("nan"), float("inf"))):
            k[~live], v[~live] = kx, vx
            bk.k_pool[0].copy_(k)
            bk.v_pool[0].copy_(v)
            outs.append(bk.attend(q, 0, 0.125, meta))
        assert torch.isfinite(outs[0]).all(), label
        assert torch.equal(outs[0], outs[1]), label
    bk.check_device_errors()
