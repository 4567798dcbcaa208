"""
The fp32 matrix-core attention kernel (csrc/attention_f32.hip) at the sizes
where it can go wrong: page and wave-split edges (its eight waves take every
eighth page), row tiles of 16 and 32 rows and their remainders, group sizes
that do not divide a tile, long histories, non-finite values behind the
causal mask, and the bitwise equality of a token decoded and prefilled.

Tolerance against the fp32 oracle (values N(0, 1), scores of a few units):
both sides sum at most 2048 products p * v with relative rounding 2^-24 a
term and probabilities off by a few 2^-24 times the score, so outputs below
5 in size differ by at most about 1e-5.
"""

from __future__ import annotations

import pytest
import torch

from llm_serving_layer_amd import BlockAllocator, SequenceBlocks
from llm_serving_layer_amd.backend import MI355XBackend

from ._util import fragmented_allocator, grow_and_assemble, make_meta
from .test_gpu_attention import Pair, check

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ATOL, RTOL = 1e-5, 1e-3


@pytest.mark.parametrize("geom", [(8, 32, 64), (2, 14, 64), (1, 1, 64), (1, 40, 64), (2, 32, 128),
                                  (2, 6, 128)])
def test_prefill_mixed_and_decode_vs_oracle(geom):
    n_kv, n_heads, d = geom
    print(f"f32 geom={geom}", flush=True)
    p = Pair(2, 512, 16, n_kv, n_heads, d, dtype=torch.float32)
    p.poison(1)
    alloc, _keep = fragmented_allocator(512, 16)
    hist = [1, 15, 16, 17, 127, 128, 129, 300, 1000]
    seqs = [SequenceBlocks(alloc, seq_id=i) for i in range(len(hist))]
    check(p.step(grow_and_assemble(seqs, hist, 16), 1), "prompts", ATOL, RTOL)
    check(p.step(grow_and_assemble(seqs, [1, 2, 1, 8, 31, 1, 33, 65, 1], 16), 2), "mixed", ATOL,
          RTOL)
    check(p.step(grow_and_assemble(seqs, [1] * len(hist), 16), 3), "decode", ATOL, RTOL)
    check(p.step(grow_and_assemble(seqs, [1] * len(hist), 16), 4, scale=-0.1), "negative scale",
          ATOL, RTOL)


@pytest.mark.parametrize("geom", [(8, 32, 64), (2, 6, 128)])
def test_a_token_has_the_same_bits_decoded_prefilled_alone_or_batched(geom):
    n_kv, n_heads, d = geom
    print(f"f32 bits geom={geom}", flush=True)
    bk = MI355XBackend(1, 128, 16, n_kv, n_heads, d, device=DEV, dtype=torch.float32)
    a = BlockAllocator(128, 16)
    g = torch.Generator(device=DEV).manual_seed(5)
    lens = [270, 45]
    seqs = [SequenceBlocks(a, seq_id=i) for i in range(2)]
    meta = grow_and_assemble(seqs, lens, 16, device=DEV)
    k, v = [torch.randn(sum(lens), n_kv, d, generator=g, device=DEV) for _ in range(2)]
    q = torch.randn(sum(lens), n_heads, d, generator=g, device=DEV)
    bk.append_kv(0, k, v, meta)
    whole = bk.attend(q, 0, 0.125, meta)
    assert torch.equal(whole[:270], bk.attend(q[:270], 0, 0.125, make_meta(seqs[:1], [270], 16,
                                                                           device=DEV)))
    tail = bk.attend(q[250:270], 0, 0.125, make_meta(seqs[:1], [20], 16, device=DEV))
    assert torch.equal(tail, whole[250:270]), "a later tile"
    last = torch.stack([q[269], q[314]])
    one = bk.attend(last, 0, 0.125, make_meta(seqs, [1, 1], 16, device=DEV))
    assert torch.equal(one, torch.stack([whole[269], whole[314]])), "decode"


def test_values_behind_the_causal_mask_do_not_reach_earlier_rows():
    """An infinite or NaN V (and K) row is seen only by the rows at or past
    its position, whose outputs are not finite; the others keep theirs."""
    print("f32 non-finite values", flush=True)
    bk = MI355XBackend(1, 16, 16, 2, 8, 64, device=DEV, dtype=torch.float32)
    g = torch.Generator(device=DEV).manual_seed(6)
    s = [SequenceBlocks(BlockAllocator(16, 16), seq_id=0)]
    meta = grow_and_assemble(s, [40], 16, device=DEV)
    k, v = [torch.randn(40, 2, 64, generator=g, device=DEV) for _ in range(2)]
    q = torch.randn(40, 8, 64, generator=g, device=DEV)
    bk.append_kv(0, k, v, meta)
    base = bk.attend(q, 0, 0.125, meta)
    for bad in (float("inf"), float("nan")):
        v2, k2 = v.clone(), k.clone()
        v2[37], k2[39] = bad, bad
        bk.append_kv(0, k2, v2, meta)
        out = bk.attend(q, 0, 0.125, meta)
        assert torch.allclose(out[:37], base[:37], atol=1e-6, rtol=1e-6)
        assert not torch.isfinite(out[37:]).any()


def test_kernel_reads_at_16_bytes_only_when_aligned():
    """A contiguous q that starts 4 bytes into its storage still gives the
    result (the generic kernel serves it)."""
    print("f32 unaligned q", flush=True)
    bk = MI355XBackend(1, 16, 16, 2, 8, 64, device=DEV, dtype=torch.float32)
    g = torch.Generator(device=DEV).manual_seed(7)
    s = [SequenceBlocks(BlockAllocator(16, 16), seq_id=0)]
    meta = grow_and_assemble(s, [33], 16, device=DEV)
    k, v = [torch.randn(33, 2, 64, generator=g, device=DEV) for _ in range(2)]
    buf = torch.randn(33 * 8 * 64 + 1, generator=g, device=DEV)
    q = buf[1:].view(33, 8, 64)
    assert q.is_contiguous() and q.data_ptr() % 16
    bk.append_kv(0, k, v, meta)
    a, b = bk.attend(q, 0, 0.125, meta), bk.attend(q.clone(), 0, 0.125, meta)
    assert torch.allclose(a, b, atol=ATOL, rtol=RTOL)
