"""
The two decode kernels (csrc/decode.hip) give one result: a sequence's output
has the same bits whether its batch is small (a workgroup per piece and KV
head) or large (bins of pieces streamed by resident workgroups), and whether
its bin holds one piece or many, with the step's rows appended inside the
launch, at the sizes where the small-batch
kernel can go wrong: one row, page edges, the pages its four waves share, its
chunks of 20 pages and their remainders, every group size, and non-finite
values in the unused rows of a last page.
"""

from __future__ import annotations

import pytest
import torch

from llm_serving_layer_amd import BlockAllocator, SequenceBlocks
from llm_serving_layer_amd.backend import MI355XBackend

from ._util import grow_and_assemble, make_meta, other_stride, takes_pieces

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# history tokens; the step appends one more: whole sequences (17 pages), cut
# ones (with and without a folded tail), and with part_pages=64 chunks of 20
EDGES = [0, 1, 14, 15, 16, 17, 31, 63, 64, 79, 80, 255, 270, 271, 272, 303, 304, 319, 320, 335,
         336, 543, 640, 660, 1023, 1071]


@pytest.mark.parametrize("n_heads, d, dtype, part_pages", [
    (1, 64, torch.float16, 17), (2, 128, torch.float16, 17), (4, 64, torch.bfloat16, 17),
    (8, 128, torch.bfloat16, 17), (16, 64, torch.float16, 17), (16, 128, torch.float16, 64),
    (4, 64, torch.float16, 64)])
def test_small_and_large_batches_give_the_same_bits(n_heads, d, dtype, part_pages):
    print(f"decode pieces heads={n_heads} d={d} {dtype} part_pages={part_pages}", flush=True)
    lens = (EDGES * 12)[:300]          # 300 pieces or more: the streaming kernel
    nb = sum(n // 16 + 1 for n in lens)
    alloc = BlockAllocator(nb, 16)
    seqs = [SequenceBlocks(alloc, seq_id=i) for i in range(len(lens))]
    for s, n in zip(seqs, lens):
        s.append(n)
    g = torch.Generator(device=DEV).manual_seed(3)
    rand = lambda *s: torch.randn(s, generator=g, device=DEV).to(dtype)  # noqa: E731
    big, few = [MI355XBackend(1, nb, 16, 1, n_heads, d, device=DEV, dtype=dtype,
                              part_pages=part_pages) for _ in range(2)]
    k, v = rand(nb, 16, 1, d), rand(nb, 16, 1, d)
    for s, n in zip(seqs, lens):       # rows past the history hold no numbers
        if n % 16:
            k[s.block_ids[-1], n % 16:] = float("nan")
            v[s.block_ids[-1], n % 16:] = float("inf")
    for bk in (big, few):
        bk.k_pool[0].copy_(k)
        bk.v_pool[0].copy_(v)
    q = 2.0 * rand(len(lens), n_heads, d)   # scores wide enough to move the reference
    kn, vn = rand(len(lens), 1, d), rand(len(lens), 1, d)
    meta = grow_and_assemble(seqs, [1] * len(lens), 16, device=DEV)
    big.append_kv(0, kn, vn, meta)
    want = big.attend(q, 0, d ** -0.5, meta)
    assert big._planned.n_work >= 256 and not takes_pieces(big._planned, 1, d)
    assert torch.isfinite(want).all()
    for at in range(0, len(lens), 26):
        part = slice(at, min(at + 26, len(lens)))
        for s in seqs[part]:           # the step's token again, in a batch of its own
            s.num_tokens -= 1
        meta = grow_and_assemble(seqs[part], [1] * len(seqs[part]), 16, device=DEV)
        few.append_kv(0, kn[part], vn[part], meta)
        got = few.attend(q[part], 0, d ** -0.5, meta)
        assert takes_pieces(few._planned, 1, d)
        assert torch.equal(got, want[part]), f"sequences from {at}"
    assert torch.equal(few.k_pool[0].view(torch.int16), big.k_pool[0].view(torch.int16))
    assert torch.equal(few.v_pool[0].view(torch.int16), big.v_pool[0].view(torch.int16))
    big.check_device_errors()
    few.check_device_errors()


@pytest.mark.parametrize("n_decode", [3, 300])
def test_decodes_of_a_mixed_batch_read_and_write_their_token_rows(n_decode):
    """Decodes between prompt chunks (rows 7, 8, ... of q and out, then past a
    second chunk): either kernel gives them the bits they have alone."""
    print(f"mixed rows n_decode={n_decode}", flush=True)
    lens = [0] + (EDGES * 12)[1:n_decode + 1] + [33]
    counts = [7] + [1] * n_decode + [20]
    alloc = BlockAllocator(8192, 16)
    seqs = [SequenceBlocks(alloc, seq_id=i) for i in range(len(lens))]
    for s, n in zip(seqs, lens):
        if n:
            s.append(n)
    bk = MI355XBackend(1, 8192, 16, 1, 4, 64, device=DEV)
    g = torch.Generator(device=DEV).manual_seed(4)
    bk.k_pool[0].normal_(generator=g)
    bk.v_pool[0].normal_(generator=g)
    q = torch.randn(sum(counts), 4, 64, generator=g, device=DEV).half()
    meta = grow_and_assemble(seqs, counts, 16, device=DEV)
    out = bk.attend(q, 0, 0.125, meta)
    assert (bk._planned.dec.n_work >= 256) == (n_decode == 300)
    alone = make_meta(seqs[1:-1], [1] * n_decode, 16, device=DEV)
    assert torch.equal(bk.attend(q[7:7 + n_decode], 0, 0.125, alone), out[7:7 + n_decode])
    bk.check_device_errors()


@pytest.mark.parametrize("scale", [-0.125, 0.0, 1e-50])
def test_a_mixed_batch_takes_q_at_any_address_where_its_chunks_do(scale):
    """A scale that is not positive in fp32 runs the chunks on the generic
    kernel, so a q that starts 2 bytes into its storage is served, decodes
    included; with a positive scale it is refused."""
    print(f"mixed unaligned q scale={scale}", flush=True)
    bk = MI355XBackend(1, 64, 16, 2, 8, 64, device=DEV)
    alloc = BlockAllocator(64, 16)
    seqs = [SequenceBlocks(alloc, seq_id=i) for i in range(3)]
    grow_and_assemble(seqs, [30, 5, 300], 16)
    meta = grow_and_assemble(seqs, [1, 20, 1], 16, device=DEV)
    g = torch.Generator(device=DEV).manual_seed(8)
    bk.k_pool[0].normal_(generator=g)
    bk.v_pool[0].normal_(generator=g)
    q = torch.randn(22 * 8 * 64 + 1, generator=g, device=DEV).half()[1:].view(22, 8, 64)
    assert q.is_contiguous() and q.data_ptr() % 16
    out = bk.attend(q, 0, scale, meta)
    assert bk._planned.dec is not None and torch.isfinite(out).all()
    assert torch.equal(out, bk.attend(q.clone(), 0, scale, meta))
    with pytest.raises(ValueError, match="16-byte aligned"):
        bk.attend(q, 0, 0.125, meta)


@pytest.mark.parametrize("bins", [None, 1, 5])
@pytest.mark.parametrize("n_kv, n_heads, d, dtype, part_pages", [
    (8, 32, 64, torch.float16, 2), (8, 8, 64, torch.bfloat16, 5), (4, 8, 64, torch.bfloat16, 17),
    (1, 16, 64, torch.bfloat16, 3), (2, 16, 64, torch.float16, 64), (1, 1, 128, torch.bfloat16, 3),
    (2, 4, 128, torch.float16, 5), (1, 4, 128, torch.bfloat16, 17), (2, 16, 128, torch.bfloat16, 2),
    (1, 16, 128, torch.float16, 5)])
def test_either_kernel_serves_any_plan_with_the_same_bits(bins, n_kv, n_heads, d, dtype,
                                                          part_pages):
    """One plan through both kernels, with one piece a bin and with many (the
    streaming kernel's item slots refilled, its output and row rings filled and
    flushed, deferred arrivals, merges by the last arriver and by a last piece
    with its own partial in registers), the step's rows appended in the launch.
    Bins of several pieces stream."""
    print(f"one plan, two kernels n_kv={n_kv} heads={n_heads} d={d} {dtype} bins={bins}",
          flush=True)
    lens = [0, 1, 15, 16, 17, 47, 48, 80, 303] + [3 * i for i in range(20)] + [500]
    if bins is None:                   # few enough for a workgroup a piece and head
        lens = lens[1:6] + [90]
    groups = n_kv // min(n_kv, 4)
    alloc = BlockAllocator(256, 16)
    seqs = [SequenceBlocks(alloc, seq_id=i) for i in range(len(lens))]
    for s, n in zip(seqs, lens):
        s.append(n)
    g = torch.Generator(device=DEV).manual_seed(9)
    rand = lambda *s: torch.randn(s, generator=g, device=DEV).to(dtype)  # noqa: E731
    bks = [MI355XBackend(1, 256, 16, n_kv, n_heads, d, device=DEV, dtype=dtype,
                         part_pages=part_pages,
                         decode_workgroups=None if bins is None else bins * groups)
           for _ in range(2)]
    k, v = rand(256, 16, n_kv, d), rand(256, 16, n_kv, d)
    for bk in bks:
        bk.k_pool[0].copy_(k)
        bk.v_pool[0].copy_(v)
    n = len(lens)
    for _ in range(2):
        meta = grow_and_assemble(seqs, [1] * n, 16, device=DEV)
        q, kn, vn = 2.0 * rand(n, n_heads, d), rand(n, n_kv, d), rand(n, n_kv, d)
        outs, kinds = [], []
        for i, bk in enumerate(bks):
            bk.append_kv(0, kn, vn, meta)
            assert bk._pending is not None, "the append rides in the launch"
            p = bk._planned
            if i:
                other_stride(bk, p.n_work // groups)
            kinds.append(takes_pieces(p, n_kv, d))
            outs.append(bk.attend(q, 0, d ** -0.5, meta))
        assert kinds == [bins is None, bins is not None]
        assert torch.isfinite(outs[0]).all() and torch.equal(*outs)
        for a, b in zip(*(bk.k_pool + bk.v_pool for bk in bks)):
            assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    for bk in bks:
        bk.check_device_errors()
