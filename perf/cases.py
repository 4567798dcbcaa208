"""
Performance cases of the paged-KV framework: the work a serving engine has it
do, through its public entry points (``MI355XBackend.append_kv`` / ``attend``
/ ``copy_blocks``, ``build_batch_meta``, ``greedy``, ``KVSwapSpace``), and the
same work in 64 bits with plain torch.

Four kinds of case:

* ``attend``  one engine step: per layer the KV append of the step's tokens and
  the attention over every sequence's history. ``n_decode`` sequences bring
  one token each, ``n_chunk`` sequences a prompt chunk behind a history (their
  own, or one paged prefix that all of them share). With ``describe`` the
  batch's metadata is built in the pass too, as a scheduler does each step.
* ``copy``    copy-on-write of whole blocks, every layer, K and V.
* ``greedy``  the greedy pick of a step's logits.
* ``swap``    preempted sequences out to pinned host memory and back into
  other blocks.

Lengths follow the serving benchmark's laws (lognormal with sigma 0.8 clipped
to 2048 tokens, or uniform) and are fixed by the case; block tables, cache
contents and activations come from the seed.
"""

from __future__ import annotations

import math
import random

import torch

from llm_serving_layer_amd import (BlockAllocator, KVSwapSpace, MI355XBackend, ScheduledSeq,
                                   SequenceBlocks, build_batch_meta)
from llm_serving_layer_amd.sampling import greedy

DEV = "cuda:0"
PAGE = 16
MAX_SEQ = 2048
DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}
BITS = {"float16": torch.int16, "bfloat16": torch.int16, "float32": torch.int32}

# 32 query heads over 8 KV heads at head_dim 64, the benchmark's geometry
BASE = {"n_kv": 8, "n_heads": 32, "head_dim": 64}


def _step(name, dtype, layers, *, n_decode=0, law="lognormal", mean=0, lo=0, hi=0, n_chunk=0,
          chunk_lo=0, chunk_hi=0, history=0, shared=False, describe=False, lens_seed=20260731,
          **geom):
    case = {"kind": "attend", "dtype": dtype, "layers": layers, **BASE, **geom,
            "n_decode": n_decode, "law": law, "mean": mean, "lo": lo, "hi": hi,
            "n_chunk": n_chunk, "chunk_lo": chunk_lo, "chunk_hi": chunk_hi,
            "history": history, "shared": shared, "describe": describe,
            "lens_seed": lens_seed}
    return {"name": name, **case} if name else case


def listed():
    return [
        # one user alone: the latency of a decode step, 16 layers
        _step("decode_single", "float16", 16, n_decode=1, law="uniform", lo=1371, hi=1371),
        # a lightly loaded server of a model with head_dim 128, in bf16
        _step("decode_few", "bfloat16", 8, n_decode=16, mean=258, head_dim=128),
        # the headline decode step: batch 256, lognormal lengths of mean 258
        _step("decode_batch", "float16", 4, n_decode=256, mean=256),
        # high concurrency: thousands of short conversations
        _step("decode_short", "float16", 4, n_decode=4096, law="uniform", lo=16, hi=64),
        # high concurrency with long histories, the largest step
        _step("decode_long", "float16", 4, n_decode=512, mean=2048),
        # chunked prefill of eight requests over one radix-cached system prompt
        _step("prefill_shared", "float16", 4, n_chunk=8, chunk_lo=512, chunk_hi=512,
              history=1536, shared=True),
        # one request's whole prompt, odd length, nothing cached
        _step("prefill_prompt", "bfloat16", 8, n_chunk=1, chunk_lo=777, chunk_hi=777,
              head_dim=128),
        # continuous batching, described and planned in the pass: one prompt
        # chunk behind a cached history rides along with running decodes
        _step("mixed_step", "float16", 16, n_decode=48, mean=258, n_chunk=1, chunk_lo=300,
              chunk_hi=300, history=720, describe=True),
        # an fp32 pool, as the preemption gate runs it: two prompts rebuilt by
        # recompute while others decode
        _step("mixed_fp32", "float32", 4, n_decode=24, mean=258, n_chunk=2, chunk_lo=60,
              chunk_hi=200),
        # radix copy-on-write, 27% of the sources from a shared prefix
        {"name": "copy_on_write", "kind": "copy", "dtype": "float16", "layers": 16, **BASE,
         "pairs": 4096, "lens_seed": 20260731},
        # the greedy pick of a batch-256 step over a 128 256-entry vocabulary
        {"name": "greedy_batch", "kind": "greedy", "dtype": "float16", "rows": 256,
         "vocab": 128256},
        # preemption: 64 sequences of 256 tokens leave and come back
        {"name": "swap_cycle", "kind": "swap", "dtype": "float16", "layers": 16, **BASE,
         "victims": 64, "tokens": 256},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


GEOMS = [(8, 32, 64), (8, 32, 64), (8, 32, 128), (2, 8, 128), (8, 8, 64), (4, 8, 64), (2, 32, 64),
         (4, 16, 64)]


def draw(rng):
    kind = rng.choices(["decode", "prefill", "mixed", "copy", "greedy", "swap"],
                       [45, 25, 10, 7, 8, 5])[0]
    n_kv, n_heads, d = rng.choice(GEOMS)
    geom = {"n_kv": n_kv, "n_heads": n_heads, "head_dim": d}
    dtype = rng.choices(["float16", "bfloat16", "float32"], [5, 3, 2])[0]
    seed = rng.randrange(1 << 30)
    row = 2 * n_kv * d * (4 if dtype == "float32" else 2)      # K and V bytes of a token
    if kind == "greedy":
        return {"kind": "greedy", "dtype": dtype, "rows": _log(rng, 1, 256),
                "vocab": rng.choice([_log(rng, 1000, 152000), 32000, 128256])}
    if kind == "copy":
        return {"kind": "copy", "dtype": dtype, "layers": rng.choice([2, 8, 16]), **geom,
                "pairs": _log(rng, 1, 2048), "lens_seed": seed}
    if kind == "swap":
        return {"kind": "swap", "dtype": dtype, "layers": rng.choice([4, 16]), **geom,
                "victims": _log(rng, 1, 32), "tokens": rng.randint(17, 300)}
    if kind == "prefill":
        n, hi = _log(rng, 1, 8), _log(rng, 2, 900)
        if dtype == "float32":
            n, hi = min(n, 3), min(hi, 300)
        shared = n > 1 and rng.random() < 0.4
        history = rng.choice([0, rng.randint(1, 1100)])
        history = min(history, 400) if dtype == "float32" else history
        return _step(None, dtype, 4, n_chunk=n, chunk_lo=max(2, hi // 2), chunk_hi=hi,
                     history=history // PAGE * PAGE if shared else history, shared=shared,
                     lens_seed=seed, **geom)
    # decode (and the decodes of a mixed step): tokens bounded by 400 MB a layer
    n, mean = _log(rng, 1, 1024), _log(rng, 24, 1100)
    cap = 4e8 / row if dtype != "float32" else 12000
    n = max(1, min(n, int(cap / mean)))
    if kind == "decode":
        if rng.random() < 0.3:
            return _step(None, dtype, 4, n_decode=n, law="uniform", lo=max(1, mean // 4),
                         hi=2 * mean, lens_seed=seed, **geom)
        return _step(None, dtype, 4, n_decode=n, mean=mean, lens_seed=seed, **geom)
    hi = _log(rng, 2, 512 if dtype != "float32" else 150)
    return _step(None, dtype, 8, n_decode=min(n, 256), mean=mean, n_chunk=rng.randint(1, 3),
                 chunk_lo=max(2, hi // 2), chunk_hi=hi, history=rng.choice([0, rng.randint(1, 800)]),
                 describe=rng.random() < 0.5, lens_seed=seed, **geom)


# ------------------------------------------------------------------ inputs ---

def _lengths(case):
    """(history, new tokens) of every sequence: decodes first, then chunks."""
    rng = random.Random(case["lens_seed"])
    out = []
    mu = math.log(max(case["mean"], 1)) - 0.8 ** 2 / 2.0
    for _ in range(case["n_decode"]):
        n = (rng.randint(case["lo"], case["hi"]) if case["law"] == "uniform"
             else int(round(rng.lognormvariate(mu, 0.8))))
        out.append((max(1, min(MAX_SEQ, n)) - 1, 1))   # the step appends the n-th token
    for _ in range(case["n_chunk"]):
        out.append((case["history"], rng.randint(case["chunk_lo"], case["chunk_hi"])))
    return out


def _pages(n):
    return -(-n // PAGE)


def _tables(case, seed):
    """(blocks of the pool, their order on the free list, page ids of every
    sequence, the shared prefix's pages), as an allocator hands them out in
    that order."""
    lens = _lengths(case)
    pre = _pages(case["history"]) if case["shared"] else 0
    own = [_pages(h + n) - (pre if case["shared"] and n > 1 else 0) for h, n in lens]
    used = pre + sum(own)
    nb = used + max(8, used // 4)
    order = list(range(nb))
    random.Random(seed).shuffle(order)
    prefix, at, tables = order[:pre], pre, []
    for (h, n), k in zip(lens, own):
        ids = order[at:at + k]
        at += k
        tables.append(prefix + ids if case["shared"] and n > 1 else ids)
    return nb, order, tables, prefix


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _values(shape, dtype, g):
    return torch.randn(shape, generator=g, device=DEV).mul_(0.5).to(dtype)


def _activations(case, n_tokens, g):
    """q, k and v of each layer's step."""
    dt, d = DTYPES[case["dtype"]], case["head_dim"]
    return [tuple(_values((n_tokens, h, d), dt, g)
                  for h in (case["n_heads"], case["n_kv"], case["n_kv"]))
            for _ in range(case["layers"])]


def _cache(case, nb, g):
    """K and V of each layer's whole pool, one layer at a time."""
    shape = (nb, PAGE, case["n_kv"], case["head_dim"])
    for _ in range(case["layers"]):
        yield (_values(shape, DTYPES[case["dtype"]], g), _values(shape, DTYPES[case["dtype"]], g))


def _backend(case, nb, g):
    bk = MI355XBackend(case["layers"], nb, PAGE, case["n_kv"], case["n_heads"],
                       case["head_dim"], device=DEV, dtype=DTYPES[case["dtype"]])
    kp, vp = bk.k_pool, bk.v_pool
    for l, (k, v) in enumerate(_cache(case, nb, g)):
        kp[l].copy_(k)
        vp[l].copy_(v)
    # the cache is an output too: data movement, compared as bytes
    bits = BITS[case["dtype"]]
    return bk, [p.view(bits) for p in kp], [p.view(bits) for p in vp]


def _allocator(nb, order):
    alloc = BlockAllocator(nb, PAGE)
    alloc.allocate(nb)
    alloc.free(order)
    return alloc


def _copy_pairs(case, seed):
    """(pool blocks, sources, destinations): 27% of the sources repeat blocks
    of a shared prefix, destinations are distinct free blocks."""
    pairs = case["pairs"]
    shared = max(1, min(64, pairs // 8))
    nb = shared + 2 * pairs
    order = list(range(nb))
    random.Random(seed).shuffle(order)
    uniq, dst = order[shared:shared + pairs], order[shared + pairs:]
    rng = random.Random(case["lens_seed"])
    src = [order[rng.randrange(shared)] if rng.random() < 0.27 else uniq[i]
           for i in range(pairs)]
    return nb, src, dst


def _logits(case, seed):
    return torch.randn((case["rows"], case["vocab"]), generator=_gen(seed),
                       device=DEV).mul_(4.0).to(DTYPES[case["dtype"]])


def prepare(case, seed):
    g = _gen(seed)
    if case["kind"] == "greedy":
        return {"kind": "greedy", "logits": _logits(case, seed)}
    if case["kind"] == "copy":
        nb, src, dst = _copy_pairs(case, seed)
        bk, k, v = _backend(case, nb, g)
        return {"kind": "copy", "bk": bk, "src": src, "dst": dst, "k": k, "v": v}
    if case["kind"] == "swap":
        n = case["victims"]
        nb = 2 * n * _pages(case["tokens"]) + 8
        order = list(range(nb))
        random.Random(seed).shuffle(order)
        bk, k, v = _backend(case, nb, g)
        alloc = _allocator(nb, order)
        seqs = [SequenceBlocks(alloc, seq_id=i) for i in range(n)]
        for s in seqs:
            s.append(case["tokens"])
        return {"kind": "swap", "bk": bk, "space": KVSwapSpace(bk), "alloc": alloc,
                "seqs": seqs, "tokens": case["tokens"], "k": k, "v": v}
    lens = _lengths(case)
    nb, order, _, prefix = _tables(case, seed)
    bk, k, v = _backend(case, nb, g)
    alloc = _allocator(nb, order)
    pre = alloc.allocate(len(prefix))
    seqs = []
    for i, (h, n) in enumerate(lens):
        s = SequenceBlocks(alloc, seq_id=i)
        if case["shared"] and n > 1:
            alloc.incref(pre)
            s.block_ids, s.num_tokens = list(pre), h
            s.append(n)
        else:
            s.append(h + n)
        seqs.append(ScheduledSeq(s, [0] * n))
    acts = _activations(case, sum(n for _, n in lens), g)
    meta = None if case["describe"] else build_batch_meta(seqs, DEV, PAGE)
    return {"kind": "attend", "bk": bk, "seqs": seqs, "meta": meta, "acts": acts,
            "scale": case["head_dim"] ** -0.5, "k": k, "v": v}


def run(state):
    kind = state["kind"]
    if kind == "greedy":
        return greedy(state["logits"])
    bk = state["bk"]
    if kind == "copy":
        bk.copy_blocks(state["src"], state["dst"])
        return {"k": state["k"], "v": state["v"]}
    if kind == "swap":
        space, seqs = state["space"], state["seqs"]
        handles = [space.swap_out(str(s.seq_id), s) for s in seqs]
        back = []
        for s in seqs:
            s.free()
        for h in handles:
            s = SequenceBlocks(state["alloc"], seq_id=h.seq_id)
            s.append(state["tokens"])
            space.swap_in(h, s)
            back.append(s)
        for h in handles:
            space.release(h)
        state["seqs"] = back
        return {"k": state["k"], "v": state["v"]}
    meta = state["meta"]
    if meta is None:
        meta = build_batch_meta(state["seqs"], DEV, PAGE)
    out = []
    for l, (q, k, v) in enumerate(state["acts"]):
        bk.append_kv(l, k, v, meta)
        out.append(bk.attend(q, l, state["scale"], meta))
    return {"out": out, "k": state["k"], "v": state["v"]}


# ------------------------------------------------------------ work, exact ---

def work(case):
    eb = 4 if case["dtype"] == "float32" else 2
    if case["kind"] == "greedy":
        return {"bytes": case["rows"] * (case["vocab"] * eb + 8), "flops": 0}
    block = 2 * case["layers"] * PAGE * case["n_kv"] * case["head_dim"] * eb
    if case["kind"] == "copy":
        _, src, dst = _copy_pairs(case, 0)
        return {"bytes": (len(set(src)) + len(dst)) * block, "flops": 0}
    if case["kind"] == "swap":   # out: read and write; in: read and write
        return {"bytes": 4 * case["victims"] * _pages(case["tokens"]) * block, "flops": 0}
    lens = _lengths(case)
    hq, hkv, d = case["n_heads"], case["n_kv"], case["head_dim"]
    n_new = sum(n for _, n in lens)
    keys = sum(h + n for h, n in lens)
    if case["shared"]:           # the prefix is read once
        keys -= (case["n_chunk"] - 1) * case["history"]
    pairs = sum(n * h + n * (n + 1) // 2 for h, n in lens)
    per_layer = keys * 2 * hkv * d * eb          # cached and new K, V rows
    per_layer += 2 * n_new * hq * d * eb         # q read, output written
    per_layer += 2 * n_new * 2 * hkv * d * eb    # new rows read and stored
    return {"bytes": case["layers"] * per_layer, "flops": case["layers"] * 4 * d * hq * pairs}


def tolerance(case):
    if case["kind"] != "attend":
        return "exact"
    # four times the distance from 64 bits measured per type (2.9e-4 in fp16
    # and 2.3e-3 in bf16, where the probabilities and the output are rounded
    # to the pool's type); fp32 measures 1e-7, and sums of up to 2048 terms in
    # another order may be a few roundings further off
    return {"float16": {"rel": 1.2e-3}, "bfloat16": {"rel": 1e-2},
            "float32": {"rel": 2e-6}}[case["dtype"]]


def exact(case, seed):
    if case["kind"] == "greedy":
        return torch.argmax(_logits(case, seed), dim=-1)
    if case["kind"] != "attend":
        return None
    lens = _lengths(case)
    nb, _, tables, _ = _tables(case, seed)
    g = _gen(seed)
    d, groups = case["head_dim"], case["n_heads"] // case["n_kv"]
    # cache and activations come from one generator, in prepare's order; each
    # layer keeps the rows of the sequences only
    ids = [torch.tensor(t, device=DEV) for t in tables]
    caches = [(k, v) for k, v in _cache(case, nb, g)]
    acts = _activations(case, sum(n for _, n in lens), g)
    outs = []
    for (kc, vc), (q, k, v) in zip(caches, acts):
        out, at = torch.empty_like(q, dtype=torch.float64), 0
        for (h, n), t in zip(lens, ids):
            kk = torch.cat([kc[t].flatten(0, 1)[:h], k[at:at + n]]).double().transpose(0, 1)
            vv = torch.cat([vc[t].flatten(0, 1)[:h], v[at:at + n]]).double().transpose(0, 1)
            qq = q[at:at + n].double().transpose(0, 1).reshape(case["n_kv"], groups * n, d)
            s = torch.matmul(qq, kk.transpose(1, 2).contiguous()).mul_(d ** -0.5)
            if n > 1:
                pos = torch.arange(h, h + n, device=DEV).repeat(groups)
                s.masked_fill_(torch.arange(h + n, device=DEV)[None, :] > pos[:, None],
                               -math.inf)
            o = torch.matmul(torch.softmax(s, dim=-1), vv.contiguous())
            out[at:at + n] = o.view(case["n_heads"], n, d).transpose(0, 1)
            at += n
        outs.append(out)
    none = [None] * case["layers"]   # the pools: bytes moved, no arithmetic
    return {"out": outs, "k": none, "v": none}
