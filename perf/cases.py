"""The work that users of this framework have it do, as measurable cases.

A case is a dict of plain values.  `path` says which public entry point it goes through:

  decode   one new token per sequence over a contiguous K/V cache (SparseAttention.forward)
  paged    one new token per sequence over a paged K/V cache (SparseAttention.paged_decode)
  prefill  causal forward over unpadded sequences, with the log-sum-exp
  padded   causal forward over left- or right-padded prompts
  packed   forward over packed sequences of a user-defined pattern, the keys split in two
           partitions that combine_attn_partitions merges
  train    forward and backward through autograd

The listed cases are the configurations that bench.py and the benchmark scripts run plus generic
ones between and below them; draw() spreads the same paths over their ranges of sizes.
"""
import functools
import math
import random
import warnings

import numpy as np
import torch

from dkernel_amd import LocalStrideSparseAttention, SparseAttention, combine_attn_partitions

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
DEV = "cuda"


def listed():
    """From the smallest call to the largest."""
    pattern = dict(block=64, local=16, vert=8)
    gqa = dict(heads=32, kv_heads=8, head_dim=128, dtype="bf16")
    return [
        # one user chatting: the next token of a single conversation of ordinary length
        dict(name="decode_one_sequence", path="decode", batch=1, min_len=1000, max_len=1000, padding="none",
             heads_first=False, **gqa, **pattern),
        # a serving step over a batch of conversations of unequal length, left-padded (bench.py's decode)
        dict(name="decode_left_padded_batch", path="decode", batch=32, min_len=1024, max_len=8192, padding="left",
             heads_first=False, **gqa, **pattern),
        # the same behind a block manager: scattered 16-token pages, many shorter conversations
        dict(name="decode_paged_batch", path="paged", batch=48, min_len=256, max_len=6000, page=16, fp8=False, **gqa,
             **pattern),
        # the prompt of one request
        dict(name="prefill_short_prompt", path="prefill", batch=1, length=333, heads_first=False, **gqa, **pattern),
        # prompts of a batch of requests, padded to the longest one, heads in front of the tokens
        dict(name="prefill_left_padded_prompts", path="padded", batch=6, min_len=200, max_len=2000, padding="left",
             heads=32, kv_heads=32, head_dim=96, dtype="fp16", heads_first=True, block=64, local=8, vert=4),
        # documents read into the cache (bench.py's headline)
        dict(name="prefill_8k_documents", path="prefill", batch=2, length=8192, heads_first=False, **gqa, **pattern),
        # one very long document
        dict(name="prefill_long_document", path="prefill", batch=1, length=32700, heads_first=False, **gqa, **pattern),
        # a pattern of the user's own over packed sequences, keys in two partitions (sequence parallelism)
        dict(name="packed_key_partitions", path="packed", sequences=8, min_len=512, max_len=4096, tokens=16384, heads=16,
             kv_heads=16, head_dim=128, dtype="bf16", block=64, density=0.2),
        # pre-training step at long context (bench.py's backward)
        dict(name="train_8k_context", path="train", batch=1, length=8192, heads=32, kv_heads=32, head_dim=128,
             dtype="bf16", fused_qkv=False, pattern="local_stride", **pattern),
        # fine-tuning step on a batch of shorter samples, grouped heads out of one fused projection
        dict(name="train_grouped_fused_qkv", path="train", batch=4, length=2048, fused_qkv=True, pattern="local_stride",
             **gqa, **pattern),
        # a bidirectional encoder with global blocks and fine-grained blocks, ragged length
        dict(name="train_encoder_small_blocks", path="train", batch=4, length=3000, heads=12, kv_heads=12, head_dim=64,
             dtype="fp16", fused_qkv=False, pattern="global_window", block=32, local=3, vert=0),
        # single precision: a smaller model trained, or a larger one checked, without 16-bit rounding
        dict(name="train_fp32", path="train", batch=1, length=2000, heads=16, kv_heads=16, head_dim=128, dtype="fp32",
             fused_qkv=False, pattern="local_stride", block=64, local=8, vert=4),
    ]


def _log(rng, lo, hi):
    """A whole number spread evenly over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _pattern(rng, blocks=(64, 64, 64, 32, 128)):
    block = rng.choice(blocks)
    return dict(block=block, local=max(1, rng.choice((256, 512, 1024)) // block), vert=rng.choice((4, 8, 16)))


def _heads(rng):
    heads, kv = rng.choice(((32, 8), (32, 8), (32, 32), (16, 16), (16, 4), (24, 8), (8, 8), (12, 12)))
    return dict(heads=heads, kv_heads=kv, head_dim=rng.choice((128, 128, 128, 64, 96, 256)),
                dtype=rng.choice(("bf16", "bf16", "fp16")))


def _draw_once(rng):
    path = rng.choice(("decode", "decode", "paged", "prefill", "prefill", "padded", "packed", "train", "train", "train"))
    if path in ("decode", "paged"):
        longest = _log(rng, 200, 16000)
        case = dict(path=path, batch=_log(rng, 1, 96), min_len=max(1, longest // 8), max_len=longest, **_heads(rng))
        if path == "decode":
            case.update(padding=rng.choice(("left", "right")), heads_first=rng.random() < 0.4, **_pattern(rng))
            if case["batch"] == 1:
                case.update(padding="none", min_len=longest)
        else:
            case.update(page=rng.choice((16, 16, 32, 64)), fp8=rng.random() < 0.3, **_pattern(rng, (64,)))
            if case["head_dim"] not in (64, 128):
                case["fp8"] = False
        return case
    if path == "prefill":
        return dict(path=path, batch=_log(rng, 1, 4), length=_log(rng, 100, 32000), heads_first=rng.random() < 0.4,
                    **_heads(rng), **_pattern(rng))
    if path == "padded":
        longest = _log(rng, 200, 8000)
        return dict(path=path, batch=_log(rng, 2, 16), min_len=max(1, longest // 10), max_len=longest,
                    padding=rng.choice(("left", "right")), heads_first=rng.random() < 0.4, **_heads(rng), **_pattern(rng))
    if path == "packed":
        longest = _log(rng, 300, 6000)
        return dict(path=path, sequences=_log(rng, 2, 24), min_len=max(1, longest // 8), max_len=longest, tokens=20000,
                    **_heads(rng), block=64, density=round(rng.uniform(0.1, 0.4), 2))
    case = dict(path="train", batch=_log(rng, 1, 6), length=_log(rng, 300, 10000), **_heads(rng))
    case["fused_qkv"] = rng.random() < 0.4
    if rng.random() < 0.3:
        case.update(dtype="fp32", head_dim=rng.choice((64, 96, 128)))
    if rng.random() < 0.3:
        case.update(pattern="global_window", block=rng.choice((64, 32, 32)), local=rng.randint(1, 4), vert=0)
    else:
        case.update(pattern="local_stride", **_pattern(rng))
    return case


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        case = _draw_once(rng)
        if _cost(case) <= most:
            return case


# ---- the parts of a case that do not depend on the inputs' values --------------------------------

def _lengths(case):
    """Sequence lengths: the case's own, the same for every seed (the tensors' shapes follow them)."""
    n = case["batch"] if "batch" in case else case["sequences"]
    r = random.Random(n * 1000003 + case["max_len"])
    lens = [r.randint(case["min_len"], case["max_len"]) for _ in range(n)]
    if case["path"] == "packed":  # at most `tokens` in all
        while sum(lens) > case["tokens"]:
            lens = [max(1, x * 9 // 10) for x in lens]
    return lens


@functools.lru_cache(maxsize=4)
def _random_pattern(heads, blocks, density):
    g = torch.Generator().manual_seed(20)
    pat = torch.rand(heads, blocks, blocks, generator=g) < density
    pat |= torch.eye(blocks, dtype=torch.bool)[None]
    return torch.tril(pat.to(torch.uint8))


def _global_window_pattern(blocks, block, window):
    """The first 128 tokens attend and are attended by everything, a window around the diagonal,
    three random blocks a row."""
    g = torch.Generator().manual_seed(1)
    i = torch.arange(blocks)
    pat = (i[:, None] - i[None, :]).abs() <= window
    pat[:128 // block, :] = True
    pat[:, :128 // block] = True
    return pat | (torch.rand(blocks, blocks, generator=g) < 3 / blocks)


@functools.lru_cache(maxsize=16)
def _local_module(heads, kv_heads, length, block, local, vert, heads_first):
    return LocalStrideSparseAttention(heads, length, block, local, vert, num_kv_heads=kv_heads,
                                      seq_dim=2 if heads_first else 1).to(DEV)


@functools.lru_cache(maxsize=8)
def _global_window_module(length, block, window):
    return SparseAttention(block, _global_window_pattern(-(-length // block), block, window), causal=False).to(DEV)


@functools.lru_cache(maxsize=4)
def _partition_modules(heads, length, block, density):
    """The user's pattern with its key blocks split in two halves."""
    pat = _random_pattern(heads, -(-length // block), density)
    half = max(1, pat.size(2) // 2)
    first, second = pat.clone(), pat.clone()
    first[:, :, half:] = 0
    second[:, :, :half] = 0
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        return SparseAttention(block, first).to(DEV), SparseAttention(block, second).to(DEV)


def _module(case):
    longest = case["length"] if "length" in case else case["max_len"]
    if case["path"] == "packed":
        return _partition_modules(case["heads"], longest, case["block"], case["density"])
    if case.get("pattern") == "global_window":
        return _global_window_module(longest, case["block"], case["local"])
    return _local_module(case["heads"], case["kv_heads"], longest, case["block"], case["local"], case["vert"],
                         case.get("heads_first", False))


# ---- inputs and the pass ------------------------------------------------------------------------

def prepare(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    dtype, Hq, Hkv, D = DTYPES[case["dtype"]], case["heads"], case["kv_heads"], case["head_dim"]

    def rand(*shape):
        return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32).to(dtype)

    def tensor(batch, length, heads):  # (batch, length, heads, dim), or heads in front of the tokens
        return rand(batch, heads, length, D) if case.get("heads_first") else rand(batch, length, heads, D)

    def i32(values):
        return torch.tensor(values, dtype=torch.int32, device=DEV)

    state = dict(path=case["path"], mod=_module(case), scale=1.0 / math.sqrt(D))
    path = case["path"]
    if path == "decode" or path == "padded":
        lens, longest = _lengths(case), case["max_len"]
        state["q"] = tensor(case["batch"], 1 if path == "decode" else longest, Hq)
        state["k"], state["v"] = tensor(case["batch"], longest, Hkv), tensor(case["batch"], longest, Hkv)
        state["lengths"] = {"none": {}, "left": {"left_paddings": i32([longest - x for x in lens])},
                            "right": {"seqlens": i32(lens)}}[case["padding"]]
    elif path == "paged":
        lens, page = _lengths(case), case["page"]
        per_seq = -(-case["max_len"] // page)
        used = [-(-x // page) for x in lens]
        pages = sum(used)
        where = torch.randperm(pages, generator=g, device=DEV).to(torch.int32)
        table = torch.zeros(case["batch"], per_seq, dtype=torch.int32, device=DEV)
        at = 0
        for i, n in enumerate(used):
            table[i, :n] = where[at:at + n]
            at += n
        state["q"] = rand(case["batch"], Hq, D)
        pools = [rand(pages, page, Hkv, D) for _ in range(2)]
        state["scales"] = {}
        if case["fp8"]:
            pools = [(p.float() * 32).to(torch.float8_e4m3fn) for p in pools]
            state["scales"] = {"k_scale": 1 / 32, "v_scale": 1 / 32}
        state["k"], state["v"], state["table"], state["lens"] = pools[0], pools[1], table, i32(lens)
    elif path == "packed":
        lens = _lengths(case)
        total = sum(lens)
        state["q"], state["k"], state["v"] = rand(total, Hq, D), rand(total, Hkv, D), rand(total, Hkv, D)
        state["cu"] = i32([0] + list(np.cumsum(lens)))
    else:
        B, L = case["batch"], case["length"]
        if case.get("fused_qkv"):
            state["qkv"] = rand(B, L, Hq + 2 * Hkv, D).requires_grad_()
            state["split"] = lambda x: (x[:, :, :Hq], x[:, :, Hq:Hq + Hkv], x[:, :, Hq + Hkv:])
        else:
            state["q"], state["k"], state["v"] = tensor(B, L, Hq), tensor(B, L, Hkv), tensor(B, L, Hkv)
        if path == "train":
            state["dout"] = tensor(B, L, Hq)
            for name in ("q", "k", "v"):
                if name in state:
                    state[name].requires_grad_()
    return state


def run(state):
    s, mod = state, state["mod"]
    if s["path"] == "train":
        if "qkv" in s:
            out = mod(s["qkv"], sm_scale=s["scale"], split_qkv=s["split"])
            return (out.detach(), *torch.autograd.grad(out, (s["qkv"],), s["dout"]))
        out = mod(s["q"], s["k"], s["v"], s["scale"])
        return (out.detach(), *torch.autograd.grad(out, (s["q"], s["k"], s["v"]), s["dout"]))
    with torch.no_grad():
        if s["path"] == "paged":
            return mod.paged_decode(s["q"], s["k"], s["v"], s["table"], s["lens"], s["scale"], **s["scales"])
        if s["path"] == "packed":
            parts = [m(s["q"], s["k"], s["v"], s["scale"], cu_seqlen_k=s["cu"], return_lse=True) for m in mod]
            return (combine_attn_partitions(*parts, hdim=1), parts[0][1], parts[1][1])
        if s["path"] == "prefill":
            return mod(s["q"], s["k"], s["v"], s["scale"], return_lse=True)
        return mod(s["q"], s["k"], s["v"], s["scale"], **s["lengths"])


# ---- what a pass cannot do without --------------------------------------------------------------

def _verticals(n, head, case):
    """Vertical columns of kv head `head` among the first n column blocks (arrays welcome)."""
    vert = case["vert"]
    shift = head * max(1, vert // case["heads"])
    return (n + shift + vert - 1) // vert - (shift + vert - 1) // vert if vert > 1 else n


def _local_stride_pairs(case, length):
    """Visible (query, key) pairs of one sequence, all kv heads together."""
    bs, local = case["block"], case["local"]
    r = np.arange(-(-length // bs))
    rows = np.minimum(bs, length - r * bs)
    pairs = 0
    for h in range(case["kv_heads"]):
        blocks = np.minimum(r, local - 1) + _verticals(np.maximum(r - local + 1, 0), h, case)
        pairs += int((blocks * bs * rows + rows * (rows + 1) // 2).sum())
    return pairs


def _listed_pairs(pattern, bs, length, causal):
    """The same for a block pattern (heads, blocks, blocks) that is given."""
    n = -(-length // bs)
    size = torch.clamp(length - torch.arange(n) * bs, max=bs).double()
    p = pattern[:, :n, :n].double()
    pairs = (p * size[:, None] * size[None, :]).sum()
    if causal:
        pairs -= (p.diagonal(dim1=1, dim2=2) * (size * (size - 1) / 2)).sum()
    return float(pairs)


@functools.lru_cache(maxsize=256)
def _work(items):
    case = dict(items)
    Hq, Hkv, D = case["heads"], case["kv_heads"], case["head_dim"]
    es, group, path = (4 if case["dtype"] == "fp32" else 2), case["heads"] // case["kv_heads"], case["path"]
    if path in ("decode", "paged"):
        keys = 0
        for n in _lengths(case):
            r = (n - 1) // case["block"]
            for h in range(Hkv):
                full = min(r, case["local"] - 1) + int(_verticals(max(r - case["local"] + 1, 0), h, case))
                keys += full * case["block"] + n - r * case["block"]
        kv = 1 if case.get("fp8") else es
        return {"bytes": 2 * keys * D * kv + 2 * case["batch"] * Hq * D * es, "flops": 4 * keys * group * D}
    if path == "packed":
        lens = _lengths(case)
        pat = _random_pattern(Hq, -(-case["max_len"] // case["block"]), case["density"])
        pairs = sum(_listed_pairs(pat, case["block"], n, True) for n in lens)
        row = D * es + 4  # one output row and its log-sum-exp
        # per partition q and its share of k / v read and its result written; the merge reads both
        # results and writes one
        return {"bytes": sum(lens) * (2 * (Hq * D + Hkv * D) * es + 4 * Hq * row + Hq * D * es), "flops": 4 * pairs * D}
    if path == "padded":
        lens = _lengths(case)
        pairs = sum(_local_stride_pairs(case, n) for n in lens) * group
        # padding rows of the output are written (zeros), those of the inputs are not needed
        return {"bytes": sum(lens) * (Hq + 2 * Hkv) * D * es + case["batch"] * case["max_len"] * Hq * D * es,
                "flops": 4 * pairs * D}
    B, L = case["batch"], case["length"]
    if case.get("pattern") == "global_window":
        pat = _global_window_pattern(-(-L // case["block"]), case["block"], case["local"])
        pairs = _listed_pairs(pat[None], case["block"], L, False) * Hq
    else:
        pairs = _local_stride_pairs(case, L) * group
    qo, kv = B * L * Hq * D * es, B * L * Hkv * D * es
    forward = 2 * qo + 2 * kv + B * L * Hq * 4
    if path == "prefill":
        return {"bytes": forward, "flops": 4 * B * pairs * D}
    # backward: q, k, v, o, dO and the log-sum-exp read, dq, dk, dv written; five products to the forward's two
    return {"bytes": forward + 4 * qo + 4 * kv + B * L * Hq * 4, "flops": 14 * B * pairs * D}


def work(case):
    return dict(_work(tuple(sorted((k, v) for k, v in case.items() if k != "name"))))


def _cost(case):
    """A drawn case's expense next to the listed ones (arbitrary unit): products at the matrix rate
    of their type, every byte at the memory's."""
    w = work(case)
    return w["flops"] * (16 if case["dtype"] == "fp32" else 1) + 300 * w["bytes"]


def tolerance(case):
    # Four times what outputs and gradients differ from the same attention in 64 bits (lengths of 333 and 2000,
    # head dims 64 and 128: relative 2.6e-3, 3.3e-4 and 1.3e-6, largest 0.07, 0.018 and 2.8e-5): 16-bit results
    # carry one rounding of their own and one of the probabilities, gradients also one of dS; fp32 results the
    # order of sums of a few thousand products.
    return {"bf16": {"rel": 1e-2, "max": 0.28}, "fp16": {"rel": 1.3e-3, "max": 0.07},
            "fp32": {"rel": 5e-6, "max": 1.1e-4}}[case["dtype"]]
