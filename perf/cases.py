"""The calls this framework's speed is judged by: attention forward, training and few-rows decode over the range of
sizes, masks, element types and layouts that programs call it with.

A case is a dict of plain values.  ``prepare`` makes what a program holds before the call (inputs, and the mask metadata
where such a program keeps it), ``run`` is one pass through the public entry points, ``work`` the bytes and operations
that pass cannot do without.
"""
from __future__ import annotations

import math
import random

import torch

import sparseattention_amd as sa

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def listed() -> list[dict]:
    return [
        # the smallest configuration: float32, four heads, a block mask of 32 x 32 blocks; a unit test's or a toy model's call
        dict(name="plumbing_fp32", kind="forward", B=1, H=4, Sq=512, Sk=512, D=64, dtype="fp32", layout="bhsd",
             mask="blocks", block=32, p=0.5, BQ=64, BK=32),
        # one short prompt, the mask handed over as a tensor with nothing kept: the reference's plain call
        dict(name="prompt_mask_tensor", kind="forward_fresh", B=1, H=32, Sq=1024, Sk=1024, D=128, dtype="bf16",
             layout="bshd", mask="causal", BQ=128, BK=64),
        # a chunk of a long prompt against the keys already cached: few query tiles, long lists
        dict(name="chunked_prefill", kind="forward", B=1, H=32, Sq=512, Sk=16384, D=128, dtype="bf16", layout="bhsd",
             mask="causal", BQ=128, BK=64),
        # packed documents of no round length, a head dim between the kernels' and half precision, on a tile grid
        # chosen once
        dict(name="ragged_documents_fp16", kind="tiled", B=2, H=16, Sq=1499, Sk=1499, D=80, dtype="fp16", layout="bhsd",
             mask="documents", lo=64, hi=700, BQ=128, BK=64),
        # the headline: causal mask as a tensor, metadata kept over the layers
        dict(name="causal", kind="forward", B=8, H=32, Sq=4096, Sk=4096, D=128, dtype="bf16", layout="bhsd",
             mask="causal", BQ=128, BK=32),
        # random blocks, three quarters of them empty, a mask per batch element as the reference's sweep draws them
        dict(name="random_blocks", kind="forward", B=8, H=16, Sq=4096, Sk=4096, D=128, dtype="bf16", layout="bhsd",
             mask="blocks_batch", block=128, p=0.75, BQ=128, BK=32),
        # sliding window and bidirectional prefix at 32768 keys: a 1 GiB mask tensor classified and used
        dict(name="composed_mask_tensor", kind="forward_fresh", B=1, H=32, Sq=32768, Sk=32768, D=128, dtype="bf16",
             layout="bhsd", mask="composed", window=1024, prefix=2048, BQ=128, BK=32),
        # a training step's attention at the largest size listed, forward and gradients, metadata kept over the steps
        dict(name="train_causal", kind="train", B=8, H=16, Sq=4096, Sk=4096, D=128, dtype="bf16", layout="bhsd",
             mask="causal", BQ=128, BK=64),
        # a training step on packed documents: the documents of a batch are new at every step, so the lists are too
        dict(name="train_packed_documents", kind="train_terms", B=4, H=12, Sq=2048, Sk=2048, D=64, dtype="bf16",
             layout="bshd", mask="documents", lo=64, hi=1024, BQ=128, BK=64),
        # one token of a small batch, the padding mask new at every token: latency
        dict(name="decode_token", kind="decode_fresh", B=4, H=32, Sq=1, Sk=2048, D=128, dtype="bf16", layout="bhsd",
             mask="lengths", BK=64),
        # one token against a long context, every key
        dict(name="decode_long", kind="decode", B=8, H=32, Sq=1, Sk=32768, D=128, dtype="bf16", layout="bhsd",
             mask="all", BK=128),
        # sixteen rows (speculative or chunked tail): window, sink keys and a quarter of the far blocks
        dict(name="decode_rows16", kind="decode", B=8, H=16, Sq=16, Sk=16384, D=128, dtype="bf16", layout="bhsd",
             mask="window_sinks", window=4096, p=0.75, BK=128),
    ]


# ---- masks --------------------------------------------------------------------------------------------------------
def _document_ids(S: int, lo: int, hi: int, r: random.Random) -> list[int]:
    """Document number of every position: lengths uniform in [lo, hi], the last one cut off."""
    ids, n = [], 0
    while len(ids) < S:
        ids += [n] * min(r.randint(lo, hi), S - len(ids))
        n += 1
    return ids


def _documents(case: dict, r: random.Random) -> torch.Tensor:
    """int32 [B,S]: a layout of its own per batch element."""
    return torch.tensor([_document_ids(case["Sq"], case["lo"], case["hi"], r) for _ in range(case["B"])],
                        dtype=torch.int32, device="cuda")


def _mask(case: dict, r: random.Random, g: torch.Generator) -> torch.Tensor:
    """bool [B or 1, 1, Sq, Sk] on the GPU; query i stands at position i + Sk - Sq, as in a chunk against a cache."""
    B, Sq, Sk, kind = case["B"], case["Sq"], case["Sk"], case["mask"]
    q = (torch.arange(Sq, device="cuda", dtype=torch.int32) + (Sk - Sq))[:, None]
    k = torch.arange(Sk, device="cuda", dtype=torch.int32)[None, :]
    if kind == "all":
        return torch.ones(1, 1, Sq, Sk, dtype=torch.bool, device="cuda")
    if kind == "causal":
        return (k <= q)[None, None]
    if kind == "window":
        return ((k <= q) & (q - k < case["window"]))[None, None]
    if kind == "composed":
        m = (k <= q) & (q - k < case["window"])
        m[:case["prefix"], :case["prefix"]] = True
        return m[None, None]
    if kind == "documents":
        d = _documents(case, r)
        return ((d[:, :, None] == d[:, None, :]) & (k <= q)[None])[:, None]
    if kind in ("blocks", "blocks_batch"):
        # a block is empty with probability p, a tenth of them hold coin flips, the rest are full; the diagonal attends
        n, nq, nk = (B if kind == "blocks_batch" else 1), Sq // case["block"], Sk // case["block"]
        u = torch.rand(n, 1, nq, nk, device="cuda", generator=g)
        up = lambda t: t.repeat_interleave(case["block"], 2).repeat_interleave(case["block"], 3)  # noqa: E731
        coin = torch.randint(0, 2, (n, 1, Sq, Sk), device="cuda", generator=g, dtype=torch.uint8).bool()
        m = torch.where(up(u >= 0.9), coin, up(u > case["p"]))
        m.diagonal(dim1=-2, dim2=-1).fill_(True)
        return m
    if kind == "lengths":
        # a cache of Sk slots of which every sequence has filled its own number
        filled = torch.tensor([r.randint(Sk // 2, Sk) for _ in range(B)], dtype=torch.int32, device="cuda")
        rows = filled[:, None, None, None] - Sq + torch.arange(1, Sq + 1, device="cuda", dtype=torch.int32)[None, None, :, None]
        return k[None, None] < rows
    if kind == "window_sinks":
        far = torch.rand(1, 1, 1, Sk // 128, device="cuda", generator=g) > case["p"]
        m = (q - k < case["window"])[None, None] | (k < 512)[None, None] | far.repeat_interleave(128, 3)
        return m & (k <= q)[None, None]
    raise ValueError(kind)


def _attended(case: dict) -> float:
    """How many (query, key) pairs of one plane attend, in the mean over the seeds."""
    Sq, Sk, kind = case["Sq"], case["Sk"], case["mask"]
    causal = Sq * (Sk - Sq) + Sq * (Sq + 1) / 2
    if kind == "all":
        return float(Sq * Sk)
    if kind == "causal":
        return causal
    if kind in ("window", "composed"):
        short = max(0, min(Sq, case["window"] - (Sk - Sq)))  # rows that have fewer than `window` keys behind them
        n = (Sq - short) * min(case["window"], Sk) + short * (Sk - Sq) + short * (short + 1) / 2
        p = case.get("prefix", 0)
        return n + p * (p - 1) / 2 + (max(0, p - case["window"]) ** 2) / 2
    if kind == "documents":
        lo, hi = case["lo"], min(case["hi"], Sq)
        mean, square = (lo + hi) / 2, (lo * lo + lo * hi + hi * hi) / 3
        return Sq * (square / mean + 1) / 2
    if kind in ("blocks", "blocks_batch"):
        return Sq * Sk * (0.9 - min(0.9, case["p"]) + 0.05)
    if kind == "lengths":
        return Sq * Sk * 0.75
    near = min(Sk, case["window"] + 512)
    return Sq * (near + (Sk - near) * (1 - case["p"]))


# ---- one case -----------------------------------------------------------------------------------------------------
def _tensor(case: dict, S: int, g: torch.Generator) -> torch.Tensor:
    """Unit normal values, [B,H,S,D]; "bshd": as a projection leaves them, [B,S,H,D] seen through a transpose."""
    B, H, D, dt = case["B"], case["H"], case["D"], DTYPES[case["dtype"]]
    if case["layout"] == "bshd":
        return torch.randn(B, S, H, D, device="cuda", generator=g, dtype=dt).transpose(1, 2)
    return torch.randn(B, H, S, D, device="cuda", generator=g, dtype=dt)


def prepare(case: dict, seed: int) -> dict:
    r = random.Random(seed)
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind, B, H, Sq, Sk = case["kind"], case["B"], case["H"], case["Sq"], case["Sk"]
    st = dict(case, q=_tensor(case, Sq, g), k=_tensor(case, Sk, g), v=_tensor(case, Sk, g))
    if kind.startswith("train"):
        st["do"] = _tensor(case, Sq, g)
        for t in ("q", "k", "v"):
            st[t].requires_grad_(True)
    if kind == "train_terms":
        st["documents"] = _documents(case, r)  # (the data loader gives them; lists are made from them in the step)
        return st
    mask = _mask(case, r, g).expand(B, H, Sq, Sk)
    st["mask"] = mask
    if kind in ("forward", "train"):
        st["md"] = sa.compute_mask_kernel(mask, case["BQ"], case["BK"])
    if kind == "train":
        st["bmd"] = sa.compute_backward_metadata(mask)
    if kind == "tiled":
        st["tiling"] = sa.select_tiling(mask, candidates=((case["BQ"], case["BK"]),))
    if kind == "decode":
        st["md"] = sa.compute_mask_kernel(mask, Sq, case["BK"])
    return st


def run(st: dict):
    kind, q, k, v = st["kind"], st["q"], st["k"], st["v"]
    if kind == "forward":
        return sa.sparse_attention(q, k, v, st["mask"], st["BQ"], st["BK"], mask_metadata=st["md"])
    if kind == "forward_fresh":
        return sa.sparse_attention(q, k, v, st["mask"], st["BQ"], st["BK"])
    if kind == "tiled":
        return sa.sparse_attention_tiled(q, k, v, st["tiling"])
    if kind == "decode":
        return sa.sparse_attention_decode(q, k, v, st["mask"], st["BK"], st["md"])
    if kind == "decode_fresh":
        return sa.sparse_attention_decode(q, k, v, st["mask"], st["BK"])
    if kind == "train":
        o = sa.sparse_attention_trainable(q, k, v, st["mask"], st["BQ"], st["BK"], st["md"], st["bmd"])
    else:
        shape, docs, terms = (st["B"], st["H"], st["Sq"], st["Sk"]), st["documents"], [sa.causal_term(same_doc=True)]
        md = sa.compute_mask_terms(terms, *shape, st["BQ"], st["BK"], docs, docs)
        bmd = sa.compute_backward_metadata_terms(terms, *shape, docs, docs)
        o = sa.sparse_attention_trainable(q, k, v, None, st["BQ"], st["BK"], md, bmd)
    return (o.detach(), *torch.autograd.grad(o, (q, k, v), st["do"]))


def work(case: dict) -> dict:
    """q, k, v (and dO, o, gradients) once, of the keys only what some query row of the plane attends, the mask tensor
    where it is read; 4 D operations per attended pair forward, 10 D more for the gradients."""
    B, H, Sq, Sk, D, kind = (case[n] for n in ("B", "H", "Sq", "Sk", "D", "kind"))
    size = 4 if case["dtype"] == "fp32" else 2
    pairs = _attended(case)
    keys = min(Sk, pairs / Sq if Sq <= 32 else Sq + case["window"] if case["mask"] == "window" else Sk)
    rows = B * H * D * size
    train = kind.startswith("train")
    moved = rows * (2 * Sq + 2 * keys) + (rows * (3 * Sq + 4 * keys) if train else 0)
    if kind.endswith("fresh"):
        moved += Sq * Sk * (B if case["mask"] in ("documents", "blocks_batch", "lengths") else 1)
    return {"bytes": float(moved), "flops": float(B * H * pairs * D * (14 if train else 4))}


def tolerance(case: dict) -> dict:
    return TOLERANCE["train" if case["kind"].startswith("train") else "forward", case["dtype"]]


# Four times the distance (relative 2-norm, largest difference) that outputs and gradients showed from the same function
# in float64, over all kinds of case: 3.8e-7 / 3.4e-6 in fp32, 2.9e-3 / 3.6e-2 and 3.2e-3 / 9.4e-2 in bf16 (an output's
# own rounding is 1.7e-3 of it), 3.1e-4 / 3.9e-3 and 3.8e-4 / 1.1e-2 in fp16.
TOLERANCE = {
    ("forward", "fp32"): {"rel": 1.5e-6, "max": 1.5e-5},
    ("forward", "bf16"): {"rel": 1e-2, "max": 0.15},
    ("forward", "fp16"): {"rel": 1.3e-3, "max": 0.018},
    ("train", "bf16"): {"rel": 1.3e-2, "max": 0.4},
    ("train", "fp16"): {"rel": 1.6e-3, "max": 0.045},
}


# ---- more cases of the same ranges --------------------------------------------------------------------------------
def _between(r: random.Random, lo: float, hi: float) -> int:
    """Uniform over the logarithm."""
    return int(round(math.exp(r.uniform(math.log(lo), math.log(hi)))))


def _whole(r: random.Random, lo: int, hi: int, unit: int) -> int:
    return max(unit, _between(r, lo, hi) // unit * unit)


def _draw_once(r: random.Random) -> dict:
    kind = r.choice(["forward", "forward", "forward", "forward_fresh", "forward_fresh", "tiled", "train", "train",
                     "train_terms", "decode", "decode", "decode_fresh"])
    c = dict(kind=kind, B=_between(r, 1, 8), H=r.choice([4, 8, 12, 16, 16, 24, 32, 32]),
             D=r.choice([64, 128, 128, 128]), dtype=r.choice(["bf16", "bf16", "bf16", "fp16"]),
             layout=r.choice(["bhsd", "bhsd", "bshd"]))
    if kind in ("decode", "decode_fresh"):
        c["BK"] = r.choice([32, 64, 128, 128])
        c["Sq"], c["Sk"] = r.choice([1, 1, 1, 2, 4, 8, 16, 32]), _whole(r, 512, 32768, 512)
        c["mask"] = r.choice(["all", "causal", "window_sinks"]) if kind == "decode" else "lengths"
        if c["mask"] == "window_sinks":
            c.update(window=r.choice([512, 1024, 4096]), p=r.choice([0.5, 0.75, 0.9]))
        return c
    c["BQ"], c["BK"] = r.choice([128, 128, 128, 64]), r.choice([32, 64, 64, 128])
    if kind == "forward" and r.random() < 0.1:
        c.update(dtype="fp32", B=_between(r, 1, 4), BQ=64, BK=32)
    S = _whole(r, 256, 16384, 128)
    if kind == "tiled":
        S = _between(r, 200, 6000)
        c["D"] = r.choice([64, 80, 96, 128])
    if kind == "train" and r.random() < 0.3:
        S = max(160, S - 32 * r.randint(1, 3))  # no multiple of the gradient kernels' 128 rows
        c.update(BQ=32, BK=32)
    c["Sq"] = c["Sk"] = S
    if kind == "forward" and r.random() < 0.3:
        c["Sq"], c["Sk"] = _whole(r, 128, 2048, 128), _whole(r, 2048, 32768, 1024)
        c["mask"] = r.choice(["causal", "causal", "window"])
    elif kind == "train_terms":
        c["mask"] = "documents"
    else:
        c["mask"] = r.choice(["causal", "causal", "window", "documents", "blocks", "blocks_batch"])
    if c["mask"].startswith("blocks"):
        c.update(block=r.choice([32, 64, 128]), p=r.choice([0.25, 0.5, 0.75, 0.9]))
        if S % 128:
            c["block"] = 32
        if S % 32:
            c["mask"] = "documents"
    if c["mask"] == "window":
        c["window"] = _between(r, 100, 4096)
    if c["mask"] == "documents":
        c.update(lo=r.choice([32, 64, 256]), hi=r.choice([512, 1024, 4096]))
    return c


#: what a drawn case may cost: the largest listed ones' operations (train_causal) and bytes (decode_long)
MOST_FLOPS, MOST_BYTES = 1.9e12, 4.3e9


def draw(rng: random.Random) -> dict:
    while True:
        c = _draw_once(rng)
        w = work(c)
        planes = c["B"] if c["mask"] in ("documents", "blocks_batch") else 1
        flops = w["flops"] * (16 if c["dtype"] == "fp32" else 1)  # (the float32 matrix rate is a sixteenth)
        if flops <= MOST_FLOPS and w["bytes"] <= MOST_BYTES and planes * c["Sq"] * c["Sk"] <= 2 ** 30:
            return c
