"""What the performance of the paged-KV path is measured on.

Every case is one call (or one layer's worth of calls) that a serving program makes through
the package's public entry points:

* ``decode``: ``paged_decode_attention`` over one layer's pool, one new token per sequence;
* ``prefix``: the step of sequences that share a prompt prefix -- the copy-on-write of their
  last shared block, then append and cascade decode through ``layers.paged_attention``;
* ``prefill``: ``paged_prefill_attention`` over prompt chunks, with or without cached prefixes;
* ``mixed``: a chunked-prefill step with decode rows through ``layers.paged_attention`` (append,
  decode kernel, prefill kernel), as every layer of a model calls it on the step's one batch;
* ``elementwise``: RMSNorm, RoPE on the projection's q and k, and SiLU x up of one layer.

A case holds sizes only. Context and chunk lengths follow from its ``lens`` (so the work is the
case's, whatever the seed); values, block placement and pools follow from the seed. Values are
N(0, 1), blocks of 16 tokens are scattered over the pool, and the last block of a sequence is
partly filled, as the engine's allocator leaves them.
"""

from __future__ import annotations

import math
import os
import random
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "inference-engine_amd"))

from engine.kernels import fused  # noqa: E402
from engine.kernels.paged_attention import (  # noqa: E402
    paged_decode_attention,
    paged_prefill_attention,
)
from engine.model import layers  # noqa: E402
from engine.runtime.paged_cache import KVShape, PagedBatch, PagedKVCache  # noqa: E402

BLOCK = 16  # tokens per block: the engine's default, and every workload's of this repository
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def listed() -> list[dict]:
    def decode(name, dtype, heads, kv_heads, head_dim, batch, lo, hi, spread, lens):
        return {"name": name, "kind": "decode", "dtype": dtype, "heads": heads,
                "kv_heads": kv_heads, "head_dim": head_dim, "batch": batch, "lo": lo, "hi": hi,
                "spread": spread, "lens": lens}  # fmt: skip

    return [
        # A few short chats on a 1B-shaped model: latency and launches count.
        decode("decode_small", "fp16", 32, 8, 64, 8, 32, 512, "even", 1),
        # One user far into a long document (8B shape): one sequence for the whole GPU.
        decode("decode_one_long", "bf16", 32, 8, 128, 1, 20011, 20011, "even", 1),
        # Many short chats (1B shape): the usual load of a small model's server.
        decode("decode_many_short", "bf16", 32, 8, 64, 64, 1, 1500, "even", 1),
        # The 3B-shaped decode step that the benchmark times.
        decode("decode_3b", "bf16", 24, 8, 128, 64, 1024, 4096, "even", 1),
        # Long and short contexts in one batch (8B shape), log-uniform up to 32k.
        decode("decode_skewed", "bf16", 32, 8, 128, 32, 128, 32768, "log", 1),
        # Eight query heads per KV head, the widest usual group of large models.
        decode("decode_wide_groups", "bf16", 64, 8, 128, 48, 256, 4096, "even", 1),
        # 256 sequences behind one system prompt, 64 of them copying its last block (3B shape).
        {"name": "prefix_step", "kind": "prefix", "dtype": "bf16", "heads": 24, "kv_heads": 8,
         "head_dim": 128, "batch": 256, "shared": 128, "tail": 1024, "copies": 64, "lens": 1},
        # A chunked-prefill step beside 120 decoding sequences (8B shape), append included.
        {"name": "mixed_step", "kind": "mixed", "dtype": "bf16", "heads": 32, "kv_heads": 8,
         "head_dim": 128, "chunks": 4, "q_lo": 512, "q_hi": 512, "prefix_step": 1024,
         "prefix_hi": 0, "batch": 120, "lo": 256, "hi": 2048, "spread": "even", "lens": 1},
        # One long prompt read from its start (8B shape): the matrix cores' own case.
        {"name": "prefill_long", "kind": "prefill", "dtype": "bf16", "heads": 32, "kv_heads": 8,
         "head_dim": 128, "chunks": 1, "q_lo": 6011, "q_hi": 6011, "prefix_step": 0,
         "prefix_hi": 0, "lens": 1},
        # Twelve ragged prompts, some behind cached prefixes, on a 1B-shaped fp16 model.
        {"name": "prefill_ragged", "kind": "prefill", "dtype": "fp16", "heads": 32,
         "kv_heads": 8, "head_dim": 64, "chunks": 12, "q_lo": 3, "q_hi": 600, "prefix_step": 0,
         "prefix_hi": 3000, "lens": 1},
        # The same kind of step on an fp32 model, as token-exactness checks run it.
        {"name": "mixed_fp32", "kind": "mixed", "dtype": "fp32", "heads": 32, "kv_heads": 8,
         "head_dim": 64, "chunks": 3, "q_lo": 60, "q_hi": 300, "prefix_step": 0,
         "prefix_hi": 700, "batch": 16, "lo": 32, "hi": 1500, "spread": "even", "lens": 1},
        # What stands around attention in a layer, on a chunked step's tokens (8B shape).
        {"name": "elementwise", "kind": "elementwise", "dtype": "bf16", "heads": 32,
         "kv_heads": 8, "head_dim": 128, "hidden": 4096, "inner": 14336, "tokens": 2168},
    ]  # fmt: skip


def _spread(rng: random.Random, lo: float, hi: float) -> int:
    """A whole number from lo to hi, even over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["decode"] * 9 + ["prefill"] * 4 + ["mixed"] * 3 + ["prefix"] * 2 + ["elementwise"] * 2)
    lens = rng.randrange(1 << 30)
    kv_heads = rng.choice([2, 4, 8, 8])
    head_dim = rng.choice([64, 128])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    if kind == "elementwise":
        heads = kv_heads * rng.choice([1, 2, 3, 4, 8])
        return {"kind": kind, "dtype": dtype, "heads": heads, "kv_heads": kv_heads,
                "head_dim": head_dim, "hidden": rng.choice([2048, 3072, 4096]),
                "inner": rng.choice([5632, 8192, 14336]), "tokens": _spread(rng, 1, 2168)}  # fmt: skip
    if kind == "decode":
        heads = kv_heads * rng.choice([1, 2, 3, 4, 4, 5, 6, 7, 8])
        hi = _spread(rng, 64, 32768)
        batch = _spread(rng, 1, 256)
        # no more K/V than the largest listed case reads
        batch = max(1, min(batch, 64 * 2560 * 8 * 128 // (hi * kv_heads * head_dim)))
        return {"kind": kind, "dtype": dtype, "heads": heads, "kv_heads": kv_heads,
                "head_dim": head_dim, "batch": batch, "lo": rng.randint(1, hi), "hi": hi,
                "spread": rng.choice(["even", "log"]), "lens": lens}  # fmt: skip
    if kind == "prefix":
        batch = _spread(rng, 16, 256)
        return {"kind": kind, "dtype": dtype, "heads": kv_heads * rng.choice([2, 3, 4]),
                "kv_heads": kv_heads, "head_dim": head_dim, "batch": batch,
                "shared": rng.randint(17, 128), "tail": _spread(rng, 16, 1024),
                "copies": rng.randint(1, batch // 2), "lens": lens}  # fmt: skip
    fp32 = rng.random() < 0.2
    heads = kv_heads * rng.choice([1, 2, 3, 4, 5, 7, 8])
    q_hi = _spread(rng, 8, 300 if fp32 else 3000)
    chunks = rng.randint(1, max(1, min(12, (900 if fp32 else 3000) // q_hi)))
    case = {"kind": kind, "dtype": "fp32" if fp32 else dtype, "heads": min(heads, 32),
            "kv_heads": kv_heads if heads <= 32 else 4, "head_dim": 64 if fp32 else head_dim,
            "chunks": chunks, "q_lo": rng.randint(2, q_hi), "q_hi": q_hi, "prefix_step": 0,
            "prefix_hi": rng.choice([0, _spread(rng, 16, 1000 if fp32 else 3000)]),
            "lens": lens}  # fmt: skip
    if kind == "mixed":
        hi = _spread(rng, 64, 1500 if fp32 else 2048)
        case.update(batch=_spread(rng, 1, 16 if fp32 else 120), lo=rng.randint(1, hi), hi=hi,
                    spread="even")  # fmt: skip
    return case


def _contexts(case: dict) -> list[int]:
    """The decoding sequences' context lengths, the new token included."""
    rng = random.Random(case["lens"])
    lo, hi = case["lo"], case["hi"]
    if case["spread"] == "log":
        return [_spread(rng, lo, hi) for _ in range(case["batch"])]
    return [rng.randint(lo, hi) for _ in range(case["batch"])]


def _chunks(case: dict) -> list[tuple[int, int]]:
    """Every prompt chunk as (new tokens, cached tokens before them)."""
    rng = random.Random(case["lens"] + 1)
    return [(rng.randint(case["q_lo"], case["q_hi"]),
             i * case["prefix_step"] + rng.randint(0, case["prefix_hi"]))
            for i in range(case["chunks"])]  # fmt: skip


def _inputs(case: dict, seed: int) -> dict:
    """Tables, lengths and tensors of a case, from the seed alone."""
    dev, dt = torch.device("cuda"), DTYPES[case["dtype"]]
    gen = torch.Generator(device=dev).manual_seed(seed)
    order = random.Random(seed)

    def randn(*shape):
        return torch.randn(shape, generator=gen, device=dev, dtype=dt)

    nh, nkv, hd = case["heads"], case["kv_heads"], case["head_dim"]
    if case["kind"] == "elementwise":
        n = case["tokens"]
        angle = torch.arange(n, device=dev)[:, None] * 5e5 ** (-torch.arange(0, hd, 2, device=dev) / hd)
        angle = torch.cat([angle, angle], dim=-1).float()
        return {"x": randn(n, case["hidden"]), "w": randn(case["hidden"]),
                "qkv": randn(n, nh + 2 * nkv, hd), "cos": angle.cos(), "sin": angle.sin(),
                "gate": randn(n, case["inner"]), "up": randn(n, case["inner"])}  # fmt: skip
    x: dict = {"ctx": [], "new": []}
    if case["kind"] in ("prefill", "mixed"):
        for new, cached in _chunks(case):
            x["ctx"].append(cached + new)
            x["new"].append(new)
    if case["kind"] in ("decode", "mixed"):
        x["ctx"] += _contexts(case)
        x["new"] += [1] * case["batch"]
    if case["kind"] == "prefix":
        rng = random.Random(case["lens"])
        x["ctx"] = [case["shared"] * BLOCK + rng.randint(1, case["tail"] + 1) for _ in range(case["batch"])]
        x["new"] = [1] * case["batch"]
    need = [-(-n // BLOCK) for n in x["ctx"]]
    total = case["shared"] + sum(n - case["shared"] for n in need) + case["copies"] \
        if case["kind"] == "prefix" else sum(need)  # fmt: skip
    blocks = total + total // 4 + 1  # a pool that is not quite full
    free = list(range(blocks))
    order.shuffle(free)
    if case["kind"] == "prefix":
        prefix = [free.pop() for _ in range(case["shared"])]
        x["tables"] = [prefix + [free.pop() for _ in range(n - case["shared"])] for n in need]
        pairs = []
        for row in x["tables"][: case["copies"]]:
            pairs.append((row[case["shared"] - 1], free.pop()))
            row[case["shared"] - 1] = pairs[-1][1]
        x["pairs"] = torch.tensor(pairs, dtype=torch.int64, device=dev)
    else:
        x["tables"] = [[free.pop() for _ in range(n)] for n in need]
    x["blocks"] = blocks
    x["k"], x["v"] = randn(blocks * BLOCK, nkv, hd), randn(blocks * BLOCK, nkv, hd)
    x["q"] = randn(sum(x["new"]), nh, hd)
    if case["kind"] in ("prefix", "mixed"):
        x["new_k"], x["new_v"] = randn(sum(x["new"]), nkv, hd), randn(sum(x["new"]), nkv, hd)
    return x


def _table_tensor(rows: list[list[int]], width: int) -> torch.Tensor:
    return torch.tensor([r + [0] * (width - len(r)) for r in rows], dtype=torch.int32, device="cuda")


def prepare(case: dict, seed: int) -> dict:
    x = _inputs(case, seed)
    s: dict = {"kind": case["kind"]}
    if case["kind"] == "elementwise":
        return s | x | {"heads": case["heads"], "kv_heads": case["kv_heads"]}
    s["q"] = x["q"]
    if case["kind"] in ("decode", "prefill"):
        # the engine's tables are as wide as the longest context it admits
        width = -(-case["hi"] // BLOCK) if case["kind"] == "decode" else max(map(len, x["tables"]))
        s["k"], s["v"] = x["k"], x["v"]
        s["tables"] = _table_tensor(x["tables"], width)
        s["ctx"] = torch.tensor(x["ctx"], dtype=torch.int32, device="cuda")
        if case["kind"] == "prefill":
            offsets = [0]
            for n in x["new"]:
                offsets.append(offsets[-1] + n)
            s["cu_q"] = torch.tensor(offsets, dtype=torch.int32, device="cuda")
            s["longest"] = max(x["new"])
        return s
    # The pool and the step's batch, which a model builds once for all its layers.
    cache = PagedKVCache(KVShape(1, case["kv_heads"], case["head_dim"]), x["blocks"], BLOCK,
                         "cuda", DTYPES[case["dtype"]])  # fmt: skip
    cache.k[0].copy_(x["k"])
    cache.v[0].copy_(x["v"])
    s["cache"], s["new_k"], s["new_v"] = cache, x["new_k"], x["new_v"]
    s["batch"] = PagedBatch.build(cache, x["tables"], x["ctx"], x["new"], "cuda", use_kernel=True,
                                  cascade=case["kind"] == "prefix", num_heads=case["heads"])  # fmt: skip
    s["pairs"] = x.get("pairs")
    return s


def run(s: dict):
    if s["kind"] == "decode":
        return paged_decode_attention(s["q"], s["k"], s["v"], s["tables"], s["ctx"], BLOCK)
    if s["kind"] == "prefill":
        return paged_prefill_attention(s["q"], s["k"], s["v"], s["tables"], s["ctx"], BLOCK,
                                       s["cu_q"], s["longest"])  # fmt: skip
    if s["kind"] == "elementwise":
        normed = fused.rms_norm(s["x"], s["w"], 1e-5)
        qkv = s["qkv"].clone()  # stands for the projection's fresh output: RoPE is in place
        nh, nkv = s["heads"], s["kv_heads"]
        fused.rope_(qkv[:, :nh], s["cos"], s["sin"])
        fused.rope_(qkv[:, nh : nh + nkv], s["cos"], s["sin"])
        return normed, qkv, fused.silu_mul(s["gate"], s["up"])
    cache = s["cache"]
    if s["pairs"] is not None:
        cache.copy_blocks(s["pairs"])
    out = layers.paged_attention(0, s["q"], s["new_k"], s["new_v"], s["batch"])
    return out, cache.k, cache.v


def work(case: dict) -> dict:
    elt = 4 if case["dtype"] == "fp32" else 2
    nh, nkv, hd = case["heads"], case["kv_heads"], case["head_dim"]
    if case["kind"] == "elementwise":
        n, rot = case["tokens"], nh + nkv
        values = 2 * n * case["hidden"] + case["hidden"] + 2 * n * (rot + nkv) * hd + 3 * n * case["inner"]
        flops = n * (6 * case["hidden"] + 6 * rot * hd + 5 * case["inner"])
        return {"bytes": values * elt + 2 * n * hd * 4, "flops": flops}
    token = 2 * nkv * hd * elt  # one token's K and V
    pairs = rows = keys = 0  # (query, visible key) pairs, query rows, keys read
    moved = 0  # appended rows and copied blocks
    if case["kind"] in ("prefill", "mixed"):
        for new, cached in _chunks(case):
            pairs += new * cached + new * (new + 1) // 2
            rows += new
            keys += cached + new
    if case["kind"] in ("decode", "mixed"):
        ctx = _contexts(case)
        pairs, rows, keys = pairs + sum(ctx), rows + len(ctx), keys + sum(ctx)
    if case["kind"] == "prefix":
        rng = random.Random(case["lens"])
        tails = [rng.randint(1, case["tail"] + 1) for _ in range(case["batch"])]
        rows = len(tails)
        pairs = sum(tails) + rows * case["shared"] * BLOCK
        # every block once: the shared prefix, the copies, the private tails
        keys = sum(tails) + (case["shared"] + case["copies"]) * BLOCK
        moved = (1 + case["copies"]) * BLOCK * token
    if case["kind"] in ("prefix", "mixed"):
        moved += 2 * rows * token
    return {"bytes": keys * token + 2 * rows * nh * hd * elt + moved, "flops": 4 * pairs * nh * hd}


def tolerance(case: dict):
    # RMSNorm, RoPE and SiLU x up promise the bits of the PyTorch ops that they replace.
    if case["kind"] == "elementwise":
        return "exact"
    # Attention sums in fp32 whatever the cache holds; the result is rounded to the cache's
    # type. About four times the distance from the same call in 64 bits.
    return {"rel": {"bf16": 7e-3, "fp16": 1.2e-3, "fp32": 2e-6}[case["dtype"]]}


def _attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> torch.Tensor:
    """q [n, nh, hd], the last n of the tokens of k, v [c, nkv, hd], all float64."""
    n, nh, hd = q.shape
    c, nkv = k.shape[:2]
    kt, vt = k.permute(1, 2, 0).contiguous(), v.transpose(0, 1).contiguous()
    key = torch.arange(c, device=q.device)
    out = torch.empty_like(q)
    for lo in range(0, n, 512):  # some rows at a time: the scores are large
        part = q[lo : lo + 512]
        m = part.shape[0]
        rows = part.view(m, nkv, nh // nkv, hd).permute(1, 0, 2, 3).reshape(nkv, -1, hd)
        s = (rows @ kt).view(nkv, m, nh // nkv, c) * hd**-0.5
        last = c - n + lo + torch.arange(m, device=q.device)
        s.masked_fill_((key[None] > last[:, None])[None, :, None], -math.inf)
        o = torch.softmax(s, -1).view(nkv, -1, c) @ vt
        out[lo : lo + 512] = o.view(nkv, m, nh // nkv, hd).permute(1, 0, 2, 3).reshape(m, nh, hd)
    return out


def exact(case: dict, seed: int):
    x = _inputs(case, seed)
    if case["kind"] == "elementwise":
        h = x["x"].double()
        normed = x["w"].double() * h * torch.rsqrt(h.square().mean(-1, keepdim=True) + 1e-5)
        qkv, rot = x["qkv"].double(), case["heads"] + case["kv_heads"]
        p, half = qkv[:, :rot], case["head_dim"] // 2
        turned = torch.cat([-p[..., half:], p[..., :half]], -1)
        turned = p * x["cos"].double()[:, None] + turned * x["sin"].double()[:, None]
        g = x["gate"].double()
        return normed, torch.cat([turned, qkv[:, rot:]], 1), g / (1 + torch.exp(-g)) * x["up"].double()
    k, v = x["k"], x["v"]
    token = torch.arange(BLOCK, device=k.device)
    places = [(torch.tensor(t, device=k.device)[:, None] * BLOCK + token).view(-1)[:n]
              for t, n in zip(x["tables"], x["ctx"], strict=True)]  # fmt: skip
    if case["kind"] == "prefix":
        src, dst = ((x["pairs"][:, j, None] * BLOCK + token).view(-1) for j in (0, 1))
        k[dst], v[dst] = k[src], v[src]
    if "new_k" in x:
        slots = torch.cat([p[-n:] for p, n in zip(places, x["new"], strict=True)])
        k[slots], v[slots] = x["new_k"], x["new_v"]
    out, at = [], 0
    for p, n in zip(places, x["new"], strict=True):
        out.append(_attend(x["q"][at : at + n].double(), k[p].double(), v[p].double()))
        at += n
    out = torch.cat(out)
    if "new_k" not in x:
        return out
    return out.flatten(1), k.double()[None], v.double()[None]
