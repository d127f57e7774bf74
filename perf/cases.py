"""Performance cases of the flash_evict public API: the calls a program makes once per layer.

Three kinds of call, each through the package's entry points:

  evict    `evict(q, k, v, budget, ...)`: exact attention, replay importance, selection
           (or `prefill(score=False)`, the same attention without importance)
  snap     `snap_scores` + `snap_select`: the SnapKV baseline's selection
  compact  `select_tokens` + `gather_tokens` of K and V: one layer's cache cut to a budget
           from stored importance, as a controller's compress() does

`listed()` holds one case per situation, `draw(rng)` makes more of the same ranges, and
`exact(case, seed)` computes the same results in 64 bits with plain torch.

q and k of the evict and snap cases share one direction that some keys have more of (about one
logit of spread per key): attention then prefers some tokens over others, as in trained models,
and importance scores spread over orders of magnitude instead of lying within a few percent.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flash-evict-prefill_amd"))

from flash_evict import evict, gather_tokens, prefill, select_tokens  # noqa: E402
from flash_evict.baselines import snap_scores, snap_select  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}


def _evict(name, B, Hq, Hkv, N, D, dtype="bf16", **kw):
    case = {"name": name, "kind": "evict", "B": B, "Hq": Hq, "Hkv": Hkv, "N": N, "D": D, "dtype": dtype,
            "layout": "bhnd", "causal": True, "score": True, "value_weighted": True, "budget": -(-N // 10),
            "decay": 0.0, "window": 0, "recent": 0, "pool": 1, "qk_scale": 1.0, "outliers": 0}
    case.update(kw)
    return case


def listed():
    return [
        # the smallest layer: latency, host work and launches
        _evict("tiny_512", 1, 4, 4, 512, 64, "f16", budget=64),
        # two short prompts of ragged length at a head dim between the tile sizes
        _evict("ragged_d80", 2, 12, 4, 1531, 80, "f16", layout="bnhd", budget=256, recent=32),
        # the reference benchmark's default heads at 8K, every row replayed
        _evict("harness_8k_d64", 1, 4, 2, 8192, 64),
        # non-causal grouped attention over [B,N,H,D] views with peaked logits, plain attention mass
        _evict("noncausal_4000", 2, 8, 2, 4000, 128, "f16", layout="bnhd", causal=False, value_weighted=False, qk_scale=2.0),
        # Llama-3-8B-shaped layer, outlier channels, recency decay
        _evict("llama_8k", 1, 32, 8, 8192, 128, outliers=4, budget=1024, decay=0.1, recent=64),
        # Qwen-shaped layer from a model's [B,N,H,D] projections, every row replayed
        _evict("qwen_8k_full", 1, 28, 4, 8192, 128, layout="bnhd"),
        # a wide-head layer at the largest head dim
        _evict("wide_d256", 1, 16, 4, 6000, 256, decay=0.05, budget=1024, recent=64),
        # Qwen-shaped long prompt, short observation window, pooled selection
        _evict("qwen_32k_w128", 1, 28, 4, 32768, 128, budget=2048, window=128, recent=64, pool=5),
        # the headline layer
        _evict("headline_32k", 1, 32, 8, 32768, 128, budget=1024, decay=0.1, recent=64),
        # the long-context layer
        _evict("long_131k", 1, 32, 8, 131072, 128, budget=1024, decay=0.1, recent=64),
        # SnapKV's selection for a 32K prompt
        {"name": "snap_32k", "kind": "snap", "B": 1, "Hq": 28, "Hkv": 4, "N": 32768, "D": 128, "dtype": "bf16",
         "layout": "bnhd", "budget": 1024, "window": 32},
        # one layer's 128K cache cut to a tenth
        {"name": "compact_131k", "kind": "compact", "B": 1, "Hkv": 8, "N": 131072, "D": 128, "dtype": "bf16",
         "layout": "bnhd", "budget": 13108, "recent": 64, "pool": 1},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["evict"] * 7 + ["snap", "compact", "compact"])
    dtype = rng.choice(["bf16", "bf16", "f16"])
    layout = rng.choice(["bhnd", "bnhd"])
    if kind == "compact":
        n = _log_int(rng, 2048, 131072)
        return {"kind": kind, "B": rng.choice([1, 1, 2]), "Hkv": rng.choice([2, 4, 8]), "N": n,
                "D": rng.choice([64, 80, 128, 128, 256]), "dtype": dtype, "layout": layout,
                "budget": max(64, int(n * rng.choice([0.02, 0.1, 0.5]))), "recent": rng.choice([0, 32, 64]),
                "pool": rng.choice([1, 1, 5, 7])}
    hkv = rng.choice([1, 2, 4, 8])
    if kind == "snap":
        n = _log_int(rng, 2048, 65536)
        return {"kind": kind, "B": 1, "Hq": hkv * rng.choice([2, 4, 7]), "Hkv": hkv, "N": n,
                "D": rng.choice([64, 128, 128]), "dtype": dtype, "layout": layout,
                "budget": rng.choice([256, 512, 1024]), "window": rng.choice([16, 32, 64, 128])}
    d = rng.choice([64, 64, 64, 128, 128, 128, 128, 128, 128, 32, 80, 96, 100, 160, 192, 256])
    n = _log_int(rng, 300, 32768 if d <= 128 else 12288)
    hq = hkv * rng.choice([1, 2, 4, 4, 7])
    return _evict("", rng.choice([1, 1, 1, 2]) if hq <= 16 else 1, hq, hkv, n, d, dtype, layout=layout,
                  causal=rng.random() < 0.85, score=rng.random() < 0.9, value_weighted=rng.random() < 0.8,
                  budget=max(64, -(-n // rng.choice([8, 10, 20]))), decay=rng.choice([0.0, 0.0, 0.01, 0.1]),
                  window=rng.choice([0, 0, 0, 32, 128]), recent=rng.choice([0, 32, 64]), pool=rng.choice([1, 1, 5]),
                  qk_scale=rng.choice([1.0, 1.0, 2.0]))


def _randn(gen, b, h, n, d, layout, dtype):
    """N(0,1) [B,H,N,D]; "bnhd": a transposed view of contiguous [B,N,H,D] projections."""
    shape = (b, n, h, d) if layout == "bnhd" else (b, h, n, d)
    x = torch.randn(shape, device="cuda", generator=gen, dtype=dtype)
    return x.transpose(1, 2) if layout == "bnhd" else x


def _qkv(case, gen):
    b, hq, hk, n, d = case["B"], case["Hq"], case["Hkv"], case["N"], case["D"]
    dt = DTYPES[case["dtype"]]
    q = _randn(gen, b, hq, n, d, case["layout"], dt)
    k = _randn(gen, b, hk, n, d, case["layout"], dt)
    v = _randn(gen, b, hk, n, d, case["layout"], dt)
    u = torch.nn.functional.normalize(torch.randn(d, device="cuda", generator=gen), dim=0) * d ** 0.25
    sal = torch.randn((b, hk, n, 1), device="cuda", generator=gen)
    q += u.to(dt)
    k += (sal * u).to(dt)
    if case.get("outliers"):
        ch = torch.randperm(d, generator=gen, device="cuda")[: case["outliers"]]
        q[..., ch] *= 8
        k[..., ch] *= 8
    if case.get("qk_scale", 1.0) != 1.0:
        q *= case["qk_scale"]
    return q, k, v


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if case["kind"] == "compact":
        dt = DTYPES[case["dtype"]]
        shape = (case["B"], case["Hkv"], case["N"], case["D"])
        importance = torch.exp(1.5 * torch.randn(shape[:3], device="cuda", generator=gen))
        return {"case": case, "importance": importance, "k": _randn(gen, *shape, case["layout"], dt),
                "v": _randn(gen, *shape, case["layout"], dt)}
    q, k, v = _qkv(case, gen)
    return {"case": case, "q": q, "k": k, "v": v}


def run(state):
    c = state["case"]
    if c["kind"] == "compact":
        idx, keep = select_tokens(state["importance"], min(c["budget"], c["N"]), recent=c["recent"], pool_kernel=c["pool"])
        return {"indices": idx, "keep": keep, "k": gather_tokens(state["k"], idx), "v": gather_tokens(state["v"], idx)}
    if c["kind"] == "snap":
        scores = snap_scores(state["q"], state["k"], c["window"])
        idx, keep = snap_select(scores, c["budget"], c["window"])
        return {"scores": scores, "indices": idx, "keep": keep}
    kw = {"causal": c["causal"], "value_weighted": c["value_weighted"], "recency_decay": c["decay"],
          "observation_window": c["window"]}
    if not c["score"]:
        return {"out": prefill(state["q"], state["k"], state["v"], score=False, causal=c["causal"])[0]}
    out, importance, idx, evicted = evict(state["q"], state["k"], state["v"], min(c["budget"], c["N"]),
                                          reserved_recent=c["recent"], pool_kernel=c["pool"], **kw)
    return {"out": out, "importance": importance, "indices": idx, "evicted": evicted}


def _replayed(case):
    """Query rows whose recency weight is not zero in 32 bits."""
    rows = min(case["N"], case["window"] or case["N"])
    return min(rows, math.ceil(105.0 / case["decay"])) if case["decay"] > 0 else rows


def work(case):
    b, hk, n, d = case["B"], case["Hkv"], case["N"], case["D"]
    if case["kind"] == "compact":
        kept = min(case["budget"], n)
        return {"bytes": b * hk * (n * 4 + n + kept * 8 + 2 * kept * d * 2 * 2), "flops": 0}
    hq = case["Hq"]
    if case["kind"] == "snap":
        w = min(case["window"], n)
        return {"bytes": 2 * d * (b * hk * n + b * hq * w) + b * hk * (n * 4 + n + min(case["budget"], n) * 8),
                "flops": 2 * d * b * hq * w * n}
    r = _replayed(case) if case["score"] else 0
    if case["causal"]:
        pairs, replay = n * (n + 1) // 2, r * (2 * n - r + 1) // 2
    else:
        pairs, replay = n * n, r * n
    nbytes = 2 * d * b * n * (2 * hq + 2 * hk) + (b * hk * (n * 4 + n + min(case["budget"], n) * 8) if case["score"] else 0)
    return {"bytes": nbytes, "flops": b * hq * d * (4 * pairs + 2 * replay)}


def tolerance(case):
    if case["kind"] == "compact":
        return "exact"
    if case["kind"] == "snap":
        return {"rel": 1e-5, "differ": 0.01}
    # attention output: probabilities and output rounded to the type (2.1e-3 in bf16 and 2.7e-4 in
    # fp16 against 64 bits); indices: two scores that tie but for the order of their sums
    return {"rel": 8e-3 if case["dtype"] == "bf16" else 1e-3, "differ": 0.01}


def _exact_evict(case, q, k, v):
    b, hq, n, d = q.shape
    hk = k.shape[1]
    g = hq // hk
    rows = _replayed(case) if case["score"] else 0
    out = torch.empty((b, hq, n, d), dtype=torch.float64, device=q.device)
    imp = torch.zeros((b, hk, n), dtype=torch.float64, device=q.device)
    block = max(32, min(n, (1 << 28) // (8 * n)))
    for i in range(b):
        for j in range(hk):
            kj, vj = k[i, j].double(), v[i, j].double()
            for h in range(j * g, (j + 1) * g):
                for lo in range(0, n, block):
                    hi = min(n, lo + block)
                    end = hi if case["causal"] else n
                    s = (q[i, h, lo:hi].double() * d ** -0.5) @ kj[:end].T
                    if case["causal"]:
                        pos = torch.arange(lo, hi, device=q.device)[:, None]
                        s[:, lo:].masked_fill_(torch.arange(lo, end, device=q.device)[None] > pos, -math.inf)
                    s -= s.amax(1, keepdim=True)
                    s.exp_()
                    s /= s.sum(1, keepdim=True)
                    out[i, h, lo:hi] = s @ vj[:end]
                    if hi > n - rows:
                        first = max(lo, n - rows)
                        w = torch.exp(case["decay"] * (torch.arange(first, hi, device=q.device, dtype=torch.float64) - (n - 1)))
                        imp[i, j, :end] += w @ s[first - lo:]
            if case["value_weighted"]:
                imp[i, j] *= vj.abs().sum(1)
    return out, imp


def exact(case, seed):
    if case["kind"] == "compact" or case["kind"] == "evict" and case["N"] > 65536:
        return None
    state = prepare(case, seed)
    q, k = state["q"], state["k"]
    if case["kind"] == "evict":
        out, imp = _exact_evict(case, q, k, state["v"])
        if not case["score"]:
            return {"out": out}
        return {"out": out, "importance": imp, "indices": None, "evicted": None}
    # SnapKV: products rounded to the input type, scaled and masked, softmax, summed over the
    # window's rows, mean over the heads of a group
    b, hq, n, d = q.shape
    hk = k.shape[1]
    g, w = hq // hk, min(case["window"], n)
    scores = torch.zeros((b, hk, n), dtype=torch.float64, device=q.device)
    late = torch.arange(n, device=q.device)[None] > torch.arange(n - w, n, device=q.device)[:, None]
    for i in range(b):
        for h in range(hq):
            s = (q[i, h, n - w:].double() @ k[i, h // g].double().T).to(q.dtype).double() * d ** -0.5
            scores[i, h // g] += torch.softmax(s.masked_fill(late, -math.inf), dim=1).sum(0) / g
    return {"scores": scores, "indices": None, "keep": None}
