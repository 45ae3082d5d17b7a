"""The attention path's work as a serving program gives it: which calls are timed, and what they return.

A continuous-batching server over the paged cache makes these calls, layer by layer: it scatters new
tokens' K/V into their pages (with or without the rotary embedding), attends prompts and chunks of
prompts (prefill) and single tokens (decode) to the paged cache, and samples from the logits.  Each
kind of call is here from a handful of tokens up to the largest batches of the benchmark workloads,
in fp16, bf16 and fp32, over the head layouts the package is used with (query / KV heads, head size).

A case holds plain values; the lengths of its sequences come from the case alone (``lengths`` seeds
them), its tensors' values from the seed given to ``prepare``.  The cache's pages are a random
permutation of the pool, as a pool leaves them after serving for a while, and slots no sequence owns
hold stale values of finished ones.
"""
import math
import random

import torch

from ecahlang_amd import ops, sampling
from ecahlang_amd.wrappers import BatchDecodeWithPagedKVCacheWrapper, BatchPrefillWithPagedKVCacheWrapper

DEV = "cuda"
PS = 16  # page size of the serving loop's pool
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
# sampling requests of a mixed batch: (top_k, top_p); 0 and 1.0 leave a filter out
REQUESTS = [(0, 1.0), (50, 0.9), (0, 0.9), (40, 1.0), (20, 0.8), (1, 1.0), (0, 0.95), (100, 0.95)]


def _heads(hq, hkv, d, dtype):
    return {"hq": hq, "hkv": hkv, "d": d, "dtype": dtype}


QWEN3B = _heads(16, 2, 128, "fp16")     # the headline configuration's attention
LLAMA8B = _heads(32, 8, 128, "bf16")    # the long-context configuration's
LLAMA1B = _heads(32, 8, 64, "fp32")     # the fp32 configuration's
GQA7 = _heads(28, 4, 128, "bf16")       # seven query heads a KV head, a common group size


def listed():
    return [
        # The smallest step: four short chats.  plan, then the first layer's append and attention,
        # called eagerly: launches and host work.
        {"name": "decode_b4_short_fp16", "kind": "decode", **QWEN3B, "batch": 4, "lo": 16, "hi": 300, "dist": "uniform",
         "lengths": 11, "append": True, "plan": True},
        # One layer of the headline decode step (64 sequences of 512 to 4096 tokens), its append in the same
        # call; the plan is the step's and shared by its 36 layers.
        {"name": "decode_b64_fp16", "kind": "decode", **QWEN3B, "batch": 64, "lo": 512, "hi": 4096, "dist": "uniform",
         "lengths": 1002, "append": True, "plan": False},
        # One layer of a long-context step: 128 sequences, log-uniform 1k to 32k tokens.
        {"name": "decode_b128_long_bf16", "kind": "decode", **LLAMA8B, "batch": 128, "lo": 1024, "hi": 32768, "dist": "log",
         "lengths": 1004, "append": False, "plan": False},
        # One layer of a decode step over an fp32 cache (a model kept in full precision).
        {"name": "decode_b16_fp32", "kind": "decode", **LLAMA1B, "batch": 16, "lo": 16, "hi": 2048, "dist": "log",
         "lengths": 1001, "append": True, "plan": False},
        # A whole decode step's attention: 36 layers, 128 sequences on one 2048-token system prompt, one graph
        # replay of the plan (prefix read once per group) and every layer's append and attention.
        {"name": "step36_shared_fp16", "kind": "step", **QWEN3B, "layers": 36, "batch": 128, "prefix": 2048, "lo": 64,
         "hi": 1024, "lengths": 1005},
        # A single short prompt: the first token of a chat that starts on an idle server.
        {"name": "prefill_b1_short_fp16", "kind": "prefill", **QWEN3B, "requests": 1, "lo": 37, "hi": 37, "prefix": 0,
         "lengths": 21},
        # Chunked prefill: eight requests' 512-token chunks on prefixes of up to 8192 tokens.
        {"name": "prefill_chunks_fp16", "kind": "prefill", **QWEN3B, "requests": 8, "lo": 512, "hi": 512, "prefix": 8192,
         "lengths": 1003},
        # A batch of new prompts of ragged lengths, nothing cached before them.
        {"name": "prefill_prompts_bf16", "kind": "prefill", **GQA7, "requests": 11, "lo": 20, "hi": 1500, "prefix": 0,
         "lengths": 23},
        # Prompts over an fp32 cache, some with earlier turns cached.
        {"name": "prefill_prompts_fp32", "kind": "prefill", **LLAMA1B, "requests": 6, "lo": 12, "hi": 512, "prefix": 300,
         "lengths": 24},
        # The append of a large prefill batch: 65,536 tokens into scattered pages.
        {"name": "append_bulk_fp16", "kind": "append", **QWEN3B, "tokens": 65536, "requests": 128, "lengths": 31,
         "rope": False},
        # A prefill chunk's rotary embedding and append, an odd number of tokens.
        {"name": "rope_append_bf16", "kind": "append", **LLAMA8B, "tokens": 4003, "requests": 9, "lengths": 32, "rope": True},
        # Sampling for a full batch whose requests ask for different filters, with the serving loop's
        # repetition penalty and temperature.
        {"name": "sample_b128_mixed_fp16", "kind": "sample", "rows": 128, "vocab": 151936, "dtype": "fp16", "mix": "mixed",
         "scale": True, "lengths": 41},
    ]


def _logint(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "step", "prefill", "prefill", "prefill", "append", "sample"])
    seed = {"lengths": rng.randrange(1 << 20)}
    if kind == "sample":
        rows = _logint(rng, 1, 128)
        return {"kind": kind, "rows": rows, "vocab": rng.choice([32000, 50257, 128256, 151936, _logint(rng, 1000, 151936)]),
                "dtype": rng.choice(["fp16", "bf16", "fp32"]) if rows <= 64 else rng.choice(["fp16", "bf16"]),
                "mix": rng.choice(["mixed", "filtered", "open"]), "scale": rng.random() < 0.5, **seed}
    heads = rng.choice([QWEN3B, QWEN3B, LLAMA8B, GQA7, _heads(12, 2, 128, "fp16"), _heads(14, 2, 64, "bf16"),
                        _heads(40, 8, 128, "fp16"), _heads(32, 8, 64, "bf16"), _heads(24, 8, 128, "bf16"),
                        _heads(16, 16, 64, "fp16"), LLAMA1B, _heads(16, 2, 128, "fp32")])
    es = 4 if heads["dtype"] == "fp32" else 2
    if kind == "decode":
        batch = _logint(rng, 1, 256 if es == 2 else 64)
        hi = _logint(rng, 32, 32768 if es == 2 else 4096)
        # at most about as many bytes as the long-context case
        most = 2_000_000_000 if es == 2 else 200_000_000
        hi = max(32, min(hi, most // (batch * 2 * heads["hkv"] * heads["d"] * es)))
        return {"kind": kind, **heads, "batch": batch, "lo": max(1, hi // rng.choice([1, 4, 16, 32])), "hi": hi,
                "dist": rng.choice(["uniform", "log"]), "append": rng.random() < 0.5, "plan": rng.random() < 0.3, **seed}
    if kind == "step":
        return {"kind": kind, **rng.choice([QWEN3B, _heads(12, 2, 128, "fp16")]), "layers": rng.choice([4, 8, 12]),
                "batch": _logint(rng, 4, 128), "prefix": _logint(rng, 256, 2048), "lo": 64, "hi": _logint(rng, 80, 1024), **seed}
    if kind == "prefill":
        if es == 4:
            hi = _logint(rng, 8, 384)
            return {"kind": kind, **heads, "requests": rng.randint(1, 5), "lo": max(1, hi // 16), "hi": hi,
                    "prefix": rng.choice([0, 0, _logint(rng, 16, 300)]), **seed}
        if rng.random() < 0.5:  # new prompts
            hi = _logint(rng, 16, 1500)
            return {"kind": kind, **heads, "requests": rng.randint(1, 8), "lo": max(1, hi // 32), "hi": hi, "prefix": 0, **seed}
        hi = _logint(rng, 64, 512)  # chunks
        return {"kind": kind, **heads, "requests": rng.randint(1, 4), "lo": hi if rng.random() < 0.5 else max(1, hi // 4),
                "hi": hi, "prefix": _logint(rng, 64, 2048), **seed}
    rope = rng.random() < 0.5
    tokens = _logint(rng, 1, 8192 if rope or es == 4 else 32768)
    return {"kind": kind, **heads, "tokens": tokens, "requests": max(1, min(tokens, _logint(rng, 1, 128))), "rope": rope, **seed}


# ---------------------------------------------------------------- lengths and page tables

def _spread(rng, n, lo, hi, dist):
    if dist == "log":
        return [_logint(rng, lo, hi) for _ in range(n)]
    return [rng.randint(lo, hi) for _ in range(n)]


def _lengths(case):
    """(tokens per sequence, new tokens per sequence), from the case alone."""
    rng = random.Random(case["lengths"])
    if case["kind"] == "decode":
        kv = [c + 1 for c in _spread(rng, case["batch"], case["lo"], case["hi"], case["dist"])]
        return kv, [1] * len(kv)
    if case["kind"] == "step":
        kv = [case["prefix"] + c + 1 for c in _spread(rng, case["batch"], case["lo"], case["hi"], "uniform")]
        return kv, [1] * len(kv)
    if case["kind"] == "prefill":
        new = _spread(rng, case["requests"], case["lo"], case["hi"], "log")
        return [n + (rng.randint(0, case["prefix"]) if case["prefix"] else 0) for n in new], new
    cuts = sorted(rng.sample(range(1, case["tokens"]), case["requests"] - 1))  # append: a share of the tokens each
    new = [b - a for a, b in zip([0] + cuts, cuts + [case["tokens"]])]
    return [n + rng.randint(0, 100) for n in new], new


def _i32(values):
    return torch.tensor(values, dtype=torch.int32, device=DEV)


def _cumsum(values):
    out = [0]
    for v in values:
        out.append(out[-1] + v)
    return out


def _table(kv, gen, shared=0):
    """indptr, indices, last_page_len and the pool's pages; the first ``shared`` pages of every sequence are the same."""
    npages = [-(-n // PS) for n in kv]
    own = sum(npages) - shared * len(kv) + shared
    pool = own + own // 4 + 1
    perm = torch.randperm(pool, generator=gen, device=DEV)[:own].to(torch.int32)
    if shared:
        at, rows = shared, []
        for n in npages:
            rows += [perm[:shared], perm[at:at + n - shared]]
            at += n - shared
        perm = torch.cat(rows)
    return _i32(_cumsum(npages)), perm, _i32([(n - 1) % PS + 1 for n in kv]), pool


def _randn(gen, shape, dtype, scale=1.0):
    return torch.randn(shape, generator=gen, device=DEV, dtype=dtype).mul_(scale)


# ---------------------------------------------------------------- states

def _inputs(case, seed):
    """Everything but the wrappers: the cache, its table and the call's tensors."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    st = {"case": case}
    if case["kind"] == "sample":
        rows, vocab = case["rows"], case["vocab"]
        # a language model's logits: a wide body and a few likely tokens
        x = torch.randn((rows, vocab), generator=gen, device=DEV) * 2.5
        hot = torch.randint(0, vocab, (rows, 24), generator=gen, device=DEV)
        x.scatter_add_(1, hot, 4 + 10 * torch.rand((rows, 24), generator=gen, device=DEV))
        st["logits"] = x.to(dtype)
        rng = random.Random(case["lengths"])
        pick = {"mixed": REQUESTS, "filtered": [(50, 0.9)], "open": [(0, 1.0)]}[case["mix"]]
        asked = [rng.choice(pick) for _ in range(rows)]
        st["top_k"], st["top_p"] = _i32([k for k, _ in asked]), torch.tensor([p for _, p in asked], device=DEV)
        st["uniform"] = torch.rand(rows, generator=gen, device=DEV)
        if case["scale"]:
            st["penalty"] = torch.ones((rows, vocab), dtype=dtype, device=DEV)
            seen = torch.randint(0, vocab, (rows, 400), generator=gen, device=DEV)
            st["penalty"].scatter_(1, seen, 1.15)
            st["slots"] = torch.randperm(rows, generator=gen, device=DEV).to(torch.int32)
            st["temperature"] = 0.6 + 0.6 * torch.rand(rows, generator=gen, device=DEV)
        return st
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    kv, new = _lengths(case)
    shared = case["prefix"] // PS if case["kind"] == "step" else 0
    st["kv"], st["new"] = kv, new
    st["indptr"], st["indices"], st["last"], pool = _table(kv, gen, shared)
    layers = case.get("layers", 1)
    st["cache"] = _randn(gen, (layers, pool, 2, PS, hkv, d), dtype)
    nnz = sum(new)
    st["q"] = _randn(gen, (layers, nnz, hq, d), dtype)
    st["k"] = _randn(gen, (layers, nnz, hkv, d), dtype)
    st["v"] = _randn(gen, (layers, nnz, hkv, d), dtype)
    if case["kind"] == "step":
        st["shared"] = _i32([0] + [shared] * (len(kv) - 1))
    if case["kind"] in ("prefill", "append"):
        st["qo_indptr"] = _i32(_cumsum(new))
        pos = [torch.arange(n - c, n, dtype=torch.int32) for n, c in zip(kv, new)]
        st["positions"] = torch.cat(pos).to(DEV)
        st["batch_indices"] = torch.repeat_interleave(torch.arange(len(new), dtype=torch.int32), torch.tensor(new)).to(DEV)
    if case.get("rope"):
        # the model's position embeddings of these tokens
        inv = 1.0 / (10000.0 ** (torch.arange(0, d, 2, device=DEV, dtype=torch.float32) / d))
        ang = st["positions"].float()[:, None] * inv[None, :]
        ang = torch.cat([ang, ang], dim=1)
        st["cos"], st["sin"] = ang.cos().to(dtype), ang.sin().to(dtype)
    return st


def _plan(st):
    case = st["case"]
    more = {"kv_shared_pages": st["shared"], "cascade": True} if case["kind"] == "step" else {}
    st["wrapper"].plan(st["indptr"], st["indices"], st["last"], case["hq"], case["hkv"], case["d"], PS,
                       pos_encoding_mode="NONE", q_data_type=DTYPES[case["dtype"]], **more)


def _step(st):
    _plan(st)
    for i in range(st["case"]["layers"]):
        st["wrapper"].run(st["q"][i], st["cache"][i], out=st["out"][i], append_kv=(st["k"][i], st["v"][i]))


def prepare(case, seed):
    st = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("decode", "step"):
        st["wrapper"] = BatchDecodeWithPagedKVCacheWrapper(torch.empty(128 << 20, dtype=torch.uint8, device=DEV), "NHD")
        _plan(st)
    if kind == "step":
        # the serving loop captures its step once per batch size and replays it
        st["out"] = torch.empty_like(st["q"])
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _step(st)
            side.synchronize()
            st["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(st["graph"], stream=side):
                _step(st)
        torch.cuda.current_stream().wait_stream(side)
    if kind == "prefill":
        # the chunk's K/V are in their pages before its attention; one plan serves every layer
        c = st["cache"][0]
        ops.append_paged_kv_cache(st["k"][0], st["v"][0], st["batch_indices"], st["positions"], c, st["indices"],
                                  st["indptr"], st["last"])
        st["wrapper"] = BatchPrefillWithPagedKVCacheWrapper(torch.empty(128 << 20, dtype=torch.uint8, device=DEV), "NHD")
        st["wrapper"].plan(st["qo_indptr"], st["indptr"], st["indices"], st["last"], case["hq"], case["hkv"], case["d"],
                           PS, causal=True, q_data_type=DTYPES[case["dtype"]])
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "decode":
        if case["plan"]:
            _plan(st)
        if case["append"]:
            return st["wrapper"].run(st["q"][0], st["cache"][0], append_kv=(st["k"][0], st["v"][0])), st["cache"]
        return st["wrapper"].run(st["q"][0], st["cache"][0])
    if kind == "step":
        st["graph"].replay()
        return st["out"], st["cache"]
    if kind == "prefill":
        return st["wrapper"].run(st["q"][0], st["cache"][0])
    if kind == "append":
        if case["rope"]:
            q = ops.append_paged_kv_cache_with_rope(st["q"][0], st["k"][0], st["v"][0], st["cos"], st["sin"],
                                                    st["batch_indices"], st["positions"], st["cache"][0], st["indices"],
                                                    st["indptr"], st["last"])
            return q, st["cache"]
        ops.append_paged_kv_cache(st["k"][0], st["v"][0], st["batch_indices"], st["positions"], st["cache"][0],
                                  st["indices"], st["indptr"], st["last"])
        return st["cache"]
    more = {}
    if case["scale"]:
        more = {"penalty": st["penalty"], "penalty_rows": st["slots"], "temperature": st["temperature"]}
    return sampling.top_k_top_p_sampling_from_logits(st["logits"], st["top_k"], st["top_p"], uniform=st["uniform"], **more)


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    es = 4 if case["dtype"] == "fp32" else 2
    if case["kind"] == "sample":
        n = case["rows"] * case["vocab"]
        return {"bytes": n * es * (2 if case["scale"] else 1) + 24 * case["rows"], "flops": 4 * n}
    kv, new = _lengths(case)
    nnz, hq, hkv, d = sum(new), case["hq"], case["hkv"], case["d"]
    tok = 2 * hkv * d * es  # a token's K and V
    table = 4 * (sum(-(-n // PS) for n in kv) + 2 * len(kv) + 1)
    if case["kind"] == "append":
        return {"bytes": nnz * (2 * tok + 8) + table + (nnz * (2 * hq * d + 2 * d) * es if case["rope"] else 0),
                "flops": 3 * nnz * (hq + hkv) * d if case["rope"] else 0}
    if case["kind"] == "prefill":
        pairs = sum(c * (n - c) + c * (c + 1) // 2 for n, c in zip(kv, new))
        return {"bytes": sum(kv) * tok + 2 * nnz * hq * d * es + table, "flops": 4 * hq * d * pairs}
    layers = case.get("layers", 1)
    pages = case["prefix"] // PS * PS if case["kind"] == "step" else 0  # tokens every sequence shares
    unique = sum(kv) - pages * (len(kv) - 1)
    rows = tok * nnz if case["kind"] == "step" or case["append"] else 0
    return {"bytes": layers * (unique * tok + 2 * nnz * hq * d * es + rows) + table, "flops": 4 * hq * d * sum(kv) * layers}


def tolerance(case):
    if case["kind"] in ("sample", "append"):
        return "exact"  # data movement, products rounded one by one, and integer masses: bit for bit
    # fp16 / bf16: the output's own rounding and that of the softmax weights before P.V (2.2e-4 .. 3.1e-4 and
    # 1.5e-3 .. 2.4e-3 off the 64-bit result, the matrix and the vector kernels 2.1e-4 .. 3.4e-4 and 1.5e-3 .. 2.6e-3
    # apart); fp32: the order of the sums (6e-8 .. 3.4e-7).  About four times that; "max" with room for larger samples.
    return {"fp16": {"rel": 1.2e-3, "max": 3e-2}, "bf16": {"rel": 1e-2, "max": 1e-1}, "fp32": {"rel": 1.5e-6, "max": 5e-5}}[case["dtype"]]


# ---------------------------------------------------------------- the same results in 64 bits

def _attend64(q, k, v, causal):
    """q [n, hq, d], k / v [L, hkv, d] -> [n, hq, d]: row i sees the keys up to L - n + i."""
    n, hq, d = q.shape
    L, hkv, _ = k.shape
    g = hq // hkv
    out = torch.empty((n, hq, d), dtype=torch.float64, device=q.device)
    mask = torch.ones((n, L), dtype=torch.bool, device=q.device).triu(L - n + 1) if causal and n > 1 else None
    for h in range(hkv):
        kh, vh = k[:, h].double(), v[:, h].double()
        for a in range(h * g, (h + 1) * g):
            s = q[:, a].double() @ kh.t() / math.sqrt(d)
            if mask is not None:
                s.masked_fill_(mask, -math.inf)
            out[:, a] = torch.softmax(s, dim=1) @ vh
    return out


def _slots(st):
    """Page and slot of every new token."""
    ptr, idx = st["indptr"].tolist(), st["indices"].long()
    page, slot = [], []
    for b, (n, c) in enumerate(zip(st["kv"], st["new"])):
        pos = torch.arange(n - c, n, device=DEV)
        page.append(idx[ptr[b] + pos // PS])
        slot.append(pos % PS)
    return torch.cat(page), torch.cat(slot)


def _sample64(st):
    case = st["case"]
    x = st["logits"]
    if case["scale"]:  # the serving loop's two divisions, rounded as its tensor operations round
        x = (x / st["penalty"][st["slots"].long()]) / st["temperature"][:, None]
    out = []
    for r, (k, p, u) in enumerate(zip(st["top_k"].tolist(), st["top_p"].tolist(), st["uniform"].tolist())):
        row = x[r].double()
        desc = row.sort(descending=True).values
        keep = torch.ones_like(row, dtype=torch.bool)
        if 0 < k < row.numel():
            keep = row >= desc[k - 1]
        mass = torch.exp(row - desc[0]) * keep
        if p < 1.0:
            kept = desc[: int(keep.sum())]
            run_ = torch.exp(kept - desc[0]).cumsum(0)
            keep = keep & (row >= kept[min(int((run_ < p * run_[-1]).sum()), kept.numel() - 1)])
            mass = mass * keep
        cdf = mass.cumsum(0)
        out.append(min(int((cdf <= u * cdf[-1]).sum()), row.numel() - 1))
    return torch.tensor(out, dtype=torch.int32)


def exact(case, seed):
    st = _inputs(case, seed)
    if case["kind"] == "sample":
        return _sample64(st)
    page, slot = _slots(st)
    cache = st["cache"]
    k, q = st["k"], st["q"]
    if case.get("rope"):
        def turn(x):  # each product, then the sum, rounded to the type, as the model's operations round
            h = case["d"] // 2
            return x * st["cos"][:, None] + torch.cat([-x[..., h:], x[..., :h]], dim=-1) * st["sin"][:, None]
        k, q = turn(k[0])[None], turn(q[0])[None]
    if case["kind"] != "decode" or case["append"]:
        cache[:, page, 0, slot] = k
        cache[:, page, 1, slot] = st["v"]
    if case["kind"] == "append":
        return (q[0], cache) if case["rope"] else cache
    ptr, at = st["indptr"].tolist(), _cumsum(st["new"])
    out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
    for layer in range(q.shape[0]):
        for b, n in enumerate(st["kv"]):
            pages = st["indices"][ptr[b]:ptr[b + 1]].long()
            kv = cache[layer, pages]  # [pages, 2, PS, hkv, d]
            kb, vb = (kv[:, j].reshape(-1, case["hkv"], case["d"])[:n] for j in (0, 1))
            out[layer, at[b]:at[b + 1]] = _attend64(q[layer, at[b]:at[b + 1]], kb, vb, True)
    if case["kind"] == "step":
        return out, cache
    if case["kind"] == "decode" and case["append"]:
        return out[0], cache
    return out[0]
