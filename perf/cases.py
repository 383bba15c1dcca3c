"""The attention path's calls as a serving program makes them, for timing and for comparing outputs.

A case is one call per layer of one scheduler step, through the C entry points of libmvr_attn.so: the argument block
and its workspace are prepared once and kept, as a runner keeps them per layer, and a pass is the one library call
(planning and launches included).  Head shapes are those of the models the repository names: Qwen2-0.5B (14 query / 2
KV heads, head_dim 64), Qwen2-7B (28 / 4, 128), Llama-3-8B (32 / 8, 128), Llama-3.2-1B (32 / 8, 64) and Llama-3.2-3B
(24 / 8, 128).  Every call carries the host copies of the length tables, which a runner has.

Lengths belong to the case; the seed gives the values and the pages' order.  Queries and keys are N(0, 1.5^2) and
N(0, 1), so that scores after the 1/sqrt(head_dim) scale spread by about 1.5, as in a trained model (not the nearly
uniform softmax of tiny values); values are N(0, 1).
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mini-vllm-rs_amd"))

import mvr_attn as M  # noqa: E402
import workloads as W  # noqa: E402

SHAPES = {  # query heads, KV heads, head_dim
    "qwen2-0.5b": (14, 2, 64),
    "qwen2-7b": (28, 4, 128),
    "llama-3-8b": (32, 8, 128),
    "llama-3.2-1b": (32, 8, 64),
    "llama-3.2-3b": (24, 8, 128),
}
MAX_BYTES = 2.2e9    # K/V of the largest listed decode
MAX_FLOPS = 4.9e11   # the largest listed prompt


def _case(name, kind, model, dtype, **sizes):
    """kind: decode, verify, chunk, fresh, mixed, cascade or append.  batch requests of lo..hi cached tokens (uniform
    when lo == hi) with q new tokens each; page: tokens per page; shared: tokens of a common prefix in groups of
    group requests; chunk / prefix: the prefill request that follows a mixed step's decodes."""
    c = dict(kind=kind, model=model, dtype=dtype, batch=1, lo=0, hi=0, q=1, page=16, shared=0, group=0, chunk=0,
             prefix=0)
    c.update(sizes)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # One chat with the smallest model, F32 (the dtype the reference's GPU backends use): launches and latency.
        _case("decode f32 1x512", "decode", "qwen2-0.5b", "f32", batch=1, lo=511, hi=511),
        # A few users of the small model, contexts of all lengths: one decode step.
        _case("decode f16 8 ragged", "decode", "qwen2-0.5b", "f16", batch=8, lo=127, hi=4095),
        # A busy server's decode step with short and middling chats.
        _case("decode f16 64 ragged", "decode", "llama-3-8b", "f16", batch=64, lo=511, hi=3583),
        # The headline: a full batch at long contexts, bound by HBM.
        _case("decode f16 64x8192", "decode", "llama-3-8b", "f16", batch=64, lo=8191, hi=8191),
        # An F32 server's decode step.
        _case("decode f32 16 ragged", "decode", "qwen2-7b", "f32", batch=16, lo=1023, hi=8191),
        # Speculative verification: 4 draft tokens and a bonus, groups of 4 requests on one cached prefix.
        _case("verify f16 16 ragged", "verify", "llama-3-8b", "f16", batch=16, lo=1024, hi=16384, q=5, shared=1024,
              group=4),
        # A prefill step of 4 requests, 256 new tokens each on a cached 2K prefix.
        _case("chunk f16 4x256", "chunk", "qwen2-7b", "f16", batch=4, lo=2048, hi=2048, q=256),
        # The same in F32 at odd sizes: 3 requests, 217 new tokens on cached prefixes of any length.
        _case("chunk f32 3x217 ragged", "chunk", "qwen2-7b", "f32", batch=3, lo=300, hi=3000, q=217),
        # A whole long prompt at once: the largest contraction.
        _case("fresh f16 8192", "fresh", "qwen2-7b", "f16", batch=1, lo=0, hi=0, q=8192),
        # One scheduler step under load: decodes first, then the prefill chunk that the token budget admits.
        _case("mixed f16 63+256", "mixed", "llama-3-8b", "f16", batch=63, lo=8192, hi=8192, chunk=256, prefix=2048),
        # Many users behind one long system prompt, whose pages are shared.
        _case("cascade f16 64 on 8192", "cascade", "llama-3-8b", "f16", batch=64, lo=8448, hi=10240, shared=8192,
              group=64),
        # Rotary embedding and page append of a prefill step's new tokens.
        _case("append f16 4x256", "append", "qwen2-7b", "f16", batch=4, lo=2048, hi=2048, q=256),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        kind = rng.choice(["decode", "decode", "verify", "chunk", "chunk", "fresh", "mixed", "cascade", "append"])
        model = rng.choice(sorted(SHAPES))
        dtype = "f16" if rng.random() < 0.7 else "f32"
        page = rng.choice([16, 16, 16, 16, 32, 24, 8])
        s = dict(page=page)
        if kind in ("decode", "verify"):
            s["batch"] = _log(rng, 1, 64)
            s["hi"] = _log(rng, 200, 16384)
            s["lo"] = s["hi"] if rng.random() < 0.4 else max(1, s["hi"] // rng.randint(2, 9))
            if kind == "verify":
                s["q"] = rng.randint(2, 8)
        elif kind == "chunk":
            s["batch"] = rng.randint(1, 6)
            s["q"] = _log(rng, 40, 700)
            s["hi"] = _log(rng, 100, 8192)
            s["lo"] = s["hi"] if rng.random() < 0.4 else max(1, s["hi"] // rng.randint(2, 6))
        elif kind == "fresh":
            s["batch"] = rng.randint(1, 4)
            s["q"] = _log(rng, 150, 8192)
        elif kind == "mixed":
            s["batch"] = _log(rng, 3, 63)
            s["hi"] = _log(rng, 300, 8192)
            s["lo"] = s["hi"] if rng.random() < 0.4 else max(1, s["hi"] // rng.randint(2, 8))
            s["chunk"] = _log(rng, 60, 600)
            s["prefix"] = _log(rng, 1, 4096)
        elif kind == "cascade":
            s["page"] = rng.choice([16, 32])  # the entry point takes multiples of 16
            s["batch"] = _log(rng, 8, 64)
            s["group"] = s["batch"]
            s["shared"] = 32 * _log(rng, 32, 256)
            s["lo"] = s["shared"] + rng.randint(64, 512)
            s["hi"] = s["lo"] + _log(rng, 64, 2048)
        else:
            s["batch"] = rng.randint(1, 16)
            s["q"] = _log(rng, 1, 256)
            s["hi"] = s["lo"] = _log(rng, 16, 4096)
        c = _case("", kind, model, dtype, **s)
        w = work(c)
        if w["bytes"] <= MAX_BYTES and w["flops"] <= MAX_FLOPS / (1 if dtype == "f16" else 8) and \
                _pool_bytes(c) <= MAX_BYTES:
            return c


def _lengths(c):
    """(new tokens, total tokens) per request; seq_lens counts the new ones."""
    rng = np.random.default_rng([c["batch"], c["lo"], c["hi"], c["q"]])
    q = np.full(c["batch"], c["q"], np.int32)
    cached = rng.integers(c["lo"], c["hi"], size=c["batch"], endpoint=True).astype(np.int32)
    if c["kind"] == "mixed":
        q = np.concatenate([q, [c["chunk"]]]).astype(np.int32)
        cached = np.concatenate([cached, [c["prefix"]]]).astype(np.int32)
    return q, (cached + q).astype(np.int32)


def _pages(c, seq_lens):
    """(pages of each group's prefix, private pages of each request)."""
    shared = min(c["shared"], int(seq_lens.min())) // c["page"] if c["group"] else 0
    return shared, [math.ceil(int(n) / c["page"]) - shared for n in seq_lens]


def _pool_pages(c):
    shared, private = _pages(c, _lengths(c)[1])
    return sum(private) + (shared * math.ceil(c["batch"] / c["group"]) if c["group"] else 0)


def _pool_bytes(c):
    _, hkv, d = SHAPES[c["model"]]
    return 2 * _pool_pages(c) * c["page"] * hkv * d * _es(c)


def _es(c):
    return 2 if c["dtype"] == "f16" else 4


def _pairs(q, n):
    """Causally visible (query, key) pairs of one request."""
    return q * (n - q) + q * (q + 1) // 2


def work(c):
    hq, hkv, d = SHAPES[c["model"]]
    q, n = _lengths(c)
    tokens = int(q.sum())
    if c["kind"] == "append":  # q, k, v in and out, one cos and one sin row, one page id
        return {"bytes": tokens * ((hq + 2 * hkv) * d * _es(c) * 2 + d * _es(c) + 4),
                "flops": tokens * (hq + hkv) * d * 3}
    keys = int(n.sum())
    if c["group"]:  # a shared prefix is read once
        shared, _ = _pages(c, n)
        keys -= shared * c["page"] * (c["batch"] - math.ceil(c["batch"] / c["group"]))
    ids = sum(math.ceil(int(x) / c["page"]) for x in n)
    return {"bytes": keys * hkv * d * _es(c) * 2 + tokens * hq * d * _es(c) * 2 + 4 * ids,
            "flops": 4 * hq * d * sum(_pairs(int(a), int(b)) for a, b in zip(q, n))}


def _inputs(c, seed):
    hq, hkv, d = SHAPES[c["model"]]
    dt = torch.float16 if c["dtype"] == "f16" else torch.float32
    q_lens, seq_lens = _lengths(c)
    shared, private = _pages(c, seq_lens)
    num_pages = _pool_pages(c)
    order = np.random.default_rng(seed).permutation(num_pages).astype(np.int32)
    table = np.zeros((len(seq_lens), max(private) + shared), np.int32)
    used = 0
    for s in range(len(seq_lens)):
        if shared:
            if s % c["group"] == 0:
                prefix = order[used:used + shared]
                used += shared
            table[s, :shared] = prefix
        table[s, shared:shared + private[s]] = order[used:used + private[s]]
        used += private[s]
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(shape, std):
        return torch.empty(shape, dtype=dt, device="cuda").normal_(0.0, std, generator=gen)

    tokens = int(q_lens.sum())
    t = dict(q=normal((hq, tokens, d), 1.5), key_pool=normal((num_pages, 1, hkv, c["page"], d), 1.0),
             value_pool=normal((num_pages, 1, hkv, c["page"], d), 1.0), q_lens=q_lens, seq_lens=seq_lens,
             cu=np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32), table=table, shared=shared)
    if c["kind"] == "append":
        t["k"], t["v"] = normal((hkv, tokens, d), 1.0), normal((hkv, tokens, d), 1.0)
        cos, sin = W.rope_tables(d, 1000000.0, int(seq_lens.max()), np.float16 if c["dtype"] == "f16" else np.float32)
        t["cos"], t["sin"] = torch.from_numpy(cos).cuda(), torch.from_numpy(sin).cuda()
    return t


def prepare(c, seed):
    t = _inputs(c, seed)
    dev = {k: torch.from_numpy(t[k]).cuda() for k in ("table", "seq_lens", "cu")}
    lib = M.load_library()
    out = torch.empty_like(t["q"])
    s = dict(kind=c["kind"], lib=lib, out=out, keep=(t, dev))
    max_len = int(t["seq_lens"].max())
    if c["kind"] == "append":
        s["args"] = M.make_rope_append_args(t["q"], t["k"], t["v"], t["cos"], t["sin"], dev["table"], dev["seq_lens"],
                                            dev["cu"], t["key_pool"], t["value_pool"], out, max_seq_len=max_len)
        s["outputs"] = dict(q=out, key_pool=t["key_pool"], value_pool=t["value_pool"])
        return s
    s["args"] = a = M.make_args(t["q"], t["key_pool"], t["value_pool"], dev["table"], dev["seq_lens"], dev["cu"], out,
                                max_q_len=int(t["q_lens"].max()), max_seq_len=max_len,
                                sum_seq_lens=int(t["seq_lens"].sum()), seq_lens_host=t["seq_lens"],
                                cu_q_lens_host=t["cu"])
    if c["kind"] == "cascade":
        prefix = t["shared"] * c["page"]
        tables = [torch.from_numpy(x).cuda() for x in (
            np.array([0, c["batch"]], np.int32), np.array([prefix], np.int32), t["table"][:1].copy(),
            np.full(c["batch"], prefix, np.int32))]
        s["groups"] = M.make_cascade_groups(*tables, max_group_q_len=c["batch"], max_prefix_len=prefix,
                                            sum_prefix_lens=prefix * c["batch"])
        need = lib.mvr_paged_attention_cascade_workspace_size(ctypes.byref(a), ctypes.byref(s["groups"]))
    else:
        need = M.workspace_size(a)
    s["workspace"] = M.new_workspace(need, "cuda")
    a.workspace, a.workspace_bytes = s["workspace"].data_ptr(), need
    s["outputs"] = out
    return s


def run(s):
    lib, a = s["lib"], ctypes.byref(s["args"])
    if s["kind"] == "append":
        rc = lib.mvr_rope_append(a)
    elif s["kind"] == "cascade":
        rc = lib.mvr_paged_attention_cascade(a, ctypes.byref(s["groups"]))
    else:
        rc = lib.mvr_paged_attention(a)
    if rc != 0:
        raise M.MvrError(rc, lib.mvr_last_error().decode())
    return s["outputs"]


def tolerance(c):
    if c["kind"] == "append":
        # Each product and sum is rounded to the dtype by contract, so the results are bit-exact.
        return "exact"
    # F16: the output's own rounding (2^-11 at most) and the probabilities' in the P V product; F32: sums of up to
    # 16K terms in another order.
    return {"rel": 1.2e-3, "max": 1e-2} if c["dtype"] == "f16" else {"rel": 4e-6, "max": 4e-5}


def _exact_append(c, t):
    hq, hkv, d = SHAPES[c["model"]]
    key, val = t["key_pool"].double(), t["value_pool"].double()
    pos = torch.cat([torch.arange(n - q, n) for q, n in zip(t["q_lens"].tolist(), t["seq_lens"].tolist())]).cuda()
    cos, sin = t["cos"].double()[pos], t["sin"].double()[pos]

    def rope(x):
        a, b = x[..., :d // 2].double(), x[..., d // 2:].double()
        return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)

    seq = torch.from_numpy(np.repeat(np.arange(len(t["q_lens"])), t["q_lens"])).cuda()
    page = torch.from_numpy(t["table"]).cuda().long()[seq, pos // c["page"]]
    key[page, 0, :, pos % c["page"]] = rope(t["k"]).transpose(0, 1)
    val[page, 0, :, pos % c["page"]] = t["v"].double().transpose(0, 1)
    return dict(q=rope(t["q"]), key_pool=key, value_pool=val)


def exact(c, seed):
    t = _inputs(c, seed)
    if c["kind"] == "append":
        return _exact_append(c, t)
    hq, hkv, d = SHAPES[c["model"]]
    out = torch.empty(t["q"].shape, dtype=torch.float64, device="cuda")
    for s, (q_len, n) in enumerate(zip(t["q_lens"].tolist(), t["seq_lens"].tolist())):
        ids = torch.from_numpy(t["table"][s, :math.ceil(n / c["page"])]).cuda().long()
        lo = int(t["cu"][s])
        for h in range(hkv):
            heads = slice(h * hq // hkv, (h + 1) * hq // hkv)
            k = t["key_pool"][ids, 0, h].reshape(-1, d)[:n].double()
            v = t["value_pool"][ids, 0, h].reshape(-1, d)[:n].double()
            for i in range(0, q_len, 1024):
                m = min(1024, q_len - i)
                scores = t["q"][heads, lo + i:lo + i + m].double().reshape(-1, d) @ k.t() / math.sqrt(d)
                scores = scores.view(-1, m, n)
                limit = torch.arange(n - q_len + i, n - q_len + i + m, device="cuda")
                scores.masked_fill_(torch.arange(n, device="cuda")[None, :] > limit[:, None], -math.inf)
                p = torch.softmax(scores, -1).view(-1, n)
                out[heads, lo + i:lo + i + m] = (p @ v).view(-1, m, d)
    return out
