"""The work that a user of this framework has it do, as cases that can be timed and compared.

A case is a dict of plain values.  Its lengths come from the case itself (``mix`` seeds them), its
values from the seed: qkv projections ~ N(0, 2^2), norm weights ~ 1 + N(0, 0.2^2), cached keys and
values ~ N(0, 1), in the model's 16-bit type.  Every case goes through the package's public entry
points:

  prefill       a step of new prompts or chunks: per layer ``attention_with_prologue`` (norms,
                rotation, store, causal attention) under the step's Context
  decode        one token per sequence: per layer ``attention_with_prologue``
  graph_decode  the same for a stack of layers, replayed by ``DecodeGraphRunner``
  flash_decode  ``flash_attn_with_kvcache`` with one query per sequence
  verify        speculative decoding: ``store_kvcache`` of the drafts, then
                ``flash_attn_with_kvcache`` with several queries per sequence
  store         ``store_kvcache``
  sample        ``Sampler``
"""
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "learn-nano-vllm_amd"))

HD, PAGE = 128, 256               # head_dim and tokens per page of Qwen3's caches
MAX_POSITION, THETA, EPS = 40960, 1e6, 1e-6
VOCAB = 151936


def listed():
    return [
        # Interactive use: three chats in the bucket of four, all 28 layers of a decode step.
        dict(name="graph_decode_3", kind="graph_decode", layers=28, batch=3, ctx_lo=100,
             ctx_hi=2048, hq=16, hkv=8, dtype="bf16", mix=11),
        # A server's decode step at the reference benchmark's lengths, one layer.
        dict(name="decode_64", kind="decode", layers=1, batch=64, ctx_lo=100, ctx_hi=2048, hq=16,
             hkv=8, dtype="bf16", mix=12),
        # Many sequences, eight q heads to a kv head (the 16/2 head split).
        dict(name="decode_192_g8", kind="decode", layers=1, batch=192, ctx_lo=256, ctx_hi=4096,
             hq=16, hkv=2, dtype="bf16", mix=13),
        # A few long documents, a float16 model, the flash-attn entry point.
        dict(name="flash_decode_long", kind="flash_decode", batch=4, ctx_lo=8192, ctx_hi=32768,
             hq=16, hkv=8, dtype="fp16", mix=14),
        # Speculative decoding: 5 drafts and the last accepted token of 32 sequences.
        dict(name="verify_32x6", kind="verify", batch=32, n_query=6, ctx_lo=1024, ctx_hi=8192,
             hq=16, hkv=8, dtype="bf16", mix=15),
        # One user's prompt of ordinary, odd length: time to first token.
        dict(name="prompt_777", kind="prefill", layers=4, nseq=1, new_lo=777, new_hi=777,
             cached_lo=0, cached_hi=0, shared=False, hq=16, hkv=8, dtype="bf16", mix=16),
        # The next chunk of one long prompt (or a follow-up question to a long document).
        dict(name="chunk_after_8k", kind="prefill", layers=2, nseq=1, new_lo=1000, new_hi=1000,
             cached_lo=8300, cached_hi=8300, shared=False, hq=16, hkv=8, dtype="bf16", mix=17),
        # A throughput run's prefill step: prompts of 100 to 1024 tokens, about 16384 in all.
        dict(name="prompts_16k_tokens", kind="prefill", layers=2, nseq=28, new_lo=100,
             new_hi=1024, cached_lo=0, cached_hi=0, shared=False, hq=16, hkv=8, dtype="bf16",
             mix=18),
        # 32 requests behind one cached system prompt of 512 tokens.
        dict(name="prefix_32", kind="prefill", layers=2, nseq=32, new_lo=100, new_hi=1024,
             cached_lo=512, cached_hi=512, shared=True, hq=16, hkv=8, dtype="bf16", mix=19),
        # The largest prefill step of the default configuration: four prompts of 4096 tokens.
        dict(name="prompts_4x4096", kind="prefill", layers=1, nseq=4, new_lo=4096, new_hi=4096,
             cached_lo=0, cached_hi=0, shared=False, hq=16, hkv=8, dtype="bf16", mix=20),
        # The KV store of a full prefill step by itself, values as a view of the packed qkv.
        dict(name="store_16384", kind="store", n_tokens=16384, hq=16, hkv=8, dtype="bf16", mix=21),
        # The next tokens of the largest decode batch of the default configuration.
        dict(name="sample_512", kind="sample", batch=512, vocab=VOCAB, dtype="bf16", mix=22),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed ones' ranges, no dearer than the largest of them."""
    while True:
        kind = rng.choice(["prefill", "prefill", "decode", "graph_decode", "flash_decode",
                           "verify", "store", "sample"])
        hq, hkv = rng.choice([(16, 8), (16, 8), (16, 8), (16, 4), (16, 2), (16, 16), (8, 4),
                              (4, 2)])
        c = dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "bf16", "fp16"]),
                 mix=rng.randrange(1 << 20))
        if kind == "sample":
            c.update(batch=_log_int(rng, 1, 512), vocab=rng.choice([VOCAB, VOCAB, 32000, 50257]))
            return c
        c.update(hq=hq, hkv=hkv)
        if kind == "store":
            c.update(n_tokens=_log_int(rng, 1, 16384))
            return c
        if kind == "prefill":
            lo = _log_int(rng, 1, 2048)
            hi = min(4096, lo + _log_int(rng, 1, 1024))
            cached = rng.choice([0, 0, 1, 1])
            clo = _log_int(rng, 16, 8192) if cached else 0
            shared = bool(cached) and rng.random() < 0.4
            if shared:
                clo = max(PAGE, clo // PAGE * PAGE)
            chi = clo if shared or not cached else min(9000, clo + _log_int(rng, 1, 1024))
            c.update(layers=1, nseq=_log_int(rng, 1, 32), new_lo=lo, new_hi=hi, cached_lo=clo,
                     cached_hi=chi, shared=shared)
            if sum(_lens(c)[0]) > 16384:
                continue
        elif kind == "verify":
            c.update(batch=_log_int(rng, 1, 64), n_query=rng.randint(2, 16 * hkv // hq or 2),
                     ctx_lo=_log_int(rng, 32, 4096))
            if c["n_query"] < 2:
                continue
            c.update(ctx_hi=c["ctx_lo"] + _log_int(rng, 1, 8192))
        elif kind == "flash_decode":
            c.update(batch=_log_int(rng, 1, 16), ctx_lo=_log_int(rng, 1024, 16384))
            c.update(ctx_hi=c["ctx_lo"] + _log_int(rng, 1, 16384))
        elif kind == "decode":
            c.update(layers=1, batch=_log_int(rng, 1, 256), ctx_lo=_log_int(rng, 16, 2048))
            c.update(ctx_hi=c["ctx_lo"] + _log_int(rng, 1, 2048))
        else:
            c.update(layers=28, batch=rng.randint(1, 4), ctx_lo=_log_int(rng, 16, 1024), hq=16,
                     hkv=8)
            c.update(ctx_hi=c["ctx_lo"] + _log_int(rng, 1, 1024))
        w = work(c)
        if w["bytes"] <= 9e8 and w["flops"] <= 2.8e11:
            return c


# ---- sizes ---------------------------------------------------------------------------------

def _lens(case):
    """(new tokens, cached tokens) of every sequence."""
    r = random.Random(case["mix"])
    kind = case["kind"]
    if kind == "prefill":
        new = [r.randint(case["new_lo"], case["new_hi"]) for _ in range(case["nseq"])]
        return new, [r.randint(case["cached_lo"], case["cached_hi"]) for _ in new]
    ctx = [r.randint(case["ctx_lo"], case["ctx_hi"]) for _ in range(case["batch"])]
    n = min(case.get("n_query", 1), case["ctx_lo"])
    return [n] * len(ctx), [c - n for c in ctx]


def _pages(case):
    """(block tables, pages in the pool): pages in shuffled order, a shared prefix's first."""
    new, cached = _lens(case)
    head = cached[0] // PAGE if case.get("shared") else 0
    need = [-(-(a + b) // PAGE) - head for a, b in zip(new, cached)]
    total = head + sum(need)
    ids = list(range(total))
    random.Random(case["mix"] + 1).shuffle(ids)
    tables, at = [], head
    for n in need:
        tables.append(ids[:head] + ids[at:at + n])
        at += n
    return tables, total


def work(case):
    if case["kind"] == "sample":
        return {"bytes": case["batch"] * (case["vocab"] * 2 + 4 + 8), "flops": 0}
    hq, hkv = case["hq"], case["hkv"]
    row = HD * 2
    if case["kind"] == "store":
        n, skipped = case["n_tokens"], case["n_tokens"] // 20
        return {"bytes": 4 * n + 4 * (n - skipped) * hkv * row, "flops": 0}
    new, cached = _lens(case)
    T = sum(new)
    pairs = sum(n * c + n * (n + 1) // 2 for n, c in zip(new, cached))
    flops = 4 * hq * HD * pairs
    keys = cached[0] if case.get("shared") else sum(cached)
    if case["kind"] == "flash_decode":
        return {"bytes": 2 * (keys + T) * hkv * row + 2 * T * hq * row, "flops": flops}
    if case["kind"] == "verify":
        drafts = T - len(new)
        return {"bytes": 2 * (keys + T) * hkv * row + 2 * T * hq * row + 4 * drafts * hkv * row,
                "flops": flops}
    # qkv in, cached keys and values in, attention out, new keys and values out, the rotation rows
    nbytes = T * (hq + 2 * hkv) * row + 2 * keys * hkv * row + T * hq * row \
        + 2 * T * hkv * row + min(T, MAX_POSITION) * HD * 4 + T * 12
    return {"bytes": case["layers"] * nbytes, "flops": case["layers"] * flops}


def tolerance(case):
    if case["kind"] == "store":
        return "exact"
    if case["kind"] == "sample":
        return {"rel": 0.0, "max": 0.0, "differ": 0.004}
    # 16-bit outputs of a softmax whose probabilities are rounded to 16 bits before P.V
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 1.5e-3}


# ---- inputs --------------------------------------------------------------------------------

def _dtype(case):
    return {"bf16": torch.bfloat16, "fp16": torch.float16}[case["dtype"]]


class _Norm:
    """What the prologue reads of an RMSNorm layer."""

    def __init__(self, weight):
        self.weight, self.eps = weight, EPS


class _Rope:
    """What the prologue reads of a rotary embedding layer."""

    def __init__(self, cos_sin_cache):
        self.cos_sin_cache = cos_sin_cache


def _rope_cache():
    inv = 1.0 / (THETA ** (torch.arange(0, HD, 2, dtype=torch.float) / HD))
    f = torch.arange(MAX_POSITION, dtype=torch.float)[:, None] * inv
    return torch.cat((f.cos(), f.sin()), dim=-1).unsqueeze(1).cuda()


def _inputs(case, seed):
    """Every tensor of a case, on the GPU, from plain torch and the seed."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt = _dtype(case)

    def randn(*shape, scale=1.0):
        out = torch.empty(*shape, dtype=dt, device="cuda")
        flat = out.view(-1)
        for i in range(0, flat.numel(), 1 << 26):
            part = flat[i:i + (1 << 26)]
            part.copy_(torch.randn(part.numel(), generator=gen, device="cuda") * scale)
        return out

    def ints(v, dtype=torch.int32):
        return torch.tensor(v, dtype=dtype, device="cuda")

    if case["kind"] == "sample":
        return dict(logits=randn(case["batch"], case["vocab"], scale=2.5),
                    temperatures=torch.rand(case["batch"], generator=gen, device="cuda") * 0.6 + 0.5)
    hq, hkv = case["hq"], case["hkv"]
    if case["kind"] == "store":
        n = case["n_tokens"]
        pages = -(-n // PAGE) + 2
        qkv = randn(n, (hq + 2 * hkv) * HD)
        slots = torch.randperm(pages * PAGE, generator=gen, device="cuda")[:n].to(torch.int32)
        slots[torch.randperm(n, generator=gen, device="cuda")[:n // 20]] = -1
        return dict(key=randn(n, hkv, HD), value=qkv[:, (hq + hkv) * HD:].view(n, hkv, HD),
                    slots=slots, k_cache=randn(pages, PAGE, hkv, HD),
                    v_cache=randn(pages, PAGE, hkv, HD))
    new, cached = _lens(case)
    tables, pages = _pages(case)
    width = max(len(t) for t in tables)
    L = case.get("layers", 1)
    kv = randn(2, L, pages, PAGE, hkv, HD)
    x = dict(kv=kv, block_tables=ints([t + [-1] * (width - len(t)) for t in tables]),
             ctx=ints([n + c for n, c in zip(new, cached)]))
    drop = 1 if case["kind"] == "verify" else 0   # the first query of a verify step is cached
    at = [[p for p in range(c + drop, c + n)] for n, c in zip(new, cached)]
    x["slots"] = ints([t[p // PAGE] * PAGE + p % PAGE for t, a in zip(tables, at) for p in a])
    T = sum(new)
    if case["kind"] == "flash_decode":
        x["q"] = randn(T, 1, hq, HD)
        return x
    if case["kind"] == "verify":
        B = len(new)
        x["q"] = randn(B, new[0], hq, HD)
        x["key"], x["value"] = (randn(T - B, hkv, HD) for _ in range(2))
        return x
    x["positions"] = ints([p for a in at for p in a], torch.int64)
    x["qkv"] = randn(T, L, (hq + 2 * hkv) * HD, scale=2.0)
    x["weights"] = [(1 + 0.2 * torch.randn(2, HD, generator=gen, device="cuda")).to(dt)
                    for _ in range(L)]
    x["cos_sin"] = _rope_cache()
    return x


def prepare(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    if kind == "sample":
        from nanovllm_amd.layers.sampler import Sampler
        torch.manual_seed(seed)
        x["sampler"] = Sampler()
    elif kind == "verify":
        # the caches before the drafts are stored, and the lengths after
        x["n_query"] = x["q"].shape[1]
    elif kind in ("prefill", "decode", "graph_decode"):
        from nanovllm_amd import Attention
        new, cached = _lens(case)
        x["rope"] = _Rope(x["cos_sin"])
        x["layers"] = []
        for i, w in enumerate(x["weights"]):
            attn = Attention(case["hq"], HD, HD ** -0.5, case["hkv"])
            attn.k_cache, attn.v_cache = x["kv"][0, i], x["kv"][1, i]
            x["layers"].append((attn, _Norm(w[0]), _Norm(w[1])))
        if kind == "prefill":
            tot = [n + c for n, c in zip(new, cached)]
            cu = lambda v: torch.tensor([sum(v[:i]) for i in range(len(v) + 1)],
                                        dtype=torch.int32, device="cuda")
            x["context"] = dict(is_prefill=True, cu_seqlens_q=cu(new), cu_seqlens_k=cu(tot),
                                max_seqlen_q=max(new), max_seqlen_k=max(tot),
                                slot_mapping=x["slots"],
                                block_tables=x["block_tables"] if any(cached) else None)
        else:
            x["context"] = dict(is_prefill=False, slot_mapping=x["slots"], context_lens=x["ctx"],
                                block_tables=x["block_tables"])
        if kind == "graph_decode":
            x["runner"] = _graph_runner(case, x)
    x["kind"] = kind
    return x


def _graph_runner(case, x):
    from nanovllm_amd import attention_with_prologue
    from nanovllm_amd.engine.graph_runner import DecodeGraphRunner
    L, hq, hkv, dt = case["layers"], case["hq"], case["hkv"], _dtype(case)
    layers, rope = x["layers"], x["rope"]

    def step(positions, qkv):
        outs = [attention_with_prologue(attn, positions, qkv[:, i], qn, kn, rope)
                .reshape(positions.numel(), hq * HD) for i, (attn, qn, kn) in enumerate(layers)]
        return torch.stack(outs, dim=1)

    # capturing runs the step on zeroed metadata: keep what it stores out of the cache
    kv = x["kv"]
    first = kv[:, :, 0].clone()
    runner = DecodeGraphRunner(step, 4, x["block_tables"].shape[1],
                               {"qkv": ((L, (hq + 2 * hkv) * HD), dt)}, ((L, hq * HD), dt))
    kv[:, :, 0].copy_(first)
    return runner


def run(state):
    kind = state["kind"]
    if kind == "sample":
        return state["sampler"](state["logits"], state["temperatures"])
    if kind == "store":
        from nanovllm_amd import store_kvcache
        store_kvcache(state["key"], state["value"], state["k_cache"], state["v_cache"],
                      state["slots"])
        return [state["k_cache"], state["v_cache"]]
    if kind in ("flash_decode", "verify"):
        from nanovllm_amd import flash_attn_with_kvcache, store_kvcache
        k_cache, v_cache = state["kv"][0, 0], state["kv"][1, 0]
        if kind == "verify" and state["n_query"] > 1:
            store_kvcache(state["key"], state["value"], k_cache, v_cache, state["slots"])
        o = flash_attn_with_kvcache(state["q"], k_cache, v_cache, cache_seqlens=state["ctx"],
                                    block_table=state["block_tables"], softmax_scale=HD ** -0.5,
                                    causal=True)
        return [o, state["kv"]] if kind == "verify" else [o]
    from nanovllm_amd import attention_with_prologue, set_context
    set_context(**state["context"])
    if kind == "graph_decode":
        return [state["runner"].run(state["positions"], qkv=state["qkv"]), state["kv"]]
    outs = [attention_with_prologue(attn, state["positions"], state["qkv"][:, i], qn, kn,
                                    state["rope"])
            for i, (attn, qn, kn) in enumerate(state["layers"])]
    return outs + [state["kv"]]


# ---- the same in 64 bits -------------------------------------------------------------------

def _norm_rope(x, w, cos, sin):
    """RMSNorm then rotary embedding of [T, H, D], in float64."""
    x = x.double()
    x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()
    a, b = x.chunk(2, dim=-1)
    return torch.cat((a * cos - b * sin, b * cos + a * sin), dim=-1)


def _attend(q, k, v, diag):
    """q [n, Hq, D], k / v [m, Hkv, D] in float64; query i sees keys j <= i + diag."""
    n, hq, _ = q.shape
    m, hkv, _ = k.shape
    g = hq // hkv
    out = torch.empty_like(q)
    for h in range(hkv):
        for i in range(0, n, 1024):
            qq = q[i:i + 1024, h * g:(h + 1) * g].reshape(-1, HD)
            s = qq @ k[:, h].t().contiguous() * HD ** -0.5
            row = torch.arange(i, min(n, i + 1024), device="cuda").repeat_interleave(g)
            s.masked_fill_(torch.arange(m, device="cuda")[None] > row[:, None] + diag,
                           float("-inf"))
            out[i:i + 1024, h * g:(h + 1) * g] = (torch.softmax(s, -1)
                                                  @ v[:, h].contiguous()).view(-1, g, HD)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("sample", "store"):     # drawn tokens; copied bits
        return None
    x = _inputs(case, seed)
    new, cached = _lens(case)
    hq, hkv = case["hq"], case["hkv"]
    kv = x["kv"].double()
    outs = []
    for i in range(kv.shape[1]):
        kc, vc = (kv[j, i].view(-1, hkv, HD) for j in range(2))
        slots = x["slots"].long()
        if kind == "verify":
            kc[slots], vc[slots] = x["key"].double(), x["value"].double()
            q = x["q"].double().view(-1, hq, HD)
        elif kind == "flash_decode":
            q = x["q"].double().view(-1, hq, HD)
        else:
            qkv = x["qkv"][:, i]
            q, k, v = (t.reshape(len(qkv), -1, HD) for t in
                       qkv.split([hq * HD, hkv * HD, hkv * HD], dim=-1))
            cos, sin = x["cos_sin"][x["positions"]].double().chunk(2, dim=-1)
            w = x["weights"][i]
            q, k = _norm_rope(q, w[0], cos, sin), _norm_rope(k, w[1], cos, sin)
            kc[slots], vc[slots] = k, v.double()
        o, at = torch.empty_like(q), 0
        for s, (n, c) in enumerate(zip(new, cached)):
            p = torch.arange(n + c, device="cuda")
            rows = x["block_tables"][s, p // PAGE].long() * PAGE + p % PAGE
            o[at:at + n] = _attend(q[at:at + n], kc[rows], vc[rows], c)
            at += n
        outs.append(o)
    if kind == "graph_decode":
        return [torch.stack([o.reshape(len(o), -1) for o in outs], dim=1), kv]
    if kind == "decode":
        return [o.unsqueeze(1) for o in outs] + [kv]
    if kind == "flash_decode":
        return [outs[0].view(x["q"].shape)]
    if kind == "verify":
        return [outs[0].view(x["q"].shape), kv]
    return outs + [kv]
