"""A prefill layer's prologue and attention in one call
(nvk_varlen_prefill_prologue, the prefill route of attention_with_prologue)
against the two calls it replaces, bit for bit: large steps, whose workgroups
norm and rotate their own q rows, and others, whose q shares the output's rows;
dense, paged, split, ranked and short-query forms, every group size, both
dtypes, positions outside the rotation table, padding slots, an empty cache and
a hooked module."""
import pytest
import torch

from gpu_utils import say
from nanovllm_amd import (Attention, attention_with_prologue, qk_norm_rope_store,
                          rope_cos_sin_cache)
from nanovllm_amd.utils.context import get_context, reset_context, set_context
from nanovllm_amd.workloads import _Norm, _Rope

pytestmark = pytest.mark.gpu

D, EPS, MAX_POS = 128, 1e-6, 6000


def _step(seed, lens_q, cached, hq, hkv, bs, dtype, paged, row_pad=0, store=True):
    g = torch.Generator().manual_seed(seed)
    T, tot = sum(lens_q), [a + b for a, b in zip(lens_q, cached)]
    pages = [-(-t // bs) for t in tot]
    perm = torch.randperm(sum(pages) + 2, generator=g).tolist()
    bt = torch.full((len(tot), max(pages)), -1, dtype=torch.int32)
    slots, pos, at = [], [], 0
    for i, n in enumerate(pages):
        bt[i, :n] = torch.tensor(perm[at:at + n])
        at += n
        pos += list(range(cached[i], tot[i]))
        slots += [int(bt[i, p // bs]) * bs + p % bs for p in range(cached[i], tot[i])]
    kc, vc = (torch.randn(sum(pages) + 2, bs, hkv, D, generator=g).to(dtype).cuda()
              for _ in range(2))
    wide = (torch.randn(T, (hq + 2 * hkv) * D + row_pad, generator=g) * 2).to(dtype).cuda()
    w = [(1 + 0.2 * torch.randn(D, generator=g)).to(dtype).cuda() for _ in range(2)]
    cu = lambda v: torch.tensor([sum(v[:i]) for i in range(len(v) + 1)], dtype=torch.int32).cuda()
    if not paged and T > 3:
        slots[2] = -1
        pos[0], pos[1] = -4, MAX_POS + 7        # clamped into the table, as by the prologue
    set_context(True, cu(lens_q), cu(tot), max(lens_q), max(tot),
                torch.tensor(slots, dtype=torch.int32).cuda(), None, bt.cuda() if paged else None)
    return (wide[:, :(hq + 2 * hkv) * D], w, torch.tensor(pos).cuda(), kc, vc,
            rope_cos_sin_cache(D, MAX_POS, 1e6).cuda())


CASES = [  # lens_q, cached, hq, hkv, bs
    ([1, 63, 64, 65, 300] * 4 + [40] * 6, [0] * 26, 16, 8, 256),     # ranked tiles
    ([700] * 7 + [1, 33], [256 * i + 7 for i in range(9)], 16, 8, 256),
    ([700] * 7 + [1, 33], [100] * 9, 16, 8, 48),                     # per-row page lookups
    ([700] * 7, [64] * 7, 16, 4, 64),
    ([700] * 7, [64 * i for i in range(7)], 16, 2, 128),
    ([1400] * 3 + [1], [0] * 4, 16, 4, 256),
    ([500] * 5, [300] * 5, 16, 4, 64),
    ([300] * 4, [64] * 4, 16, 2, 128),
    ([600] * 8, [128] * 8, 16, 16, 256),
    ([4096, 5], [0, 0], 16, 8, 256),          # a single long prompt beside a short one
    ([777], [0], 16, 8, 256),
    ([300], [4000], 16, 8, 256),              # parts
    ([6, 6, 3], [900, 50, 2000], 16, 8, 256),  # short-query kernels
    ([1], [0], 4, 2, 256),
]


@pytest.mark.parametrize("lens_q,cached,hq,hkv,bs", CASES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_one_call_equals_two(lens_q, cached, hq, hkv, bs, dtype):
    paged = any(cached)
    pad = 64 if hkv == 8 else 0
    qkv, w, pos, kc, vc, cs = _step(3 + hq + bs, lens_q, cached, hq, hkv, bs, dtype, paged, pad)
    attn = Attention(hq, D, D ** -0.5, hkv)
    attn.k_cache, attn.v_cache = kc.clone(), vc.clone()
    say(f"prefill with prologue {lens_q} after {cached}, {hq}/{hkv}, page {bs}, {dtype}")
    try:
        one = attention_with_prologue(attn, pos, qkv, _Norm(w[0], EPS), _Norm(w[1], EPS), _Rope(cs))
        k1, v1 = attn.k_cache, attn.v_cache
        attn.k_cache, attn.v_cache = kc, vc
        q, k, v = qk_norm_rope_store(pos, qkv, hq, hkv, D, w[0], w[1], EPS, cs, kc, vc,
                                     get_context().slot_mapping, return_k=not paged)
        two = attn(q, k, v, kv_stored=True)
        torch.cuda.synchronize()
    finally:
        reset_context()
    assert torch.equal(one, two)
    assert torch.equal(k1, kc) and torch.equal(v1, vc)


def test_empty_cache_and_hooks():
    qkv, w, pos, kc, vc, cs = _step(5, [900] * 6, [0] * 6, 16, 8, 256, torch.bfloat16, False)
    attn = Attention(16, D, D ** -0.5, 8)     # warmup: no cache yet, nothing stored
    args = (attn, pos, qkv, _Norm(w[0], EPS), _Norm(w[1], EPS), _Rope(cs))
    say("warmup without a cache, then with a forward hook")
    seen = []
    try:
        bare = attention_with_prologue(*args)
        handle = attn.register_forward_hook(lambda m, i, o: seen.append(o.shape))
        hooked = attention_with_prologue(*args)
        handle.remove()
        torch.cuda.synchronize()
    finally:
        reset_context()
    assert torch.equal(bare, hooked) and seen == [hooked.shape]
