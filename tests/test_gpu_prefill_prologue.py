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
from nanovllm_amd import (Attention, _lib, attention_with_prologue, qk_norm_rope_store,
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
    # own q rows behind cached ones
    ([700] * 9 + [1, 33], [256 * i + 7 for i in range(11)], 16, 8, 256),
    ([700] * 9 + [1, 33], [100] * 11, 16, 8, 48),
    ([700] * 9, [64] * 9, 16, 4, 64),
    ([600] * 11, [128] * 11, 16, 16, 256),
    # and ranked tiles
    ([700] * 12, [0] * 12, 16, 8, 256),
    ([700] * 12, [100 * i for i in range(12)], 16, 4, 64),
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


@pytest.mark.parametrize("lens_q,cached,hq,hkv,own,ranked", [
    ([600] * 8 + [599], [512] * 9, 16, 8, True, False),        # with the spare token: 5400
    ([600] * 8 + [598], [512] * 9, 16, 8, False, False),
    ([600] * 9 + [599], [512] * 10, 16, 16, True, False),      # 6000
    ([600] * 9 + [598], [512] * 10, 16, 16, False, False),
    ([512] * 7 + [511], [512] * 8, 16, 2, True, False),        # 4096
    ([512] * 7 + [510], [512] * 8, 16, 2, False, False),
    ([700] * 6 + [699], [512] * 7, 16, 2, True, False), ([700] * 7, [512] * 7, 16, 2, False, False),
    ([1024] * 4, [324] * 4, 16, 8, True, False), ([1024] * 4, [325] * 4, 16, 8, False, False),
    ([700] * 12, [0] * 12, 16, 8, True, True), ([700] * 12, [64] * 12, 16, 4, True, True),
])
def test_which_steps_norm_their_own_q(lens_q, cached, hq, hkv, own, ranked):
    """The edges of the rule, seen on a token that belongs to no sequence: its row of
    out gets q from the prologue kernel, or nothing where the attention's
    workgroups norm their own rows."""
    paged = any(cached)
    qkv, w, pos, kc, vc, cs = _step(7, lens_q + [1], cached + [0], hq, hkv, 256, torch.bfloat16,
                                    paged)
    c, lib, T, batch = get_context(), _lib.load(), sum(lens_q) + 1, len(lens_q)
    reset_context()
    mq, mk = max(lens_q), max(a + b for a, b in zip(lens_q, cached))
    sizes = (batch, mq, mk, hq, hkv)
    assert (lib.nvk_prefill_tile_order_size(*sizes, 256) > 0) == ranked
    out = torch.full((T, hq, D), 77.0, dtype=qkv.dtype, device="cuda")
    k_new = torch.empty(T, hkv, D, dtype=qkv.dtype, device="cuda")
    ws_bytes = lib.nvk_varlen_prefill_parts_workspace_size(*sizes, D)
    ws = torch.empty(ws_bytes + 256, dtype=torch.uint8, device="cuda")
    cs2, bt = cs.view(cs.shape[0], -1), c.block_tables
    say(f"own q rows of {batch} sequences, {T - 1} tokens, {hq}/{hkv} heads")
    _lib.check(lib.nvk_varlen_prefill_prologue(
        qkv.data_ptr(), qkv.stride(0), T, pos.data_ptr(), w[0].data_ptr(), w[1].data_ptr(), EPS,
        cs2.data_ptr(), cs2.stride(0), cs2.shape[0], kc.data_ptr(), vc.data_ptr(),
        c.slot_mapping.data_ptr(), kc.shape[0] * kc.shape[1], None if paged else k_new.data_ptr(),
        c.cu_seqlens_q.data_ptr(), c.cu_seqlens_k.data_ptr(), batch, mq, mk,
        bt.data_ptr() if paged else None, bt.stride(0) if paged else 0,
        bt.shape[1] if paged else 0, 256 if paged else 0, kc.shape[0] if paged else 0, hq, hkv, D,
        D ** -0.5, out.data_ptr(), out.stride(0), out.stride(1), ws.data_ptr(), ws_bytes, None, 0,
        _lib.dtype_code(qkv), _lib.stream_ptr(qkv.device)))
    torch.cuda.synchronize()
    assert out[-1].eq(77).all().item() == own
    assert not out[:-1].eq(77).any()


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


@pytest.mark.parametrize("no_query", ["no sequence", "no query bound"])
def test_tokens_of_no_sequence_are_stored(no_query):
    """As by the two calls: the prologue does not look at the sequences."""
    qkv, w, pos, kc, vc, cs = _step(6, [40], [0], 16, 8, 64, torch.bfloat16, False)
    slots = get_context().slot_mapping
    k2, v2 = kc.clone(), vc.clone()
    norms = _Norm(w[0], EPS), _Norm(w[1], EPS)
    say(f"prefill with prologue, {no_query}")
    cu = torch.zeros(1, dtype=torch.int32).cuda()
    try:
        if no_query == "no sequence":
            attn = Attention(16, D, D ** -0.5, 8)
            attn.k_cache, attn.v_cache = k2, v2
            set_context(True, cu, cu, 7, 7, slots, None, None)
            assert attention_with_prologue(attn, pos, qkv, *norms, _Rope(cs)).shape == (40, 16, D)
        else:
            k_new, out = torch.empty(40, 8, D, dtype=qkv.dtype).cuda(), torch.empty(
                40, 16, D, dtype=qkv.dtype).cuda()
            cu2 = torch.zeros(2, dtype=torch.int32).cuda()
            cs2 = cs.view(cs.shape[0], -1)
            _lib.check(_lib.load().nvk_varlen_prefill_prologue(
                qkv.data_ptr(), qkv.stride(0), 40, pos.data_ptr(), w[0].data_ptr(),
                w[1].data_ptr(), EPS, cs2.data_ptr(), cs2.stride(0), cs2.shape[0], k2.data_ptr(),
                v2.data_ptr(), slots.data_ptr(), k2.shape[0] * k2.shape[1], k_new.data_ptr(),
                cu2.data_ptr(), cu2.data_ptr(), 1, 0, 0, None, 0, 0, 0, 0, 16, 8, D, D ** -0.5,
                out.data_ptr(), out.stride(0), out.stride(1), None, 0, None, 0,
                _lib.dtype_code(qkv), _lib.stream_ptr(qkv.device)))
        qk_norm_rope_store(pos, qkv, 16, 8, D, w[0], w[1], EPS, cs, kc, vc, slots)
        torch.cuda.synchronize()
    finally:
        reset_context()
    assert torch.equal(k2, kc) and torch.equal(v2, vc)
