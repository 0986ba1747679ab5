"""Decodes that run on the short-query MFMA kernels (4 and 8 query heads per kv
head; with one and two the decode kernel) against the oracle: contexts at the edges of
chunks and pages, empty contexts, cut groups, strided q and out, both dtypes,
and the prologue form, whose prologue writes q into the output rows."""
import pytest
import torch

from gpu_utils import assert_attn_close, oracle_decode, say
from nanovllm_amd import (paged_decode, paged_decode_with_prologue, qk_norm_rope_store,
                          rope_cos_sin_cache)
from nanovllm_amd.workloads import decode_case

pytestmark = pytest.mark.gpu

EDGES = [1, 0, 31, 32, 33, 255, 256, 257, 0, 1500, 4097]


@pytest.mark.parametrize("hq,hkv,ctx,bs,width", [
    (16, 4, EDGES, 256, 0),
    (16, 2, EDGES, 32, 0),
    (8, 1, [9000], 256, 0),                       # one group over many waves: sliced combine
    (16, 2, [0, 0, 0], 256, 0),                   # nothing to read
    (16, 2, [300 + 7 * i for i in range(150)], 64, 0),
    # tables that could name 32 chunks of 32 keys for each of 1024 waves: K through LDS
    (16, 2, [300 + 7 * i for i in range(150)], 64, 56),
    (8, 1, [0, 33, 1] + [97 * i for i in range(61)], 256, 64),
    (4, 4, [1 + 37 * i for i in range(33)], 256, 0),     # one head: the decode kernel
    (4, 1, EDGES, 48, 0),                         # pages of 48 keys: too
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_decode_groups_match_oracle(hq, hkv, ctx, bs, width, dtype):
    pages = sum(-(-c // bs) for c in ctx)
    case = decode_case(seed=7, hq=hq, hkv=hkv, ctx=ctx, block_size=bs, pool_blocks=pages + 2,
                       width=max(1, width, max(-(-c // bs) for c in ctx)))
    q, kc, vc = (t.to(dtype) for t in (case.q, case.k_cache, case.v_cache))
    ref = oracle_decode(q, kc, vc, case.block_tables, case.context_lens, bs, case.scale)
    say(f"decode {hq}/{hkv} heads, {len(ctx)} sequences, page {bs}, width {width}, {dtype}")
    b = len(ctx)
    wide = torch.zeros(b, hq, 160, dtype=dtype, device="cuda")
    wide[..., 16:144] = q.cuda()
    out = torch.full((b, hq, 136), float("nan"), dtype=dtype, device="cuda")
    kc, vc, lens, bt = (t.cuda() for t in (kc, vc, case.context_lens, case.block_tables))
    paged_decode(wide[..., 16:144], kc, vc, lens, bt, case.scale, out=out[..., :128])
    plain = paged_decode(q.cuda(), kc, vc, lens, bt, case.scale)
    torch.cuda.synchronize()
    assert_attn_close(plain, ref, "contiguous")
    assert torch.equal(out[..., :128], plain), "strided rows give the same bits"
    assert out[..., 128:].isnan().all(), "nothing outside the rows is written"


@pytest.mark.parametrize("rows", ["contiguous", "padded", "head by head"])
@pytest.mark.parametrize("hq,hkv,ctx,width", [
    (16, 2, [1, 32, 33, 257, 0, 1700, 2900], 12), (16, 4, [1, 32, 33, 257, 0, 1700, 2900], 12),
    (16, 2, [1, 32, 33, 257, 0, 1700, 2900], 293),          # K through LDS
    (8, 1, [64 * i + 31 * (i % 3) for i in range(65)], 17),  # several groups to a wave
    (4, 4, [1, 32, 33, 257, 0, 1700, 2900] + [3 * i for i in range(30)], 12),   # the decode kernel
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_prologue_form_with_q_in_the_output_rows(rows, hq, hkv, ctx, width, dtype):
    bs = 256
    case = decode_case(seed=8, hq=hq, hkv=hkv, ctx=ctx, width=width,
                       pool_blocks=sum(-(-c // bs) for c in ctx) + 1)
    case.k_cache, case.v_cache = case.k_cache.to(dtype), case.v_cache.to(dtype)
    g = torch.Generator().manual_seed(9)
    qkv = (torch.randn(len(ctx), (hq + 2 * hkv) * 128, generator=g) * 2).to(dtype).cuda()
    w = (1 + 0.2 * torch.randn(2, 128, generator=g)).to(dtype).cuda()
    cs = rope_cos_sin_cache(128, 4096, 1e6).cuda()
    lens, bt = case.context_lens.cuda(), case.block_tables.cuda()
    pos = (lens - 1).long().clamp(min=0)
    slots = (bt.gather(1, (pos // bs)[:, None]).squeeze(1) * bs + pos % bs).to(torch.int32)
    slots[lens == 0] = -1
    caches = [[case.k_cache.cuda(), case.v_cache.cuda()] for _ in range(2)]
    say(f"prologue form {hq}/{hkv}, {len(ctx)} sequences, {rows} out, {dtype}")
    q, _, _ = qk_norm_rope_store(pos, qkv, hq, hkv, 128, w[0], w[1], 1e-6, cs, *caches[0], slots,
                                 return_k=False)
    ref = paged_decode(q, *caches[0], lens, bt, 128 ** -0.5)
    out = torch.empty(len(ctx), hq, 136 if rows == "padded" else 128, dtype=dtype, device="cuda")
    out = out[..., :128]
    if rows == "head by head":
        out = torch.empty(hq, len(ctx), 128, dtype=dtype, device="cuda").transpose(0, 1)
    slots[lens == 0] = 3      # a row without a context stores nothing, whatever its slot
    for _ in range(2):      # the second call finds the first one's outputs in out
        paged_decode_with_prologue(pos, qkv, hq, hkv, 128, w[0], w[1], 1e-6, cs, *caches[1], slots,
                                   lens, bt, 128 ** -0.5, out=out)
    torch.cuda.synchronize()
    assert torch.equal(out, ref)
    assert all(torch.equal(a, b) for a, b in zip(*caches))


@pytest.mark.parametrize("hq,hkv,ctx", [
    (16, 8, [1]), (16, 8, [1000]),                 # one chunk per wave
    (4, 2, [4096]), (4, 2, [4097]),                # 128 and 129 chunks per group
    (16, 8, [2048] * 2), (16, 8, [2080] * 2),          # 1024 chunks, and 65 per group
    (16, 8, [2048] * 3), (16, 8, [1024] * 5),          # more chunks, 64 and 32 per group
    (16, 8, [97] * 48), (16, 8, [129] * 32),       # 4 and 5 per group
    (16, 8, [225] * 24), (16, 8, [257] * 16), (16, 8, [1056] * 6),  # 8, 9 and 33
    (16, 8, [2048] * 4), (16, 8, [2048] * 4 + [1]),    # 2048 chunks (two for each wave) and more
    (16, 2, [3072] * 4), (16, 2, [3073] * 4),      # 768 chunks, and more, on the MFMA kernels
    (8, 1, [4096, 1]), (8, 1, [9000, 0, 1]),
])
def test_one_and_two_chunks_per_wave(hq, hkv, ctx):
    case = decode_case(seed=17, hq=hq, hkv=hkv, ctx=ctx, pool_blocks=sum(-(-c // 256) for c in ctx))
    ref = oracle_decode(case.q, case.k_cache, case.v_cache, case.block_tables, case.context_lens,
                        256, case.scale)
    c = case.to("cuda")
    say(f"decode {hq}/{hkv} over {ctx}")
    # a wider table than the contexts need: more waves in the grid than chunks
    wide = torch.full((len(ctx), c.block_tables.shape[1] + 40), -1, dtype=torch.int32, device="cuda")
    wide[:, :c.block_tables.shape[1]] = c.block_tables
    for bt in (c.block_tables, wide):
        out = paged_decode(c.q, c.k_cache, c.v_cache, c.context_lens, bt, case.scale)
        torch.cuda.synchronize()
        assert_attn_close(out, ref, f"{hq}/{hkv} {ctx}")


def _float64_decode(q, kc, vc, bt, ctx, scale):
    """The plain decode in float64, on the caches' device."""
    hkv, g, page = kc.shape[2], q.shape[1] // kc.shape[2], kc.shape[1]
    ref = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for i, n in enumerate(ctx):
        pages = bt[i, :-(-n // page)].long()
        k, v = (c[pages].flatten(0, 1)[:n].double() for c in (kc, vc))
        for h in range(hkv):
            rows = slice(h * g, (h + 1) * g)
            p = torch.softmax(q[i, rows].double() @ k[:, h].t().contiguous() * scale, -1)
            ref[i, rows] = p @ v[:, h].contiguous()
    return ref


INFINITE = [  # hq, hkv, contexts
    (16, 2, [1, 20, 32]), (16, 4, [20]),            # groups that one wave finishes
    (8, 8, [5 + i for i in range(28)] * 2),
    (16, 8, [20]), (16, 8, [64, 70]), (16, 2, [64, 200]),   # cut into 2, 3 and 7 parts
    (16, 8, [2000]), (16, 2, [2000]), (8, 1, [3000]),       # the sliced merges
]


@pytest.mark.parametrize("hq,hkv,ctx", INFINITE)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_infinite_values_stay_infinite(hq, hkv, ctx, dtype):
    """A value of +-inf gives +-inf in its dimension, not NaN: no probability here
    rounds to 0, and nothing may multiply it by 0 on the side."""
    case = decode_case(seed=19, hq=hq, hkv=hkv, ctx=ctx, pool_blocks=sum(-(-c // 256) for c in ctx))
    q, kc, vc = (t.to(dtype).cuda() for t in (case.q, case.k_cache, case.v_cache))
    bt, lens = case.block_tables.cuda(), case.context_lens.cuda()
    for i, n in enumerate(ctx):     # the first key and the last
        for pos, dim, x in ((0, 5, float("inf")), (n - 1, 100, float("-inf"))):
            vc[bt[i, pos // 256].long(), pos % 256, :, dim] = x
    say(f"infinite values, {hq}/{hkv} heads, {len(ctx)} sequences of {min(ctx)}-{max(ctx)}, {dtype}")
    out = paged_decode(q, kc, vc, lens, bt, case.scale).double()
    ref = _float64_decode(q, kc, vc, bt, ctx, case.scale)
    torch.cuda.synchronize()
    assert ref[..., 5].eq(float("inf")).all() and ref[..., 100].eq(float("-inf")).all()
    torch.testing.assert_close(out, ref, atol=2e-2, rtol=1e-2)


@pytest.mark.parametrize("hq,hkv,b", [(16, 2, 24), (16, 4, 24), (8, 8, 40)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_no_less_exact_than_the_decode_kernel(hq, hkv, b, dtype):
    """Pages of 16 keys stay on the decode kernel: over the same keys its error
    against float64 bounds the MFMA kernels'.  With one head per kv head both
    page sizes are its own, and give the same bits."""
    ctx = [200 + 61 * i for i in range(b)]
    case = decode_case(seed=27, hq=hq, hkv=hkv, ctx=ctx, pool_blocks=sum(-(-c // 256) for c in ctx))
    q, kc, vc = (t.to(dtype).cuda() for t in (case.q, case.k_cache, case.v_cache))
    bt, lens = case.block_tables.cuda(), case.context_lens.cuda()
    fine = (bt[..., None] * 16 + torch.arange(16, device="cuda", dtype=torch.int32)).flatten(1)
    fine[(bt < 0).repeat_interleave(16, 1)] = -1
    ref = _float64_decode(q, kc, vc, bt, ctx, case.scale)
    say(f"decode {hq}/{hkv} heads, {b} sequences, {dtype}, error against float64")
    here = paged_decode(q, kc, vc, lens, bt, case.scale)
    there = paged_decode(q, kc.view(-1, 16, hkv, 128), vc.view(-1, 16, hkv, 128), lens,
                         fine.contiguous(), case.scale)
    err = [((o.double() - ref).norm() / ref.norm()).item() for o in (here, there)]
    print(f"MFMA kernels {err[0]:.6f}, decode kernel {err[1]:.6f}")
    assert err[0] <= err[1]
    assert hq > hkv or torch.equal(here, there)
