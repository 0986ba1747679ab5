"""Prefill steps whose query tiles leave workgroup slots idle are cut into parts
along the keys (the workspace of nvk_varlen_prefill_parts_workspace_size), then
merged.  The parts' result is checked against the oracle and against the same
call without a workspace, at sizes on both sides of the rule, with tiles that
keep one part beside cut ones, partly empty first tiles and ragged batches."""
import pytest
import torch

from gpu_utils import assert_attn_close, oracle_prefill_paged, say
from nanovllm_amd import _lib, varlen_prefill
from test_gpu_prefill_split import _call, _paged_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens_q,lens_k,hq,hkv,bs", [
    ([65], [1500], 16, 8, 256),              # two query tiles, the first with one token
    ([100], [1100], 16, 8, 16),              # per-row page lookups
    ([130, 33, 1], [3000, 600, 700], 16, 8, 256),   # ragged: short sequences keep one part
    ([300], [2500], 4, 2, 64),
    ([129], [1300], 8, 8, 256),              # one head per kv head
    ([40], [2050], 16, 2, 256),              # eight: 16 tokens per tile
    ([200, 0, 90], [200, 900, 2000], 4, 2, 256),    # no query; no prefix
    ([1000], [1000], 4, 2, 256),             # a prompt alone: 1 to 16 key tiles
])
def test_parts_match_whole_tiles_and_oracle(lens_q, lens_k, hq, hkv, bs):
    q, kc, vc, bt, cu_q, cu_k = _paged_case(91, lens_q, lens_k, bs, hq, hkv)
    scale = 128 ** -0.5
    mq, mk = max(lens_q), max(lens_k)
    lib = _lib.load()
    old = lib.nvk_varlen_prefill_workspace_size(len(lens_q), mq, mk, hq, hkv, 128)
    new = lib.nvk_varlen_prefill_parts_workspace_size(len(lens_q), mq, mk, hq, hkv, 128)
    assert new > old, "the rule gives no parts here"
    dev = [t.cuda() for t in (q, kc, vc, cu_q, cu_k)]
    what = f"parts {lens_q} over {lens_k}, {hq}/{hkv} heads, page {bs}"
    say(what)
    whole, _ = _call(*dev, mq, mk, scale, bt=bt.cuda(), use_ws=False)
    for strided in (False, True):     # whole-row stores, then 8-byte aligned rows
        out = torch.full((q.shape[0], hq, 132), float("nan"), dtype=q.dtype, device="cuda")
        out = out[..., 4:] if strided else out[..., :128].contiguous()
        varlen_prefill(*dev[:3], dev[3], dev[4], mq, scale, block_table=bt.cuda(), out=out,
                       max_seqlen_k=mk)
        torch.cuda.synchronize()
        assert_attn_close(out, oracle_prefill_paged(q, kc, vc, bt, cu_q, cu_k, bs, scale), what)
        # both round f32 sums of the same products to bf16: at most a rounding step apart
        # (2^-8) on top of the probabilities' own rounding (2^-9 of values up to ~4)
        diff = (out.float() - whole.float()).abs()
        assert (diff <= 2.0 ** -8 * whole.float().abs() + 2.0 ** -7).all(), diff.max()


def test_rule_keeps_whole_tiles_where_parts_cost_more():
    size = _lib.load().nvk_varlen_prefill_parts_workspace_size
    assert size(1, 777, 777, 16, 8, 128) == 0        # one prompt: 104 workgroups, 13 tiles
    assert size(1, 4096, 12288, 16, 8, 128) == 0     # 512 workgroups
    assert size(1, 128, 128, 16, 8, 128) == 0
    for args in [(1, 1000, 9300, 16, 8, 128), (1, 200, 8200, 16, 8, 128), (8, 250, 8250, 16, 8, 128),
                 (1, 65, 1500, 1, 1, 128)]:
        need = size(*args)
        assert 0 < need <= 512 * 128 * 132 * 4 and need % (128 * 132 * 4) == 0
    # ranges of at most half a tile keep their own plan: up to 16 parts, 1024 workgroups and more
    plain = _lib.load().nvk_varlen_prefill_workspace_size
    for args, records in [((64, 20, 2048, 16, 8, 128), 1024), ((127, 20, 2048, 16, 8, 128), 2032),
                          ((1023, 8, 2048, 8, 1, 128), 2046), ((1024, 8, 2048, 8, 1, 128), 0)]:
        assert size(*args) == plain(*args) == records * 128 * 132 * 4
