"""flash_attn_with_kvcache with several queries per sequence through
nvk_paged_verify (lengths read as they are, no cu_seqlens) against the oracle and
against the varlen call over explicit cu_seqlens: rows up to the kernels' 16,
contexts at chunk and page edges, shorter than the query block or empty, one and
two chunks per wave, K through LDS, strided q."""
import pytest
import torch

from gpu_utils import assert_attn_close, oracle_prefill_paged, say
from nanovllm_amd import _lib, flash_attn_with_kvcache, varlen_prefill
from test_gpu_prefill_split import _paged_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nq,hq,hkv,lens,bs", [
    (6, 16, 8, [6, 31, 32, 33, 255, 256, 257, 1000], 256),
    (8, 16, 8, [3, 8, 0, 700], 64),              # shorter than the query block, empty
    (2, 16, 2, [2, 90, 4100], 32),
    (4, 8, 2, [500] * 3, 256),
    (16, 4, 4, [40, 2000], 256),
    (3, 16, 8, [9000], 256),                     # one sequence: sliced combine
    (6, 16, 8, [900 + 61 * i for i in range(40)], 256),   # K through LDS
])
def test_verify_matches_oracle_and_varlen(nq, hq, hkv, lens, bs):
    b = len(lens)
    q, kc, vc, bt, cu_q, cu_k = _paged_case(51, [nq] * b, lens, bs, hq, hkv)
    assert _lib.load().nvk_paged_verify_workspace_size(b, nq, hq, hkv, 128, bs, bt.shape[1]) > 0
    scale = 128 ** -0.5
    say(f"verify {nq} queries, {hq}/{hkv} heads over {lens}")
    kd, vd, btd, lt = kc.cuda(), vc.cuda(), bt.cuda(), torch.tensor(lens, dtype=torch.int32).cuda()
    wide = torch.zeros(b, nq, hq, 144, dtype=q.dtype, device="cuda")
    wide[..., 8:136] = q.cuda().view(b, nq, hq, 128)
    call = lambda x: flash_attn_with_kvcache(x, kd, vd, cache_seqlens=lt, block_table=btd,
                                             softmax_scale=scale, causal=True)
    out = call(q.cuda().view(b, nq, hq, 128))
    strided = call(wide[..., 8:136])
    other = varlen_prefill(q.cuda(), kd, vd, cu_q.cuda(), cu_k.cuda(), nq, scale, block_table=btd)
    torch.cuda.synchronize()
    ref = oracle_prefill_paged(q, kc, vc, bt, cu_q, cu_k, bs, scale)
    assert out.shape == (b, nq, hq, 128)
    assert_attn_close(out.view(-1, hq, 128), ref, "verify")
    assert_attn_close(other, ref, "varlen")
    assert torch.equal(strided, out)


def test_sizes_that_stay_on_the_general_path():
    size = _lib.load().nvk_paged_verify_workspace_size
    assert size(4, 9, 16, 8, 128, 256, 8) == 0       # 18 rows
    assert size(4, 6, 16, 8, 64, 256, 8) == 0        # head_dim 64
    assert size(4, 6, 16, 8, 128, 48, 8) == 0        # pages of 48 keys
    assert size(4, 5, 9, 3, 128, 256, 8) == 0        # 3 heads per kv head
    assert size(0, 6, 16, 8, 128, 256, 8) == 0
