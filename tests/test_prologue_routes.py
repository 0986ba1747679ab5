"""Which calls the prefill of attention_with_prologue makes, on the CPU: the
library is replaced by a record of the calls, so that arguments the kernels must
not see are tested without launching anything on them."""
import types

import pytest
import torch

from nanovllm_amd import Attention, _lib, attention_with_prologue
from nanovllm_amd.utils.context import reset_context, set_context

T, HQ, HKV, D, PAGE = 5, 16, 8, 128, 16


class _Calls:
    """Every library function, recorded and successful; sizes are 0."""

    def __init__(self):
        self.names = []

    def __getattr__(self, name):
        if name.endswith("_size"):
            return lambda *a: 0

        def call(*a):
            self.names.append(name)
            return 0
        return call


@pytest.fixture
def calls(monkeypatch):
    lib = _Calls()
    monkeypatch.setattr(_lib, "load", lambda: lib)
    monkeypatch.setattr(_lib, "require_gpu", lambda *ts: torch.device("cpu"))
    monkeypatch.setattr(_lib, "stream_ptr", lambda dev: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    yield lib.names
    reset_context()


ONE = ["nvk_varlen_prefill_prologue"]
TWO = ["nvk_qk_norm_rope_store", "nvk_varlen_prefill_ordered"]


def _args(k_cache=None, v_cache=None, paged=True, slots=True, scale=D ** -0.5):
    attn = Attention(HQ, D, scale, HKV)
    shape = (4, PAGE, HKV, D)
    attn.k_cache = torch.zeros(shape, dtype=torch.bfloat16) if k_cache is None else k_cache
    attn.v_cache = torch.zeros(shape, dtype=torch.bfloat16) if v_cache is None else v_cache
    cu = torch.tensor([0, T], dtype=torch.int32)
    set_context(True, cu, cu, T, T, torch.zeros(T, dtype=torch.int32) if slots else None, None,
                torch.zeros(1, 1, dtype=torch.int32) if paged else None)
    norm = types.SimpleNamespace(weight=torch.ones(D, dtype=torch.bfloat16), eps=1e-6)
    rope = types.SimpleNamespace(cos_sin_cache=torch.zeros(64, 1, D))
    qkv = torch.zeros(T, (HQ + 2 * HKV) * D, dtype=torch.bfloat16)
    return attn, torch.arange(T), qkv, norm, norm, rope


@pytest.mark.parametrize("paged", [True, False])
@pytest.mark.parametrize("slots", [True, False])
def test_ordinary_prefill_is_one_call(calls, paged, slots):
    out = attention_with_prologue(*_args(paged=paged, slots=slots))
    assert calls == ONE and out.shape == (T, HQ, D)


def _zeros(*shape, dtype=torch.bfloat16):
    return torch.zeros(*shape, dtype=dtype)


@pytest.mark.parametrize("what,k,v", [
    ("cache of another type", _zeros(4, PAGE, HKV, D, dtype=torch.float16),
     _zeros(4, PAGE, HKV, D, dtype=torch.float16)),
    ("fewer value pages than key pages", _zeros(4, PAGE, HKV, D), _zeros(2, PAGE, HKV, D)),
    ("half the head_dim, twice the heads", _zeros(4, PAGE, 2 * HKV, D // 2),
     _zeros(4, PAGE, 2 * HKV, D // 2)),
    ("three dimensions", _zeros(4, PAGE, HKV * D), _zeros(4, PAGE, HKV * D)),
    ("every other page", _zeros(8, PAGE, HKV, D)[::2], _zeros(8, PAGE, HKV, D)[::2]),
])
@pytest.mark.parametrize("slots", [True, False])
def test_caches_the_attention_refuses(calls, what, k, v, slots):
    with pytest.raises((_lib.NvkError, AssertionError)):
        attention_with_prologue(*_args(k, v, slots=slots))
    assert "nvk_varlen_prefill_prologue" not in calls
    assert "nvk_varlen_prefill_ordered" not in calls


def test_caches_of_another_head_count_are_read_as_they_are(calls):
    """Without slots nothing is stored and the caches' own head count holds."""
    attention_with_prologue(*_args(_zeros(4, PAGE, 4, D), _zeros(4, PAGE, 4, D), slots=False))
    assert calls == TWO


@pytest.mark.parametrize("where", ["instance", "class"])
def test_a_replaced_forward_runs(calls, monkeypatch, where):
    """attention_with_prologue returns what the call of the module returns, also
    where its forward was replaced (the way some libraries attach hooks)."""
    args = _args()
    attn, inner = args[0], Attention.forward
    if where == "instance":
        attn.forward = lambda *a, **kw: (inner(attn, *a, **kw), "seen")
    else:
        monkeypatch.setattr(Attention, "forward", lambda *a, **kw: (inner(*a, **kw), "seen"))
    out, mark = attention_with_prologue(*args)
    assert mark == "seen" and calls == TWO and out.shape == (T, HQ, D)


def test_a_compiled_module_is_called(calls):
    args = _args()
    attn, called = args[0], []
    attn.compile(backend="eager")
    assert attn._compiled_call_impl is not None
    attn._compiled_call_impl = lambda *a, **kw: called.append(1) or attn._call_impl(*a, **kw)
    attention_with_prologue(*args)
    assert called == [1] and calls == TWO


def test_no_scale_is_the_default_scale(calls):
    out = attention_with_prologue(*_args(scale=None))
    assert calls == ONE and out.shape == (T, HQ, D)


@pytest.mark.skipif(torch.cuda.is_available(),
                    reason="passes fake device pointers; only runs where nothing can launch")
def test_prefill_prologue_without_queries_runs_the_prologue():
    """A step of no sequence (or no query bound) still stores its k and v, so the
    prologue's own checks hold there; without tokens there is nothing to do."""
    lib = _lib.load()
    # qkv, stride, T, pos, qw, kw, eps, cos_sin, cs_stride, max_pos, k/v cache, slots,
    # cache_slots, k_new, cu_q, cu_k, batch, max_q, max_k, tables, bt_stride, max_blocks, bs, nb,
    # heads, D, scale, out, out strides, ws, ws_bytes, order, order_bytes, dtype, stream
    a = [16, 32 * 128, 4, 16, 16, 16, -1.0, 16, 128, 4096, 16, 16, 16, 1 << 20, 16, 16, 16, 0, 7, 7,
         None, 0, 0, 0, 0, 16, 8, 128, 0.088, 16, 16 * 128, 128, None, 0, None, 0, 0, None]
    assert lib.nvk_varlen_prefill_prologue(*a) == -1             # eps < 0, batch 0
    a[17], a[18] = 2, 0
    assert lib.nvk_varlen_prefill_prologue(*a) == -1             # eps < 0, max_seqlen_q 0
    empty = list(a)
    empty[6] = 1e-6
    for i in (0, 3, 10, 11, 12, 14, 29):
        empty[i] = None
    empty[2] = empty[17] = 0
    assert lib.nvk_varlen_prefill_prologue(*empty) == 0          # no token, no sequence
