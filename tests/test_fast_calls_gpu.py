"""The C++ host side of the eager calls does what the Python code does, over the forms both accept."""

from __future__ import annotations

import pytest
import torch

from liteinfer_amd import _native
from liteinfer_amd.paged_kernels import paged_decode, paged_prefill
from liteinfer_amd.rope import rope_kv_write
from tests.helpers import PagedBatch

pytestmark = pytest.mark.gpu


class _Counting:
    """The module, counting the calls it served; or one that serves none."""

    def __init__(self, serve):
        self.real, self.serve, self.served = _native.fast_calls(), serve, 0

    def _run(self, fn, args):
        out = fn(*args) if self.serve else None
        self.served += out is not None
        return out

    def decode(self, *a):
        return self._run(self.real.decode, a)

    def prefill(self, *a):
        return self._run(self.real.prefill, a)

    def rope(self, *a):
        return self._run(self.real.rope, a)


def _both(monkeypatch, call):
    """(result through C++, result through Python, calls C++ served); raised errors as (type, text)."""
    got = []
    for serve in (True, False):
        counting = _Counting(serve)
        monkeypatch.setattr(_native, "_fast", counting)
        try:
            got.append(call())
        except Exception as e:  # compared below
            got.append((type(e), str(e)))
        served = counting.served if serve else served  # noqa: F821
        monkeypatch.setattr(_native, "_fast", counting.real)
    return got[0], got[1], served


def _same(a, b):
    if isinstance(a, torch.Tensor):
        return a.dtype == b.dtype and a.stride() == b.stride() and torch.equal(a.nan_to_num(), b.nan_to_num())
    return a == b


FORMS = {
    "plain": (lambda b: {}, True),
    "strided query": (lambda b: {"query": b.query.repeat(1, 1, 2)[:, :, :b.head_dim]}, True),
    "query a copy away": (lambda b: {"query": b.query.transpose(1, 2).contiguous().transpose(1, 2)}, False),
    "int32 table": (lambda b: {"slot_table": b.slot_table.to(torch.int32)}, False),
    "int64 lengths": (lambda b: {"context_lens": b.context_lens_t.long()}, False),
    "narrowed table": (lambda b: {"slot_table": torch.cat((b.slot_table, b.slot_table), 1)[:, :b.slot_table.shape[1]]}, True),
    "transposed table": (lambda b: {"slot_table": b.slot_table.t().contiguous().t()}, False),
    "pinned splits": (lambda b: {"num_splits": 3, "kernel": "equal_splits"}, True),
    "general kernel": (lambda b: {"kernel": "generic"}, True),
    "unknown kernel": (lambda b: {"kernel": "nonsense"}, False),
    "wrong groups": (lambda b: {"num_kv_groups": 3}, False),
    "one new row": (lambda b: {"new_key": torch.zeros(b.query.shape[0], 2, b.head_dim, dtype=b.dtype, device="cuda")}, False),
    "numpy scale": (lambda b: {"scaling": __import__("numpy").float32(b.scaling)}, False),
    "pools unlike": (lambda b: {"value_pool": torch.cat((b.value_pool, b.value_pool), 2)[:, :, :b.head_dim]}, False),
}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("form", FORMS)
def test_decode(monkeypatch, dtype, form):
    b = PagedBatch([5, 70, 33], dtype=dtype, head_dim=64)
    change, fast = FORMS[form]
    kw = {"query": b.query, "key_pool": b.key_pool, "value_pool": b.value_pool, "slot_table": b.slot_table,
          "context_lens": b.context_lens_t, "scaling": b.scaling, "num_kv_groups": b.groups} | change(b)
    got, want, served = _both(monkeypatch, lambda: paged_decode(**kw))
    assert _same(got, want) and served == int(fast)


PACKED = {
    "plain": (lambda b: {}, True),
    "rows apart": (lambda b: {"one_query_rows": False}, True),
    "general kernel": (lambda b: {"kernel": "generic"}, True),
    "given out": (lambda b: {"out": torch.zeros(b.query.shape[1], b.query.shape[0], b.head_dim, dtype=b.dtype,
                                                device="cuda").transpose(0, 1)}, True),
    "out of another shape": (lambda b: {"out": b.query[:1].clone()}, False),
    "heads first": (lambda b: {"query": b.query.transpose(0, 1).contiguous().transpose(0, 1)}, True),
    "int64 offsets": (lambda b: {"query_start_loc": b.query_start_loc.long()}, False),
    "offsets of another batch": (lambda b: {"query_start_loc": b.query_start_loc[:-1]}, False),
    "splits pinned": (lambda b: {"kernel": "equal_splits"}, False),
}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("form", PACKED)
def test_prefill(monkeypatch, dtype, form):
    b = PagedBatch([5, 70, 33], [5, 40, 1], dtype=dtype, head_dim=64)
    change, fast = PACKED[form]
    kw = {"query": b.query, "key_pool": b.key_pool, "value_pool": b.value_pool, "slot_table": b.slot_table,
          "context_lens": b.context_lens_t, "query_start_loc": b.query_start_loc, "max_query_len": 40,
          "scaling": b.scaling, "num_kv_groups": b.groups} | change(b)
    got, want, served = _both(monkeypatch, lambda: paged_prefill(**kw))
    assert _same(got, want) and served == int(fast)
    if "given" in form:
        assert got is kw["out"]


@pytest.mark.parametrize("fp8", [False, True])
def test_decode_writes_the_newest_rows(monkeypatch, fp8):
    b = PagedBatch([5, 70, 33], dtype=torch.bfloat16, head_dim=128)
    b.slot_table = torch.arange(210, device="cuda").reshape(3, 70)
    new = [torch.randn(3, 2, 128, device="cuda").to(torch.bfloat16) for _ in range(2)]
    kw = {"k_scale": 0.02, "v_scale": 0.03} if fp8 else {}

    def call():
        pools = [(p.float() / 4).to(torch.float8_e4m3fn) if fp8 else p.clone() for p in (b.key_pool, b.value_pool)]
        out = paged_decode(b.query, *pools, b.slot_table, b.context_lens_t, b.scaling, b.groups, new_key=new[0],
                           new_value=new[1], **kw)
        return torch.cat([out.float().flatten()] + [p.float().flatten() for p in pools])

    got, want, served = _both(monkeypatch, call)
    assert _same(got, want) and served == 1


@pytest.mark.parametrize("case", ["plain", "broadcast tables", "fp8", "float32", "sin apart", "int32 slots", "bad scale",
                                  "wrong bad_slots", "odd dim"])
def test_rope(monkeypatch, case):
    dtype = torch.float32 if case == "float32" else torch.bfloat16
    dim = 63 if case == "odd dim" else 64
    g = torch.Generator(device="cuda").manual_seed(1)
    qkv = torch.randn(3, 5, 12, dim, generator=g, device="cuda").to(dtype)
    q, k, v = (t.transpose(1, 2) for t in qkv.split([8, 2, 2], 2))
    cos, sin = (torch.randn(1 if "broadcast" in case else 3, 5, dim, generator=g, device="cuda").to(dtype) for _ in range(2))
    if case == "sin apart":
        sin = torch.cat((sin, sin), 2)[:, :, :dim]
    slots = torch.randperm(30, generator=g, device="cuda")[:15]
    if case == "int32 slots":
        slots = slots.to(torch.int32)
    kw = {"k_scale": 0.0 if case == "bad scale" else 0.02, "v_scale": 0.03}
    bad = torch.zeros(1, dtype=torch.int64 if case == "wrong bad_slots" else torch.int32, device="cuda")
    pool_dtype = torch.float8_e4m3fn if case in ("fp8", "bad scale") else dtype

    def call():
        pools = [torch.zeros(30, 2, dim, device="cuda").to(pool_dtype) for _ in range(2)]
        out = rope_kv_write(q, k, v, cos, sin, slots, *pools, bad_slots=bad, **kw)
        assert out.transpose(1, 2).is_contiguous()
        return torch.cat([out.float().flatten()] + [p.float().flatten() for p in pools])

    got, want, served = _both(monkeypatch, call)
    assert _same(got, want) and served == int(case in ("plain", "broadcast tables", "fp8", "float32"))
