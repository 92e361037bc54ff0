"""fp32 attention on the fp32 matrix cores (head_dim 64 and 128) against the fp64 oracle.

Sizes sit at the kernel's edges: 16-key tiles, blocks of 16 rows (with
groupings that fill them oddly), a single key, more keys than four waves'
tiles, pinned splits, rows whose block reaches past keys they do not see,
more blocks than work-groups, and more sequences than one scan covers. Bound: fp32's 1e-5 (the sums run over at most a few thousand
products of N(0, 1) values, ~1e-6 off).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from liteinfer_amd.paged_kernels import paged_decode, paged_prefill
from tests.helpers import PagedBatch, to_numpy

pytestmark = pytest.mark.gpu


def _prefill(b, **kw):
    return paged_prefill(b.query, b.key_pool, b.value_pool, b.slot_table, b.context_lens_t, b.query_start_loc,
                         max(b.query_lens), b.scaling, b.groups, **kw)


def _close(actual, expected):
    np.testing.assert_allclose(to_numpy(actual), expected, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("groups", [1, 4, 5, 16, 20])
@pytest.mark.parametrize("num_splits", [None, 3])
def test_decode(head_dim, groups, num_splits):
    b = PagedBatch([1, 15, 16, 17, 63, 64, 65, 1000, 2500], num_heads=3 * groups, num_kv_heads=3, head_dim=head_dim)
    _close(paged_decode(b.query, b.key_pool, b.value_pool, b.slot_table, b.context_lens_t, b.scaling, b.groups,
                        num_splits=num_splits), b.oracle())


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("groups", [1, 3, 4, 16, 20])
def test_packed(head_dim, groups):
    q = [1, 2, 4, 8, 9, 16, 17, 33, 100, 1]
    ctx = [1, 2, 90, 8, 25, 300, 17, 64, 163, 700]
    b = PagedBatch(ctx, q, num_heads=2 * groups, num_kv_heads=2, head_dim=head_dim)
    _close(_prefill(b), b.oracle())
    # Through strided rows (the packed boundary's transposed query) too.
    wide = torch.randn(b.query.shape[1], b.query.shape[0], head_dim, device="cuda").copy_(b.query.transpose(0, 1))
    strided = paged_prefill(wide.transpose(0, 1), b.key_pool, b.value_pool, b.slot_table, b.context_lens_t,
                            b.query_start_loc, max(q), b.scaling, b.groups)
    assert torch.equal(strided, _prefill(b))


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_a_row_is_not_touched_by_values_it_does_not_see(value):
    """A later token's V row holds an infinity or a NaN: earlier rows stay what they were."""
    b = PagedBatch([70, 40], [30, 40], num_heads=8, num_kv_heads=2, head_dim=64)
    b.slot_table = torch.arange(140, device="cuda").reshape(2, 70)  # a slot per position
    want = _prefill(b)
    b.value_pool[60] = value  # position 60 of sequence 0: its queries are positions 40 .. 69
    got = _prefill(b)
    assert torch.equal(got[:20], want[:20]) or torch.allclose(got[:20], want[:20], rtol=1e-5, atol=1e-5)
    assert not torch.isfinite(got[20:30]).any()
    assert torch.equal(got[30:], want[30:])


def test_an_unaligned_row_takes_the_general_kernel():
    b = PagedBatch([40, 90], head_dim=64)
    odd = torch.zeros(b.query.numel() + 1, device="cuda")[1:].view(b.query.shape).copy_(b.query)
    _close(paged_decode(odd, b.key_pool, b.value_pool, b.slot_table, b.context_lens_t, b.scaling, b.groups), b.oracle())


def test_an_empty_context_is_nan():
    b = PagedBatch([5, 9], head_dim=64)
    lens = torch.tensor([0, 9], dtype=torch.int32, device="cuda")
    out = paged_decode(b.query, b.key_pool, b.value_pool, b.slot_table, lens, b.scaling, b.groups)
    assert torch.isnan(out[0]).all() and torch.isfinite(out[1]).all()


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("ctx", [1, 16, 17, 33, 49, 65, 1000])
@pytest.mark.parametrize("num_splits", [None, 3])
def test_a_nan_in_the_newest_key_reaches_the_result(ctx, num_splits, head_dim):
    """At 17, 33 and 49 keys one wave's only key is the newest, so every score that it sees is a NaN."""
    b = PagedBatch([ctx, 50], num_heads=8, num_kv_heads=2, head_dim=head_dim, num_slots=2048)
    b.slot_table = torch.arange(2 * max(ctx, 50), device="cuda").reshape(2, -1)
    b.key_pool[ctx - 1, 0] = float("nan")  # of the first KV head
    out = paged_decode(b.query, b.key_pool, b.value_pool, b.slot_table, b.context_lens_t, b.scaling, b.groups,
                       num_splits=num_splits)
    assert torch.isnan(out[0, :4]).all() and torch.isfinite(out[0, 4:]).all() and torch.isfinite(out[1]).all()


def test_a_packed_row_sees_a_nan_key_of_its_own():
    """The last query alone sees the last key, which is a tile and one wave's whole share."""
    b = PagedBatch([17, 33], [2, 3], num_heads=2, num_kv_heads=2, head_dim=64)
    b.slot_table = torch.arange(66, device="cuda").reshape(2, 33)
    want = _prefill(b)
    b.key_pool[[16, 65]] = float("nan")
    got = _prefill(b)
    assert torch.isnan(got[[1, 4]]).all()
    np.testing.assert_allclose(to_numpy(got[[0, 2, 3]]), to_numpy(want[[0, 2, 3]]), rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("ctx", [17, 40])
def test_infinite_scores(ctx):
    """A newest key of an infinite score: minus infinity weighs nothing, plus infinity is a NaN."""
    b = PagedBatch([ctx], num_heads=8, num_kv_heads=2, head_dim=64)
    b.slot_table = torch.arange(ctx, device="cuda").reshape(1, ctx)
    b.key_pool[ctx - 1, :, 0] = float("inf")
    args = (b.scaling, b.groups)
    got = paged_decode(b.query, b.key_pool, b.value_pool, b.slot_table, b.context_lens_t, *args)
    without = paged_decode(b.query, b.key_pool, b.value_pool, b.slot_table, b.context_lens_t - 1, *args)
    up = b.query[0, :, 0] > 0
    assert up.any() and not up.all()
    assert torch.isnan(got[0, up]).all()
    np.testing.assert_allclose(to_numpy(got[0, ~up]), to_numpy(without[0, ~up]), rtol=1e-5, atol=1e-5)


def test_the_longest_chunk_may_be_overstated():
    """`max_query_len` bounds the chunks; the grid does not grow with what it overstates."""
    b = PagedBatch([20, 9], [3, 9], num_heads=32, num_kv_heads=2, head_dim=64)
    got = paged_prefill(b.query, b.key_pool, b.value_pool, b.slot_table, b.context_lens_t, b.query_start_loc,
                        2 ** 31 - 1, b.scaling, b.groups)
    assert torch.equal(got, _prefill(b))


def test_a_decode_step_of_more_units_than_a_launch_holds():
    """2^24 units of 256 threads are past a launch's 2^32: the general kernel serves them."""
    batch, heads = 2 ** 24 // 32, 32
    b = PagedBatch([1], num_heads=heads, num_kv_heads=heads, head_dim=64)
    table = torch.arange(batch, device="cuda").remainder(512).view(batch, 1)
    lens = torch.ones(batch, dtype=torch.int32, device="cuda")
    out = paged_decode(b.query.expand(batch, heads, 64), b.key_pool, b.value_pool, table, lens, b.scaling, 1)
    assert torch.equal(out.view(-1, 512, heads, 64), b.value_pool.expand(batch // 512, 512, heads, 64))


@pytest.mark.parametrize("head_dim", [64, 128])
def test_work_groups_take_several_units(head_dim):
    """Blocks past the capped grid: 6 work-groups a CU over the KV heads walk them."""
    q = [1, 400, 150, 97, 700]
    b = PagedBatch([300, 410, 150, 160, 731], q, num_heads=32, num_kv_heads=8, head_dim=head_dim)
    per_head = sum(-(-n * b.groups // 16) for n in q)
    assert per_head > -(-torch.cuda.get_device_properties(0).multi_processor_count * 6 // 8)
    _close(_prefill(b), b.oracle())


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("batch", [64, 65, 130])
def test_packed_past_one_scan_of_the_sequences(batch, head_dim):
    """64 sequences' counts a scan, some of them bringing no query, the last one the longest chunk."""
    q = [(3, 0, 1, 17, 0)[i % 5] for i in range(batch - 1)] + [40]
    ctx = [n + 7 * i % 60 + (n == 0) for i, n in enumerate(q)]
    b = PagedBatch(ctx, q, num_heads=8, num_kv_heads=2, head_dim=head_dim)
    _close(_prefill(b), b.oracle())
