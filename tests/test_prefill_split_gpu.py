"""Small packed passes cut into pieces without a work list (at most 64 sequences), against the fp64 oracle.

Sizes at the schedule's edges: one block and several a sequence, contexts
with and without enough visible stages to cut, sequences that bring nothing,
head counts of one work queue and of eight, the largest batch the schedule
takes and one past it. The bound is the packed bf16 bar (max-abs 2^-6).
"""

from __future__ import annotations

import pytest
import torch

from liteinfer_amd.paged_kernels import paged_prefill
from tests.helpers import PagedBatch, assert_within

pytestmark = pytest.mark.gpu

CASES = [
    # contexts, queries, query heads, KV heads
    ([4196], [100], 32, 8),
    ([1024], [64], 32, 8),
    ([1030], [6], 32, 8),
    ([2500, 40, 1300], [200, 40, 1], 16, 4),
    ([1500, 1100, 1024], [65, 0, 64], 6, 3),
    ([3000], [1], 16, 1),
    ([1100] * 9, [3] * 9, 16, 1),
    ([1100] * 64, [2] * 64, 2, 1),
    ([1100] * 65, [2] * 65, 2, 1),
]


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("ctx,q,heads,kv_heads", CASES)
def test_split_pass(ctx, q, heads, kv_heads, head_dim):
    b = PagedBatch(ctx, q, dtype=torch.bfloat16, num_heads=heads, num_kv_heads=kv_heads, head_dim=head_dim,
                   num_slots=4096, seed=len(ctx) + heads)
    out = paged_prefill(b.query, b.key_pool, b.value_pool, b.slot_table, b.context_lens_t, b.query_start_loc, max(q),
                        b.scaling, b.groups, one_query_rows=False)
    assert_within(out, b.oracle(), 2 ** -6, 2e-3)
