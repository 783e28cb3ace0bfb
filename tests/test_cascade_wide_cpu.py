"""Which shared-prefix launches take wide prefix workgroups (``flashdec_amd.cascade.plan_wide_cascade``).

Worked for 256 CUs; each refused shape measured slower with them (the figures stand beside the rule).  No counterpart
in the reference.
"""

import pytest
import torch

from flashdec_amd import cascade


def _plan(hq, hkv, sizes, prefixes, tail=512, known=True, head_dim=128):
    prefixes = [prefixes] * len(sizes) if isinstance(prefixes, int) else prefixes
    rows = sum(sizes)
    g = cascade.CascadeGroups(
        members=torch.zeros((len(sizes), max(sizes)), dtype=torch.int32),
        prefix_len=torch.tensor(prefixes, dtype=torch.int32), row_prefix_len=torch.zeros(rows, dtype=torch.int32),
        max_prefix_len=max(prefixes), max_tail_len=tail, total_tail_len=rows,
        shared_tokens=sum(n * p for n, p in zip(sizes, prefixes)) if known else None)
    return cascade.plan_wide_cascade(rows, hq, hkv, head_dim, g, 256)


@pytest.mark.parametrize("case", [
    (16, 2, [4] * 12, 8192),    # 32 of 128 rows
    (16, 2, [2] * 40, 16384),   # 16
    (8, 8, [2] * 32, 16384),    # 2, on 256 workgroups a split
    (16, 2, [2] * 32, 8192),
    (16, 1, [12] * 9, 16384),   # 192 of 256 rows in two chunks
    (32, 4, [40] * 7, [16384] + [512] * 6),  # one long prefix
    (32, 4, [64] + [2] * 6, 16384),          # one large group
    (16, 1, [16], 32768),       # two workgroups a split
    (16, 2, [64], 8192, 256),   # 5.3 batches
    (64, 4, [16], 8192),
    (32, 4, [33], 16384),       # 264 of 384 rows
    (16, 2, [64], 16384, 32),   # short tails
    (16, 2, [64], 16384, 513),  # long ones
    (8, 8, [24], 32768),        # 24 of 128 rows
])
def test_launches_that_lose_keep_the_chunks(case):
    assert _plan(*case) is None


@pytest.mark.parametrize(("case", "plan"), [
    ((16, 2, [64], 16384), (24, 1)),
    ((32, 4, [24], 8192), (24, 1)),
    ((32, 8, [24], 8192, 32), (24, 1)),
    ((32, 8, [40], 8192), (12, 1)),      # 160 of 256 rows, eight KV heads
    ((16, 2, [16] * 12, 8192), (8, 1)),
    ((16, 2, [8] * 12, 8192), (8, 1)),   # half the rows of one chunk
    ((16, 2, [16] * 12, 2048), (8, 1)),  # 24 workgroups a split, 4 batches
    ((32, 8, [32] * 4, [8192, 8000, 7936, 8192]), (6, 1)),
])
def test_launches_that_gain_take_them(case, plan):
    assert _plan(*case) == plan


def test_several_groups_need_their_filled_share():
    assert _plan(16, 2, [16] * 12, 8192, known=False) is None
    assert _plan(16, 2, [64], 16384, known=False) == (24, 1)
    assert _plan(16, 2, [64], 16384, head_dim=64) is None
    bt = torch.tensor([[3, 4, 5], [3, 4, 6], [8, -1, -1], [3, 4, 7]], dtype=torch.int32)
    g = cascade.build_cascade_groups(bt, torch.tensor([40, 48, 5, 35], dtype=torch.int32), 16, 16, 2)
    assert g.shared_tokens == 3 * 32
