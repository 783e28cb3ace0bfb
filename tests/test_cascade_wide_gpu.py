"""Wide prefix workgroups (128 of a group's rows on one read of the prefix): edges of chunks, batches and splits."""

import math

import pytest
import torch

from flashdec_amd import _lib, cascade

from tests.helpers import assert_close_to_oracle
from tests.test_cascade_gpu import _oracle, make_prefix_inputs

pytestmark = pytest.mark.gpu


# (Hq, Hkv), sharers, prefix blocks: rows below, at and past one chunk of 128; 64-token batches that the splits
# cut evenly, not at all, or that end inside a batch and inside a block's tile
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("block_size", [8, 16, 32])
@pytest.mark.parametrize(("heads", "sharers", "blocks"), [((16, 2), 3, 9), ((16, 2), 16, 16), ((16, 1), 9, 21),
                                                          ((8, 8), 130, 5)])
@pytest.mark.parametrize("plan", [(1, 1), (3, 2), (64, 1)])
def test_wide_chunks_match_oracle(heads, sharers, blocks, block_size, dtype, plan, monkeypatch):
    hq, hkv = heads
    tails = [(7 * i) % 61 for i in range(sharers)]
    q, k, v, table, lens, _ = make_prefix_inputs([(blocks, tails), (3, [9, block_size])], [0, 50], hq, hkv, block_size,
                                                 dtype)
    # what no row attends must not reach a result: poison the blocks that no table row names
    used = torch.unique(table[table >= 0]).long()
    free = torch.ones(k.shape[0], dtype=torch.bool, device=k.device)
    free[used] = False
    k[free], v[free] = math.nan, math.nan
    g = cascade.build_cascade_groups(table, lens, block_size, hq, hkv)
    monkeypatch.setattr(cascade, "plan_wide_cascade", lambda *a: plan)
    monkeypatch.setattr(cascade, "_LAST_CASCADE", type(cascade._LAST_CASCADE)())
    seen = []
    launch = _lib.paged_decode_cascade
    monkeypatch.setattr(_lib, "paged_decode_cascade",
                        lambda args, cas, stream: (seen.append(cas.chunk_rows), launch(args, cas, stream)))
    out = cascade.paged_decode_attention_cascade(q, k, v, table, lens, groups=g, block_size=block_size)
    assert seen == [_lib.CASCADE_WIDE_CHUNK_ROWS]
    assert_close_to_oracle(out, _oracle(q, k, v, table, lens))
    assert torch.count_nonzero(out[sharers + 2]) == 0  # the zero-length row


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize(("heads", "sharers", "blocks"), [((16, 2), 64, 256), ((32, 8), 40, 128)])
def test_wide_chunks_are_no_further_from_64_bits_than_32_row_chunks(heads, sharers, blocks, dtype, monkeypatch):
    """Peaked scores (queries of twice unit size): a wave of a wide workgroup takes more tokens of a row than one
    of a 32-row chunk does, and a peak's probability rounds to the cache type all the same."""
    hq, hkv = heads
    q, k, v, table, lens, _ = make_prefix_inputs([(blocks, [(37 * i) % 200 + 1 for i in range(sharers)])], [], hq, hkv,
                                                 32, dtype)
    q = q * 2
    g = cascade.build_cascade_groups(table, lens, 32, hq, hkv)
    narrow = cascade.paged_decode_attention_cascade(q, k, v, table, lens, groups=g, chunk_rows=32)
    monkeypatch.setattr(cascade, "plan_wide_cascade", lambda *a: (24, 1))
    monkeypatch.setattr(cascade, "_LAST_CASCADE", type(cascade._LAST_CASCADE)())
    wide = cascade.paged_decode_attention_cascade(q, k, v, table, lens, groups=g)
    exact = torch.empty(q.shape, device=q.device, dtype=torch.float64)
    for b, n in enumerate(lens.tolist()):
        ids = table[b, : -(-n // 32)].long()
        for h in range(hkv):
            kh, vh = (t[ids, h].reshape(-1, 128)[:n].double() for t in (k, v))
            qh = q[b, h * (hq // hkv) : (h + 1) * (hq // hkv)].double()
            p = torch.softmax((kh @ qh.t().contiguous()).t() / math.sqrt(128), dim=-1)
            exact[b, h * (hq // hkv) : (h + 1) * (hq // hkv)] = p.contiguous() @ vh
    off = [float((t.double() - exact).norm() / exact.norm()) for t in (wide, narrow)]
    assert off[0] <= off[1], off


@pytest.mark.parametrize(("kv_reuse", "nt"), [(True, "false"), (False, "true")])
@pytest.mark.parametrize(("heads", "groups", "sharers", "blocks"), [((32, 8), 1, 24, 256), ((16, 2), 12, 16, 64)])
def test_the_rule_reaches_the_wide_kernel(heads, groups, sharers, blocks, kv_reuse, nt):
    hq, hkv = heads
    q, k, v, table, lens, _ = make_prefix_inputs([(blocks, [(29 * i) % 300 + 1 for i in range(sharers)])] * groups,
                                                 [40], hq, hkv, 32, torch.bfloat16)
    g = cascade.build_cascade_groups(table, lens, 32, hq, hkv)
    _lib.record_launches(True)
    try:
        out = cascade.paged_decode_attention_cascade(q, k, v, table, lens, groups=g, kv_reuse=kv_reuse)
        assert _lib.last_launch()[0] == f"fd::cascade_wide_kernel<__bf16, 32, {nt}>", _lib.last_launch()
    finally:
        _lib.record_launches(False)
    assert torch.equal(out, cascade.paged_decode_attention_cascade(q, k, v, table, lens, groups=g, kv_reuse=kv_reuse))
    assert_close_to_oracle(out, _oracle(q, k, v, table, lens))


def test_plan_and_explicit_settings():
    def groups(members, prefix, tail=512):
        return cascade.CascadeGroups(members=torch.zeros((1, members), dtype=torch.int32),
                                     prefix_len=torch.zeros(1, dtype=torch.int32),
                                     row_prefix_len=torch.zeros(members, dtype=torch.int32), max_prefix_len=prefix,
                                     max_tail_len=tail, total_tail_len=1)

    assert cascade.plan_wide_cascade(64, 16, 2, 128, groups(64, 16384), 256) == (24, 1)  # 8 units, 192 workgroups
    assert cascade.plan_wide_cascade(24, 32, 4, 128, groups(24, 8192), 256) == (24, 1)  # exactly 6 * 2^20
    assert cascade.plan_wide_cascade(23, 32, 4, 128, groups(23, 8192), 256) is None
    assert cascade.plan_wide_cascade(64, 16, 2, 128, groups(64, 16384, 513), 256) is None
    # explicit settings keep what they took and refused
    q, k, v, table, lens, _ = make_prefix_inputs([(4, [5, 6])], [], 16, 2, 16, torch.bfloat16)
    g = cascade.build_cascade_groups(table, lens, 16, 16, 2)
    with pytest.raises(ValueError, match="chunk_rows must be 16 or 32"):
        cascade.paged_decode_attention_cascade(q, k, v, table, lens, groups=g, chunk_rows=128)
