"""Which decode calls the library cuts into even shares (``fd_paged_decode_even_pays``).

Without a GPU the library plans for 256 CUs.  The rule sees the tables' capacity, not the rows' lengths, so it takes a
call only where the even-share kernel measured no slower at any length: never where the row kernel's workgroups (pairs
x splits of ``fd_paged_decode_plan``) fit one round.  No counterpart in the reference.
"""

import ctypes

import pytest

from flashdec_amd import _lib


def _pays(batch, hq, hkv, d, cap, ragged=False):
    a = _lib.PagedDecodeArgs()
    a.struct_size = ctypes.sizeof(a)
    a.dtype, a.num_seqs, a.num_q_heads, a.num_kv_heads, a.head_dim = _lib.FD_DTYPE_BF16, batch, hq, hkv, d
    a.block_size, a.num_blocks, a.max_blocks_per_seq, a.num_splits = 32, 1 << 20, cap // 32, 1
    a.q_stride[:] = a.out_stride[:] = (hq * d, d, 1)
    a.k_stride[:] = a.v_stride[:] = (hkv * 32 * d, 32 * d, d, 1)
    a.block_tables_stride[:] = (cap // 32, 1)
    a.seq_lens_stride = 1
    a.balance_target = _lib.paged_decode_balance_target(batch, hkv) if ragged else 0
    return _lib.load_library().fd_paged_decode_even_pays(ctypes.byref(a))


@pytest.mark.parametrize(("batch", "hq", "hkv", "d", "cap"), [
    (8, 16, 2, 128, 32768),    # 16 pairs x 16 splits: one round, a small batch behind wide tables
    (32, 16, 2, 128, 8192),    # 64 x 4
    (64, 16, 2, 128, 4096),    # 128 x 2
    (128, 16, 2, 128, 2048),   # 256 x 1
    (193, 16, 1, 128, 2048),   # 193 x 1
    (32, 16, 2, 128, 2048),    # 64 x 4, under 12288 tiles
    (16, 16, 2, 128, 32768),   # 32 x 16: two rounds, under 64 pairs
    (193, 16, 2, 128, 2048),   # 386 x 1: one split, two rounds
    (384, 16, 2, 128, 2048),   # 768 x 1
    (1024, 16, 1, 128, 2048),  # 1024 x 1, 16 heads per KV head
    (100, 16, 2, 64, 4096),    # 64-dim heads: 200 x 2
    (128, 16, 16, 64, 2048),   # 2048 x 1
])
def test_calls_that_lose_at_some_length_keep_the_row_kernel(batch, hq, hkv, d, cap):
    assert _pays(batch, hq, hkv, d, cap) == 0


@pytest.mark.parametrize(("batch", "hq", "hkv", "d", "cap"), [
    (193, 32, 8, 128, 2048),  # 1544 x 2
    (64, 32, 8, 128, 4096),   # 512 x 2
    (48, 16, 2, 128, 2048),   # 96 x 5
    (24, 16, 2, 128, 32768),  # 48 x 16: three rounds
    (512, 16, 2, 128, 2048),  # 1024 x 1
    (2048, 16, 1, 128, 2048),
    (100, 16, 2, 64, 8192),   # 200 x 5
])
def test_batches_of_many_rounds_take_even_shares(batch, hq, hkv, d, cap):
    assert _pays(batch, hq, hkv, d, cap) == 1


def test_ragged_calls_keep_balanced_splits_up_to_192_pairs():
    assert _pays(32, 16, 2, 128, 32768, ragged=True) == 0
    assert _pays(95, 16, 2, 128, 8192, ragged=True) == 0
    assert _pays(96, 16, 2, 128, 8192, ragged=True) == 1
