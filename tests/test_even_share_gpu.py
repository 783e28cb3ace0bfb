"""GPU parity of the even-share decode (``fd_paged_decode_even``): the batch's tokens cut into equal
shares wherever the row boundaries fall.

The result must equal plain paged decode, so the oracle is the paged-decode oracle, at its tolerance
(atol 2e-2 / rtol 1e-2).  Cases sit where the shares, segments and merges change form: rows of zero, one,
31-33 tokens, rows over many shares (the merge's later passes), several rows in one share, batches of more
than 64 and more than 256 rows (several rows per lane of the length scan), both workgroup widths (256
(row, KV head) pairs and more take four waves), every block size, head dim and layout the kernel takes.
The workspace starts as NaN: a merge that reads a slot no workgroup wrote shows.
"""

import ctypes

import numpy as np
import pytest
import torch

from oracle.attention import paged_decode_attention as oracle_decode
from tests.helpers import assert_close_to_oracle, make_paged_inputs, np32

pytestmark = pytest.mark.gpu


def _even(q, k, v, table, lens, out, append=(None, None, None), kv_reuse=False):
    from flashdec_amd import _lib
    from flashdec_amd.paged_decode import _decode_args

    args, stream = _decode_args(q, k, v, table, lens, out, None, None, 2, "token_major", None, None, 1, *append,
                                False, kv_reuse)
    args.num_splits = 1
    args.struct_size = ctypes.sizeof(_lib.PagedDecodeArgs)
    floats = _lib.load_library().fd_paged_decode_even_floats(ctypes.byref(args))
    assert floats > 0
    ws = torch.full((floats,), float("nan"), device=q.device)
    assert _lib.paged_decode_even(args, ws.data_ptr(), floats, stream)
    torch.cuda.synchronize()
    return out


def _oracle(q, k, v, table, lens):
    return oracle_decode(np32(q), np32(k), np32(v), table.cpu().numpy(), lens.cpu().numpy())


EDGES = [700, 3, 0, 129, 2000, 64, 31, 1, 33, 32, 0, 95]
MANY = [int(x) for x in np.random.default_rng(5).integers(0, 140, 300)]  # 5 rows per lane of the scan


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("block_size", [8, 16, 32])
@pytest.mark.parametrize(("hq", "hkv", "d", "lens"), [
    (16, 2, 128, EDGES),           # 24 pairs: eight waves
    (16, 1, 128, EDGES),           # 16 heads per KV head
    (4, 4, 128, EDGES),            # one
    (14, 2, 64, EDGES),            # 64-dim heads
    (32, 8, 128, [1]),             # shares past the batch's last
    (2, 1, 128, [20000, 5]),       # one row over more shares than one merge pass takes
    (8, 4, 128, MANY),             # 1200 pairs: four waves, several rows a share
    (8, 1, 64, MANY),
    (16, 8, 128, [77] * 65),       # uniform rows, one more than the lanes
])
def test_even_shares_match_oracle(hq, hkv, d, lens, block_size, dtype):
    q, k, v, table, sl = make_paged_inputs(lens, hq, hkv, d, block_size, dtype, seed=block_size + hq)
    out = _even(q, k, v, table, sl, torch.full_like(q, 7.0))
    assert_close_to_oracle(out, _oracle(q, k, v, table, sl))
    for b, n in enumerate(lens):
        if n == 0:
            assert torch.count_nonzero(out[b]) == 0


@pytest.mark.parametrize("block_size", [8, 16, 32])
def test_even_shares_on_views_wide_tables_and_bad_blocks(block_size):
    """A vLLM-style cache view, 64-bit indices, tables wider than the rows, lengths past the table, ids outside
    the pool (masked), and an output with strides of its own."""
    lens = [40, 0, 333, 5000, 64, 17]
    q, k, v, table, sl = make_paged_inputs(lens, 16, 2, 128, block_size, seed=3, table_width=5000 // block_size + 9)
    table[2, 1] = -1
    table[3, 7] = k.shape[0] + 5
    sl = sl.long()
    sl[4] = 10**6  # more than the row's table holds
    table[4] = table[3]
    kv = torch.empty((k.shape[0], 2, block_size, 2, 128), device=k.device, dtype=k.dtype)
    kv[:, 0], kv[:, 1] = k.permute(0, 2, 1, 3), v.permute(0, 2, 1, 3)
    kview, vview = kv[:, 0].permute(0, 2, 1, 3), kv[:, 1].permute(0, 2, 1, 3)
    want = _even(q, k, v, table, sl, torch.empty_like(q))
    wide = torch.zeros((len(lens), 16, 256), device=q.device, dtype=q.dtype)
    got = _even(q, kview, vview, table.long(), sl, wide[..., ::2])
    assert torch.equal(got, want)
    assert torch.count_nonzero(wide[..., 1::2]) == 0
    from flashdec_amd import paged_decode_attention

    plain = paged_decode_attention(q, k, v, table, sl)  # the row kernel at this size
    assert_close_to_oracle(want, np32(plain))


@pytest.mark.parametrize("lens", [[int(x) for x in np.random.default_rng(9).integers(0, 70, 4200)],
                                  [0] * 4133 + [33] * 3 + [0] * 64 + [5000]])
def test_even_shares_of_more_rows_than_one_search_pass_sees(lens):
    """More than 64 rows a lane: the row search carries its base from one pass to the next."""
    q, k, v, table, sl = make_paged_inputs(lens, 4, 1, 128, 16, seed=12)
    out = _even(q, k, v, table, sl, torch.full_like(q, 7.0))
    assert_close_to_oracle(out, _oracle(q, k, v, table, sl))
    assert torch.count_nonzero(out[sl == 0]) == 0


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("block_size", [8, 16, 32])
@pytest.mark.parametrize(("hq", "hkv", "d", "lens"), [(16, 2, 128, EDGES), (14, 2, 64, EDGES), (8, 4, 128, MANY),
                                                      (8, 1, 64, MANY)])
def test_even_shares_with_cached_loads_and_an_unaligned_output(hq, hkv, d, lens, block_size, dtype):
    """Rows may share blocks; an output one element past a 16-byte line takes the rows' stores all the same."""
    q, k, v, table, sl = make_paged_inputs(lens, hq, hkv, d, block_size, dtype, seed=block_size + d)
    flat = torch.full((q.numel() + 8,), 7.0, device=q.device, dtype=dtype)
    out = flat[1 : 1 + q.numel()].view(q.shape)
    assert out.data_ptr() % 16
    want = _even(q, k, v, table, sl, torch.empty_like(q))
    assert torch.equal(_even(q, k, v, table, sl, out, kv_reuse=True), want)
    assert flat[0] == 7.0 and bool((flat[1 + q.numel() :] == 7.0).all())


def test_even_shares_append_into_8_token_blocks():
    """The C ABI takes them (the Python call's grouped rule does not)."""
    from flashdec_amd import _lib
    from flashdec_amd import paged_decode as pd

    lens = [1, 9, 64, 200, 777]
    q, k, v, table, sl = make_paged_inputs(lens, 16, 2, 128, 8, seed=8)
    ak, av = (torch.randn((len(lens), 2, 128), device="cuda").to(q.dtype) for _ in range(2))
    pos = sl.long() - 1
    slots = table.long().gather(1, (pos // 8)[:, None])[:, 0] * 8 + pos % 8
    k1, v1, out = k.clone(), v.clone(), torch.empty_like(q)
    args, stream = pd._decode_args(q, k1, v1, table, sl, out, None, None, 2, "token_major", None, None, 1, None, None,
                                   None, False, False)
    args.num_splits = 1
    pd._fill_append(args, ak, av, slots)
    args.struct_size = ctypes.sizeof(_lib.PagedDecodeArgs)
    floats = _lib.load_library().fd_paged_decode_even_floats(ctypes.byref(args))
    ws = torch.full((floats,), float("nan"), device=q.device)
    assert _lib.paged_decode_even(args, ws.data_ptr(), floats, stream)
    k[slots // 8, :, slots % 8], v[slots // 8, :, slots % 8] = ak, av
    assert torch.equal(k1, k) and torch.equal(v1, v)
    assert_close_to_oracle(out, _oracle(q, k, v, table, sl))


@pytest.mark.parametrize("block_size", [16, 32])
@pytest.mark.parametrize("batch", [5, 130])
def test_even_shares_append_the_current_token(batch, block_size):
    rng = np.random.default_rng(batch)
    lens = [int(x) for x in rng.integers(1, 400, batch)]
    lens[0], lens[1], lens[2] = 1, block_size + 1, 0
    q, k, v, table, sl = make_paged_inputs(lens, 16, 2, 128, block_size, seed=batch)
    ak, av = (torch.randn((batch, 2, 128), device="cuda").to(q.dtype) for _ in range(2))
    pos = (sl.long() - 1).clamp(min=0)
    slots = table.long().gather(1, (pos // block_size)[:, None])[:, 0] * block_size + pos % block_size
    slots[3] = -1  # a padding row: nothing written, a zero row
    slots[2] = 0  # an empty row's slot is not written either
    k1, v1 = k.clone(), v.clone()
    out = _even(q, k1, v1, table, sl, torch.empty_like(q), (ak, av, slots))
    live = [b for b in range(batch) if b not in (2, 3)]
    ids, off = slots[live] // block_size, slots[live] % block_size
    k[ids, :, off], v[ids, :, off] = ak[live], av[live]
    assert torch.equal(k1, k) and torch.equal(v1, v)
    sl[3] = 0
    assert_close_to_oracle(out, _oracle(q, k, v, table, sl))


def test_large_batches_take_even_shares_and_unaligned_pointers_do_not():
    """The public call routes by shape; the same shapes at pointers off a 16-byte line keep the general path."""
    import flashdec_amd as fd
    from flashdec_amd import _lib

    lens = [900 + 3 * i for i in range(200)]
    q, k, v, table, sl = make_paged_inputs(lens, 16, 2, 128, 32, seed=1, table_width=1024)
    _lib.record_launches(True)
    try:
        out = fd.decode(q, k, v, table, sl)
        assert any("even_decode_kernel" in n for n in _lib.last_launch())
        assert torch.equal(out, fd.decode(q, k, v, table, sl, kv_reuse=True))
        fd.decode(q, k, v, table[:, :2].contiguous(), sl)  # a small batch
        assert not any("even" in n for n in _lib.last_launch())
        assert torch.equal(out, fd.decode(q, k, v, table, sl))
        flat = torch.empty(q.numel() + 1, device=q.device, dtype=q.dtype)
        shifted = flat[1:].view(q.shape)
        shifted.copy_(q)
        general = fd.decode(shifted, k, v, table, sl)
        assert not any("even" in n for n in _lib.last_launch())
    finally:
        _lib.record_launches(False)
    assert_close_to_oracle(general, np32(out))


def test_the_route_follows_each_calls_pointers():
    """Calls of one shape at pointers on and off a 16-byte line, in either order and again: each takes its own kernel
    and gives its own bits."""
    import flashdec_amd as fd
    from flashdec_amd import _lib
    from flashdec_amd import paged_decode as pd

    q, k, v, table, sl = make_paged_inputs([900 + 3 * i for i in range(200)], 16, 2, 128, 32, seed=6, table_width=1024)
    shifted = torch.empty(q.numel() + 1, device=q.device, dtype=q.dtype)[1:].view(q.shape)
    shifted.copy_(q)
    ask = []
    args = pd._decode_args

    def counted(*a, **kw):
        ask.append(1)
        return args(*a, **kw)

    pd._LAST_LAUNCH.__dict__.clear()
    pd._decode_args = counted
    _lib.record_launches(True)
    try:
        outs = {}
        for query in (shifted, q, shifted, q, q, shifted):
            out = fd.decode(query, k, v, table, sl)
            assert any("even" in n for n in _lib.last_launch()) == (query is q)
            assert torch.equal(out, outs.setdefault(query is q, out))
    finally:
        _lib.record_launches(False)
        pd._decode_args = args
    assert len(ask) == 2  # each prepared once
    assert_close_to_oracle(outs[False], np32(outs[True]))


@pytest.mark.parametrize(("lens", "width", "ragged", "kernel"), [
    ([2048] * 8, 1024, False, "decode_mfma_kernel"),  # a small batch behind wide tables: one round of row workgroups
    ([40 * i + 1 for i in range(32)], 1024, True, "decode_balanced_kernel"),  # said to be ragged, 64 pairs
    ([40 * i + 1 for i in range(96)], 256, True, "even_decode_kernel"),  # 192 pairs
])
def test_calls_that_even_shares_would_slow_keep_their_kernels(lens, width, ragged, kernel):
    import flashdec_amd as fd
    from flashdec_amd import _lib

    q, k, v, table, sl = make_paged_inputs(lens, 16, 2, 128, 32, seed=4, table_width=width)
    _lib.record_launches(True)
    try:
        out = fd.decode(q, k, v, table, sl, ragged=ragged)
        assert kernel in _lib.last_launch()[0], _lib.last_launch()
    finally:
        _lib.record_launches(False)
    assert_close_to_oracle(out, _oracle(q, k, v, table, sl))


def test_the_rule_is_asked_only_where_it_can_take_a_call(monkeypatch):
    """Each new shape pays for the question: none for layouts, groups and sizes that are below every line."""
    from flashdec_amd import _lib
    from flashdec_amd import paged_decode as pd

    asked = []
    monkeypatch.setattr(_lib, "paged_decode_even_floats", lambda args: asked.append(args.num_seqs) or 0)
    for hq, hkv, d, batch, width, layout, times in [(16, 2, 128, 100, 128, "token_major", 1),
                                                    (16, 2, 128, 100, 128, "dim_major", 0),
                                                    (71, 1, 64, 300, 128, "token_major", 0),
                                                    (14, 2, 64, 20, 1024, "token_major", 0),
                                                    (16, 2, 128, 16, 64, "token_major", 0)]:
        q, k, v, table, sl = make_paged_inputs([40] * batch, hq, hkv, d, 32, seed=1, table_width=width,
                                               kv_layout=layout)
        asked.clear()
        out = pd.paged_decode_attention(q, k, v, table, sl, kv_layout=layout)
        assert len(asked) == times
        want = oracle_decode(np32(q), np32(k), np32(v), table.cpu().numpy(), sl.cpu().numpy(), kv_layout=layout)
        assert_close_to_oracle(out, want)


def test_even_share_workspaces_are_a_graphs_own_and_a_threads_own():
    """A captured call's partials stay in the graph's memory whatever the stream ran before, and threads on
    one stream have a workspace each."""
    import threading

    import flashdec_amd as fd
    from flashdec_amd import paged_decode as pd

    q, k, v, table, sl = make_paged_inputs([900 + 3 * i for i in range(200)], 16, 2, 128, 32, seed=2,
                                           table_width=1024)
    held = pd._EVEN_WORKSPACES.__dict__
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        want = fd.decode(q, k, v, table, sl)
        ws = held[(q.device.index, side.cuda_stream)]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = fd.decode(q, k, v, table, sl)
    assert held[(q.device.index, side.cuda_stream)] is ws
    for _ in range(3):
        ws.fill_(7.0)
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert bool((ws == 7.0).all())
        with torch.cuda.stream(side):  # the same call again, eager: the stream's own workspace, not the graph's
            assert torch.equal(fd.decode(q, k, v, table, sl), want)
        torch.cuda.synchronize()
        assert not bool((ws == 7.0).all())
    seen = []

    def other():
        with torch.cuda.stream(side):
            seen.append(fd.decode(q, k, v, table, sl))
        seen.append(pd._EVEN_WORKSPACES.__dict__[(q.device.index, side.cuda_stream)].data_ptr())
        torch.cuda.synchronize()

    t = threading.Thread(target=other)
    t.start()
    t.join()
    assert torch.equal(seen[0], want) and seen[1] != ws.data_ptr()
