"""The library's own split workspaces: a captured call's are the graph's, and threads share none.

No counterpart in the reference, whose callers bring the workspace (flashdec/kernels/paged_decode.py:1076-1096).
"""

import threading

import pytest
import torch

from tests.helpers import make_paged_inputs
from tests.test_cascade_gpu import make_prefix_inputs

pytestmark = pytest.mark.gpu


def _decode_call():
    import flashdec_amd as fd

    q, k, v, table, sl = make_paged_inputs([2048, 700, 1500, 64], 16, 2, 128, 32, seed=3)
    return q, lambda: fd.decode(q, k, v, table, sl)


def _cascade_call():
    from flashdec_amd import cascade

    q, k, v, table, lens, _ = make_prefix_inputs([(16, [5, 40, 77, 1])], [90], 16, 2, 32, torch.bfloat16)
    g = cascade.build_cascade_groups(table, lens, 32, 16, 2)
    return q, lambda: cascade.paged_decode_attention_cascade(q, k, v, table, lens, groups=g)


@pytest.mark.parametrize("make", [_decode_call, _cascade_call])
def test_a_captured_calls_partials_are_the_graphs_own(make):
    """Warm-up and capture on one stream: later, larger calls there replace the stream's workspace, so that the graph
    must not write it, nor an eager call the graph's."""
    from flashdec_amd import paged_decode as pd

    q, call = make()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        want = call()
        want = call()  # the arguments kept from the last call
        # the memory that the stream's calls write (its first float is a partial of theirs)
        stream_ws = pd._auto_workspace(q, 2, 1, side.cuda_stream)[0]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = call()
        second = call()
    for _ in range(3):
        stream_ws.fill_(7.0)
        out.zero_()
        second.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(second, want)
        assert bool((stream_ws == 7.0).all())
        with torch.cuda.stream(side):  # eager again, between replays
            assert torch.equal(call(), want)
        torch.cuda.synchronize()
        assert not bool((stream_ws == 7.0).all())


def test_threads_on_one_stream_have_a_workspace_each():
    from flashdec_amd import paged_decode as pd

    q, _ = _decode_call()
    stream = torch.cuda.current_stream().cuda_stream
    mine = pd._auto_workspace(q, 2, 4, stream)[0]
    theirs = []
    t = threading.Thread(target=lambda: theirs.append(pd._auto_workspace(q, 2, 4, stream)[0]))
    t.start()
    t.join()
    assert mine.data_ptr() != theirs[0].data_ptr()
    assert mine.data_ptr() == pd._auto_workspace(q, 2, 4, stream)[0].data_ptr()


def test_a_thread_keeps_the_workspaces_of_a_few_streams_only():
    from flashdec_amd import paged_decode as pd

    q, call = _decode_call()
    want = call()
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(3 * pd._HELD_STREAMS)]
    outs = []
    for _ in range(2):
        for s in streams:
            with torch.cuda.stream(s):
                outs.append(call())
                even = pd._even_workspace(q.device, 4096, s.cuda_stream)
                assert even is pd._even_workspace(q.device, 4096, s.cuda_stream)
    torch.cuda.synchronize()
    assert all(torch.equal(o, want) for o in outs)
    for held in (pd._WORKSPACES.__dict__, pd._EVEN_WORKSPACES.__dict__):
        assert len(held) <= pd._HELD_STREAMS and (q.device.index, streams[-1].cuda_stream) in held
