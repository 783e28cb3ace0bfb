"""The one-launch value checks ahead of an append: every rule, at the first and last row, over index types."""

import pytest
import torch

from flashdec_amd import _lib

pytestmark = pytest.mark.gpu

BLOCKS, BLOCK, ROWS = 7, 16, 50


@pytest.mark.parametrize("count", [1, 255, 257, 1024 * 256 + 3])
@pytest.mark.parametrize("types", [(torch.int32,) * 3, (torch.int64,) * 3, (torch.int64, torch.int32, torch.int64)])
def test_each_rule_at_the_first_and_last_row(count, types):
    good = (BLOCKS - 1, BLOCK - 1, ROWS - 1)  # the largest values that each rule takes
    tensors = [torch.full((count,), v, dtype=t, device="cuda") for v, t in zip(good, types)]
    run = lambda rows=ROWS, ts=tensors: _lib.check_append_indices(*ts, BLOCKS, BLOCK, rows)
    assert run() == (False, False, False, False)
    for which, bad, expect in [(0, -1, (1, 0, 0, 0)), (0, BLOCKS, (1, 0, 0, 0)), (1, -1, (0, 1, 0, 0)),
                               (1, BLOCK, (0, 1, 0, 0)), (2, -1, (0, 0, 1, 0)), (2, ROWS, (0, 0, 0, 1))]:
        for row in (0, count - 1):
            tensors[which][row] = bad
            assert run() == tuple(map(bool, expect)), (which, bad, row)
            tensors[which][row] = good[which]
    for which in range(3):  # beyond 32 bits nothing wraps into range
        if types[which] == torch.int64:
            tensors[which][count - 1] = 2**32 if which < 2 else -(2**32)
            assert run()[which]
            tensors[which][count - 1] = good[which]
    tensors[2][0] = torch.iinfo(types[2]).max
    assert run(-1) == (False, False, False, False)  # no table: any position is in range
    assert run(0)[3]
    assert _lib.check_append_indices(tensors[0], tensors[1], None, BLOCKS, BLOCK) == (False, False, False, False)
    assert _lib.check_append_indices(*[t[:0] for t in tensors], BLOCKS, BLOCK, 0) == (False, False, False, False)
