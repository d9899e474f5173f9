"""Selections over more rows than the chip holds a workgroup per chunk for, so that a
workgroup takes a run of chunks: runs that end inside a row, one workgroup a row, ties at
the k-th value across and inside runs, the order flag of a chunk inside a run -- against
the oracle."""

import pytest
import torch

from maskahead_amd.kernels.keep import keep_select
from maskahead_amd.kernels.select import topk_ascending
from oracle import selection as OS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,n,k", [(130, 5000, 700), (600, 2049, 33), (40, 20000, 3000), (112, 32800, 4096),
                                      (513, 1024, 1024)])
def test_topk_of_many_rows(gpu, rows, n, k):
    g = torch.Generator().manual_seed(rows + n)
    x = torch.randn((rows, n), generator=g).exp()
    x[::2, ::3] = (x[::2, ::3] * 8).floor() / 8           # heavy ties in half of the rows
    x[1] = 0.5                                            # a row of one value
    mask = (torch.rand((rows, n), generator=g) > 0.1).to(torch.uint8)
    for _ in range(2):                                    # the state is left clean
        assert torch.equal(topk_ascending(x.to(gpu), k, mask.to(gpu)).cpu(), OS.topk_ascending(x, k, mask))


@pytest.mark.parametrize("rows,n,cap,window", [(112, 12000, 1500, 128), (600, 1500, 200, 0), (70, 33000, 9000, 64)])
def test_keep_of_many_rows(gpu, rows, n, cap, window):
    g = torch.Generator().manual_seed(rows + cap)
    pos = torch.cumsum(1 + (torch.rand((rows, n), generator=g) < 0.3).to(torch.int64) * 7, -1) - 1
    score = torch.rand((rows, n), generator=g)
    score[:, ::3] = (score[:, ::3] * 16).floor() / 16
    got = keep_select(pos.to(torch.int32).to(gpu), score.to(gpu), cap, window, sink_tokens=4)
    assert torch.equal(got.cpu(), OS.keep_select(pos, score, cap, window, 4, None))
    pos[rows - 1, n - 700] = pos[rows - 1, n - 701]       # not increasing in the middle of the last run
    with pytest.raises(ValueError):
        keep_select(pos.to(torch.int32).to(gpu), score.to(gpu), cap, window, sink_tokens=4)
