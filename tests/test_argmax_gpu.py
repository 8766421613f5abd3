"""Greedy sampling's argmax against torch on the CPU: the first of equals, a
NaN before everything, rows of nothing but -inf."""

import pytest
import torch

from llm_instance_gateway_amd import ops

pytestmark = pytest.mark.gpu
INF, NAN = float("inf"), float("nan")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("V", [1, 3, 7, 8, 9, 64, 1023, 8191, 8192, 8201, 40003, 128256])
@pytest.mark.parametrize("off", [0, 1, 5])
def test_argmax_rows(dtype, V, off):
    g = torch.Generator().manual_seed(V + off)
    whole = torch.randn(9, V + off + 3, generator=g).to(dtype)
    x = whole[:, off : off + V]  # rows at any alignment
    mid, last = V // 2, V - 1
    x[1] = 0.0                      # all equal
    x[2] = -INF
    x[3, mid] = x[3, last] = 9.0    # a tie
    x[4, last] = INF
    x[5, 0] = INF
    x[6, mid], x[6, last] = -NAN, NAN
    x[6, 0] = INF if mid else x[6, 0]
    x[7] = -INF
    x[7, last] = -3e38
    x[8] = -0.0
    x[8, mid] = 0.0
    want = [int(torch.where(r.isnan())[0][0]) if r.isnan().any() else int(torch.where(r == r.max())[0][0])
            for r in x.float()]
    dev = whole.cuda()[:, off : off + V]
    assert ops.argmax_rows(dev).tolist() == want
    assert ops.argmax_rows(dev[:0]).tolist() == []
    assert ops.argmax_rows(dev.t().contiguous().t()).tolist() == dev.argmax(-1).tolist()  # other strides: torch


def test_more_rows_than_a_grid_holds():
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randint(0, 9, (2**22 + 3, 5), generator=g, device="cuda").float()
    got = ops.argmax_rows(x)
    assert torch.equal(x.gather(1, got[:, None]).squeeze(1), x.amax(1)) and got.max() < 5 and got.min() >= 0
