"""Executor with kernel tiles on both sides of the row length and the head count from which they run as launches of their own."""
import numpy as np
import pytest
import torch

from tests.gpu_util import SCALE, lse_rel_err, max_abs
from ultraattn_amd.executor import BlockSparseExecutor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_cols,nh,launched", [(1023, 16, False), (1024, 16, True), (1024, 15, False)])
def test_long_rows(n_cols, nh, launched):
    g = torch.Generator(device="cuda:0").manual_seed(n_cols)
    mk = lambda n: torch.empty(1, n * 128, nh, 128, device="cuda:0", dtype=torch.bfloat16).normal_(generator=g)
    q, k, v = mk(64), mk(n_cols), mk(n_cols)
    one, four = (BlockSparseExecutor(np.ones((64, n_cols), np.uint8), 128, SCALE, kernel_tiles=n) for n in (1, 4))
    (o1, l1), (o4, l4) = one.forward(q, k, v), four.forward(q, k, v)
    assert four.launches_kernel_tiles(q) == (four._parts is not None) == launched
    rows = torch.tensor([0, 127, 128, 4095, 8191], device="cuda:0")
    for h in (0, nh - 1):
        s = (q[0, rows, h].float() @ k[0, :, h].float().T) * SCALE
        ref = torch.softmax(s, -1) @ v[0, :, h].float()
        # outputs of 131000 N(0, 1) keys have a standard deviation of 4.6e-3; two bf16 roundings of the largest, 0.03, are 1.2e-4
        for o, l in ((o1, l1), (o4, l4)):
            assert max_abs(o[0, rows, h], ref.cpu()) <= 2e-4 and lse_rel_err(l[0, h, rows], torch.logsumexp(s, -1).cpu()) <= 1e-5
