"""Executor with kernel tiles on both sides of the row length from which they run as launches of their own."""
import numpy as np
import pytest
import torch

from tests.gpu_util import SCALE, lse_rel_err, max_abs
from ultraattn_amd.executor import BlockSparseExecutor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_cols", [383, 384])
def test_long_rows(n_cols):
    g = torch.Generator(device="cuda:0").manual_seed(n_cols)
    mk = lambda n: torch.randn(1, n * 128, 1, 128, device="cuda:0", generator=g).to(torch.bfloat16)
    q, k, v = mk(1), mk(n_cols), mk(n_cols)
    one, four = (BlockSparseExecutor(np.ones((1, n_cols), np.uint8), 128, SCALE, kernel_tiles=n) for n in (1, 4))
    (o1, l1), (o4, l4) = one.forward(q, k, v), four.forward(q, k, v)
    assert (four._parts is not None) == (n_cols >= 384)
    s = (q.float()[0, :, 0] @ k.float()[0, :, 0].T) * SCALE
    ref = torch.softmax(s, -1) @ v.float()[0, :, 0]
    for o, l in ((o1, l1), (o4, l4)):
        assert max_abs(o[0, :, 0], ref.cpu()) <= 2e-2 and lse_rel_err(l[0, 0], torch.logsumexp(s, -1).cpu()) <= 1e-3
