"""Rows whose reference max is raised in the middle of a walk on 16x16x32 matrix instructions, where a lane holds two rows: lists of more than
256 lines (``fwd_kernel<1, false>``), the same lists in fewer lines (``fwd_short_kernel``, one row a lane) and dense rectangles without a
workspace (``fwd_plain_kernel``)."""
import numpy as np
import pytest
import torch

from oracle import attn_oracle as ao
from tests.gpu_util import ATOL_O, RTOL_LSE, SCALE, lse_rel_err, max_abs
from tests.test_gpu_dense import dense_unsplit
from ultraattn_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BLOCKS, HEADS = 8, 33                                  # 264 lines


# Keys grow along the walk, so that scores outgrow the reference by far more than 2^24 again and again, in every row or in the first or
# second 16 of every 32 alone: in either or both of a lane's rows.  An output is a mean of values, |v| <= 4.5 here, with weights
# rounded to bf16 and itself rounded: the difference stays below 4.5 * 2^-8 = 0.0176.
@pytest.mark.parametrize("quiet", [None, 0, 1])
@pytest.mark.parametrize("causal", [False, True])
def test_against_the_oracle(lib, quiet, causal):
    g = torch.Generator().manual_seed(13)
    n = BLOCKS * 128
    q, k, v, do = (torch.randn(1, n, HEADS, 128, generator=g) for _ in range(4))
    k = k * torch.logspace(-1, 1, n).view(1, -1, 1, 1)
    if quiet is not None:
        q = q * torch.where(torch.arange(n) // 16 % 2 == quiet, 0.02, 1.0).view(1, -1, 1, 1)
    q, k, v, do = (t.to(torch.bfloat16) for t in (q, k, v.clamp(-4.5, 4.5), do))
    mask = np.ones((BLOCKS, BLOCKS), np.uint8)
    keep = torch.ones(n, n, dtype=torch.bool)
    if causal:
        mask, keep = np.tril(mask, -1) + 2 * np.eye(BLOCKS, dtype=np.uint8), keep.tril()
    d = [t.to(DEV) for t in (q, k, v, do)]
    o, lse = ops.bsa_fwd(*d[:3], mask, SCALE, block=128)
    for h in (0, HEADS - 1):
        ro, rl = ao.dense_fwd(*[t[:, :, h:h + 1] for t in (q, k, v)], SCALE, keep)
        assert max_abs(o[:, :, h:h + 1], ro) <= ATOL_O and lse_rel_err(lse[:, h:h + 1], rl) <= RTOL_LSE
    few_o, few_lse = ops.bsa_fwd(*[t[:, :, :3].contiguous() for t in d[:3]], mask, SCALE, block=128)
    assert torch.equal(few_o, o[:, :, :3]) and torch.equal(few_lse, lse[:, :3])
    plain_o, plain_lse = dense_unsplit(lib, *d, causal)[:2]
    assert torch.equal(plain_o, o) and torch.equal(plain_lse, lse)
