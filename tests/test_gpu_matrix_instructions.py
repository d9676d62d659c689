"""Walks on 16x16x32 and on 32x32x16 matrix instructions: dense launches of one, two and four groups a line, of few and of many tiles, and
rows whose reference max is raised in the middle of a walk."""
import numpy as np
import pytest
import torch

from oracle import attn_oracle as ao
from tests.gpu_util import ATOL_O, RTOL_LSE, SCALE, lse_rel_err, max_abs
from ultraattn_amd import ops
from ultraattn_amd.flash_attn_interface import _flash_attn_backward, _flash_attn_forward

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _rows(tokens, heads, g):
    return torch.randn(1, tokens, heads, 128, generator=g).to(torch.bfloat16)


def _keep(sq, sk, causal):
    keep = torch.ones(sq, sk, dtype=torch.bool)
    return keep.tril(sk - sq) if causal else keep


@pytest.mark.parametrize("sq,sk,nh,causal", [
    (128, 128, 1, False), (128, 128, 1, True), (128, 128, 64, True),     # one tile a walk, four groups
    (1024, 1920, 16, False), (1024, 2048, 16, False),                    # four groups: 1920 and 2048 tiles
    (1024, 896, 32, False), (1024, 1024, 32, False),                     # two groups: 1792 and 2048
    (2048, 2048, 15, True), (2048, 2048, 16, True),                      # causal, four groups: 2040 and 2176
    (2048, 2048, 17, True),                                              # causal, two groups: 2312
    (2304, 2048, 16, True),                                              # rows above the first key
])
def test_both_instructions(sq, sk, nh, causal):
    g = torch.Generator().manual_seed(11)
    q, k, v, do = _rows(sq, nh, g), _rows(sk, nh, g), _rows(sk, nh, g), _rows(sq, nh, g)
    d = [t.to(DEV) for t in (q, k, v, do)]
    o, lse = [_flash_attn_forward(*d[:3], 0.0, SCALE, causal)[i] for i in (0, 5)]
    grads = [torch.empty_like(t) for t in d[:3]]
    _flash_attn_backward(d[3], *d[:3], o, lse, *grads, 0.0, SCALE, causal)
    keep = _keep(sq, sk, causal)
    for h in sorted({0, nh - 1}):
        s = slice(h, h + 1)
        cut = [t[:, :, s] for t in (q, k, v, do)]
        ro, rl = ao.dense_fwd(*cut[:3], SCALE, keep)
        assert max_abs(o[:, :, s], ro) <= ATOL_O and lse_rel_err(lse[:, s], rl) <= RTOL_LSE
        for a, b in zip(grads, ao.dense_bwd_autograd(*cut, SCALE, keep)):
            assert max_abs(a[:, :, s], b) <= 2e-2


# Keys grow along the walk, so that scores outgrow the reference max by far more than 2^24 again and again, in every row, or in the
# first or second 16 of every 32 alone (the two rows that one lane holds with 16x16x32).  An output is a mean of values, |v| <= 4.5 here,
# with weights rounded to bf16 and itself rounded: the difference stays below 4.5 * 2^-8 = 0.0176.
@pytest.mark.parametrize("quiet", [None, 0, 1])
@pytest.mark.parametrize("nh,tokens,listed", [(1, 512, False), (16, 2048, False), (2, 1024, True)])
def test_reference_raised_in_the_walk(quiet, nh, tokens, listed):
    g = torch.Generator().manual_seed(12)
    q, k, v = _rows(tokens, nh, g), _rows(tokens, nh, g), _rows(tokens, nh, g).clamp(-4.5, 4.5)
    k = (k.float() * torch.logspace(-1, 1, tokens).view(1, -1, 1, 1)).to(torch.bfloat16)
    if quiet is not None:
        half = (torch.arange(tokens) // 16 % 2 == quiet).view(1, -1, 1, 1)
        q = torch.where(half, q.float() * 0.02, q.float()).to(torch.bfloat16)
    d = [t.to(DEV) for t in (q, k, v)]
    if listed:
        o, lse = ops.bsa_fwd(*d, np.ones((tokens // 128,) * 2, np.uint8), SCALE, block=128)
    else:
        o, lse = [_flash_attn_forward(*d, 0.0, SCALE, False)[i] for i in (0, 5)]
    for h in sorted({0, nh - 1}):
        ro, rl = ao.dense_fwd(*[t[:, :, h:h + 1] for t in (q, k, v)], SCALE, _keep(tokens, tokens, False))
        assert max_abs(o[:, :, h:h + 1], ro) <= ATOL_O and lse_rel_err(lse[:, h:h + 1], rl) <= RTOL_LSE
